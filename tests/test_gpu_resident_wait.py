"""GPU: resident steps whose waits for other workgroups run out.

The bound of a wait is set to a single look, so that waits run out within a step or two
of every launch, as they would if the launch were never resident as a whole. Every
workgroup has to leave its steps together and the launch has to end; the instance is as
it was before the launch, and its steps are made on the other paths, so that no caller
sees a difference."""
import os
import subprocess
import sys

import numpy as np
import pytest

from dba_amd import abi, configs
from test_gpu_resident import patchy, run, same

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CH_CASES = [("ch", m, nx, ny, t) for m in (abi.MODE_REGULAR, abi.MODE_DBA)
            for nx, ny, t in ((64, 66, 32), (1024, 1024, 32), (1534, 1310, 32), (900, 700, 16), (514, 480, 8))]
K93_CASES = [("k93", m, nx, ny, t) for m in (abi.MODE_REGULAR, abi.MODE_DBA)
             for nx, ny, t in ((256, 256, 16), (512, 512, 16), (500, 500, 32))]


def problem(model, mode, nx, ny, tile):
    if model == "ch":
        p = configs.ch_params(n=nx, ny=ny, tile=tile, mode=mode, eps=1e-3, react_gamma=0.01, cbar=0.05, history_cap=256)
        return p, [patchy(nx, ny, tile)]
    p = configs.dendrite_k93_params(n=nx, ny=ny, tile=tile, mode=mode, history_cap=256)
    return p, list(configs.dendrite_k93_ic(nx, ny, seeds=[(nx // 2, ny // 3)]))


@pytest.fixture
def short_wait(ctx):
    """The session's context with waits of a single look."""
    ctx.set_resident_wait(1)
    yield ctx
    ctx.set_resident_wait(0)
    ctx.set_resident(True)


def launched(ctx, p, fields, plan):
    ctx.set_resident(False)
    try:
        return run(ctx, p, fields, 1, plan)
    finally:
        ctx.set_resident(True)


@pytest.mark.parametrize("case", CH_CASES + K93_CASES)
def test_steps_given_up_are_made_again(short_wait, case):
    """Fields, awake sets, history, counters and time as on the other paths; the tiles
    sleep and wake before and after the launch that is given up."""
    ctx = short_wait
    p, fields = problem(*case)
    plan = (40, 64, 50)
    want = launched(ctx, p, fields, plan)
    for given_up in range(len(plan)):   # the launch of that entry; before it they run to their end
        redone = ctx.resident_redone()
        ctx.set_resident_wait(0)
        inst = ctx.create(p)
        for f, v in enumerate(fields):
            inst.upload(f, v)
        got = []
        for k, n in enumerate(plan):
            if k == given_up:
                ctx.set_resident_wait(1)
            inst.step(n)
            info = inst.info()
            got.append((np.stack([inst.download(f) for f in range(len(fields))]),
                        np.stack([inst.active(f)[1] for f in range(len(fields))]), inst.history(), info.cell_updates,
                        info.field_updates, info.steps_done, info.sim_time))
        inst.destroy()
        same(got, want)
        assert ctx.resident_redone() in (redone, redone + plan[given_up])
        if case[2] > 500:
            assert ctx.resident_redone() == redone + plan[given_up]
        ctx.set_resident(True)   # (given up, the context keeps to the other paths)


@pytest.mark.parametrize("case", [CH_CASES[6], K93_CASES[4]])
@pytest.mark.parametrize("read", ["download", "sync", "field_sum", "check_finite", "worklist", "history", "active",
                                  "droplets", "growth_front"])
def test_first_read_sees_all_steps(short_wait, case, read):
    """Several launches queued before the first call that waits, whichever it is."""
    ctx = short_wait
    p, fields = problem(*case)
    calls = {"download": lambda i: i.download(0), "sync": lambda i: ctx.sync(), "field_sum": lambda i: i.field_sum(0),
             "check_finite": lambda i: i.check_finite(), "worklist": lambda i: i.worklist(),
             "history": lambda i: i.history(), "active": lambda i: i.active(0)[1],
             "droplets": lambda i: i.droplets(0)[2], "growth_front": lambda i: i.growth_front([p.nx // 2])}
    if read == "growth_front" and case[0] == "ch":
        pytest.skip("a dendrite's diagnostic")
    out = []
    for resident in (False, True):
        ctx.set_resident(resident)
        redone = ctx.resident_redone()
        inst = ctx.create(p)
        for f, v in enumerate(fields):
            inst.upload(f, v)
        for n in (40, 30, 12):
            inst.step(n)
        first = calls[read](inst)
        out.append([first, inst.download(0), inst.history(), inst.info().steps_done])
        assert ctx.resident_redone() == redone + (82 if resident else 0)
        inst.destroy()
    for a, b in zip(*out):
        assert np.array_equal(a, b)


def test_other_work_after_steps_given_up(short_wait):
    """Launched steps of the same instance, an upload, another instance and a destroyed
    one, queued behind a launch that is given up."""
    ctx = short_wait
    p, fields = problem("ch", abi.MODE_DBA, 1024, 1024, 32)
    q, kf = problem("k93", abi.MODE_DBA, 512, 512, 16)
    out = []
    for resident in (False, True):
        ctx.set_resident(resident)
        a, b, gone = ctx.create(p), ctx.create(q), ctx.create(p)
        for inst in (a, gone):
            inst.upload(0, fields[0])
        for f, v in enumerate(kf):
            b.upload(f, v)
        gone.step(30)
        gone.destroy()
        a.step(40)
        b.step(50)          # resident, or skipped behind the launch given up
        a.step(5)           # too few steps for it
        b.step(13)
        ctx.step([a, b], 4)
        if resident:
            ctx.set_resident(True)
        a.step(20)
        a.upload(0, np.ascontiguousarray(fields[0][::-1]))
        a.step(24)
        res = [a.download(0), b.download(0), b.download(1), a.history(), b.history()]
        res += [a.info().steps_done, b.info().steps_done, a.info().sim_time, a.info().cell_updates]
        out.append(res)
        if resident:        # a fresh start: resident again, to the end
            ctx.set_resident(True)
            ctx.set_resident_wait(0)
            n0, r0 = ctx.resident_calls(), ctx.resident_redone()
            a.step(30)
            ctx.sync()
            assert ctx.resident_calls() == n0 + 1 and ctx.resident_redone() == r0
        a.destroy()
        b.destroy()
    for x, y in zip(*out):
        assert np.array_equal(x, y)


PAIR = """
import sys, time
sys.path[:0] = [{root!r}, {tests!r}]
import numpy as np
from dba_amd import Context, abi
from test_gpu_resident_wait import problem
model, mode, nx, ny, tile = {cases!r}
p, fields = problem(model, mode, nx, ny, tile)
out = []
with Context(0) as ctx:
    print("ready", flush=True)
    sys.stdin.readline()
    for resident in (True, False):
        ctx.set_resident(resident)
        inst = ctx.create(p)
        for f, v in enumerate(fields):
            inst.upload(f, v)
        for _ in range(40):
            inst.step(100)
        out.append(inst.download(0))
        print("steps", ctx.resident_calls(), ctx.resident_redone(), flush=True)
        inst.destroy()
assert np.array_equal(*out)
print("ended", flush=True)
"""


def test_two_processes_on_one_gpu():
    """Two processes, each with a grid that fills the GPU, in the default mode: whichever
    of them gets cooperative launches (the runtime here gives one process at a time the
    queue for them), both get what they would get alone."""
    procs = []
    for case in (CH_CASES[6], K93_CASES[4]):
        code = PAIR.format(root=ROOT, tests=os.path.join(ROOT, "tests"), cases=case)
        procs.append(subprocess.Popen([sys.executable, "-u", "-c", code], stdin=subprocess.PIPE, stdout=subprocess.PIPE,
                                      stderr=subprocess.PIPE, text=True, cwd=ROOT))
    try:
        for q in procs:
            assert q.stdout.readline().strip() == "ready"
        for q in procs:
            q.stdin.write("go\n")
            q.stdin.flush()
        for q in procs:
            o, e = q.communicate(timeout=90)
            print(o, e)
            assert q.returncode == 0 and "ended" in o
    finally:
        for q in procs:
            if q.poll() is None:
                q.kill()
