"""GPU: resident steps whose waits for other workgroups run out.

The bound of a wait is set to a single look, so that waits run out within a step or two
of every launch, as they would if the launch were never resident as a whole. Every
workgroup has to leave its steps together and the launch has to end."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# in a process of its own: resident steps need a context alone on its device
CHILD = """
import sys
sys.path[:0] = [{root!r}, {tests!r}]
from dba_amd import Context, abi, configs
from test_gpu_resident import patchy
for model, mode, nx, ny, tile in {cases!r}:
    with Context(0) as ctx:
        if model == "ch":
            inst = ctx.create(configs.ch_params(n=nx, ny=ny, tile=tile, mode=mode, eps=1e-3, react_gamma=0.01, cbar=0.05))
            inst.upload(0, patchy(nx, ny, tile))
        else:
            inst = ctx.create(configs.dendrite_k93_params(n=nx, ny=ny, tile=tile, mode=mode))
            for f, v in enumerate(configs.dendrite_k93_ic(nx, ny, seeds=[(nx // 2, ny // 3)])):
                inst.upload(f, v)
        ctx.set_resident_wait(1)
        print("steps", model, mode, nx, ny, tile, flush=True)
        inst.step(200)
        taken = ctx.resident_calls()
        try:
            ctx.sync()
        except abi.DbaError as e:
            assert "waited" in str(e), e
        assert taken == 1
        print("ended", flush=True)
"""


def child(cases, source=CHILD, timeout=100):
    code = source.format(root=ROOT, tests=os.path.join(ROOT, "tests"), cases=cases)
    r = subprocess.run([sys.executable, "-u", "-c", code], capture_output=True, text=True, timeout=timeout, cwd=ROOT)
    print(r.stdout, r.stderr)
    return r


def test_workgroups_leave_together():
    cases = [("ch", m, nx, ny, t) for m in (0, 1)
             for nx, ny, t in ((64, 66, 32), (1024, 1024, 32), (1534, 1310, 32), (900, 700, 16), (514, 480, 8))]
    cases += [("k93", m, nx, ny, t) for m in (0, 1) for nx, ny, t in ((256, 256, 16), (512, 512, 16), (500, 500, 32))]
    r = child(cases)
    assert r.returncode == 0 and r.stdout.count("ended") == len(cases)
