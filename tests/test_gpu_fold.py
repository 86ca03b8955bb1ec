"""GPU: groups of several segments (the end-of-step kernel sums the step before it
for each instance in workgroups of its own): n steps in one call must give what n
calls of one step give, in which the last step's merge launch does those sums.

Bar: bit-identical fields and worklists, equal awake sets, histories, counters and
times. Cases: 18 instances (more than the 16 one workgroup sums), instances of one
and of several segments in one group, partial tiles, 3D blocks, the 3x3 dilation."""
import numpy as np
import pytest

from dba_amd import abi, configs

pytestmark = pytest.mark.gpu

STEPS = 7


def k93(n, ny=None, seed=0):
    ny = ny or n
    p = configs.dendrite_k93_params(n=n, ny=ny, tile=16, history_cap=STEPS)
    return p, list(configs.dendrite_k93_ic(n, ny, seeds=[(20 + 3 * seed, 24 + seed), (n // 2, ny // 2)]))


def k94(n):
    p = configs.dendrite_k94_params(n=n, nz=n)
    p.history_cap = STEPS
    return p, list(configs.dendrite_k94_ic(n, n, n))


def kh(n):
    p = configs.kh_reference_params(n=n, tile=8)
    p.history_cap = STEPS
    U = configs.kh_reference_ic(n)
    rho, u, v, pr = configs.kh_primitive(U, 5.0 / 3.0, p.dx * p.dx)
    return p, configs.kh_conserved(rho, u, v, pr, 5.0 / 3.0, p.dx * p.dx)


CASES = {
    "18 dendrites": lambda: [k93(80 + 2 * i, 96, i) for i in range(18)],
    "one and several segments": lambda: [k93(64), k93(530, 516), k93(528, 1100, 3)],
    "one instance, 5 segments": lambda: [k93(1100, 1024)],
    "3D blocks": lambda: [k94(48)],
    "3x3 dilation": lambda: [kh(512)],
}


def run(ctx, items, calls):
    ctx.set_single_launch(0)
    try:
        insts = []
        for p, fields in items:
            inst = ctx.create(p)
            for f, v in enumerate(fields):
                inst.upload(f, v)
            insts.append(inst)
        for n in calls:
            ctx.step(insts, n)
        out = []
        for inst, (p, fields) in zip(insts, items):
            info = inst.info()
            nsets = 2 if len(fields) == 2 else 1
            out.append(([inst.download(f) for f in range(len(fields))], [inst.active(s)[1] for s in range(nsets)],
                        inst.worklist(), inst.history(), info.cell_updates, info.field_updates, info.steps_done,
                        info.sim_time))
            inst.destroy()
        return out
    finally:
        ctx.set_single_launch(1)


@pytest.mark.parametrize("name", list(CASES))
def test_one_call_equals_single_steps(ctx, name):
    items = CASES[name]()
    a, b = run(ctx, items, [STEPS]), run(ctx, items, [1] * STEPS)
    for x, y in zip(a, b):
        for u, v in zip(x[0] + x[1] + [x[2], x[3]], y[0] + y[1] + [y[2], y[3]]):
            assert np.array_equal(u, v)
        assert x[4:] == y[4:]
        assert x[6] == STEPS and x[4] > 0
