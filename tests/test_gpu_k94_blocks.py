"""GPU: the K94 step (a wave per block) against the oracle where its block
arithmetic can go wrong: one block along an axis (its own neighbour on both
sides), two (the same neighbour twice), 4x4x1 blocks of flat grids, grids whose
sides differ, more blocks than the waves of a launch, several instances at once.

Tolerance: fields of order 1 through 36 steps; the two sides differ in the last
place of atan only, which a step multiplies by dt / tau < 1: a hundred times less
than the other 3D tests allow."""
import numpy as np
import pytest

from dba_amd import abi, configs
from oracle.oracle import OracleSim

pytestmark = pytest.mark.gpu

TOL = 1e-12
STEPS = (1, 5, 30)


def make(nx, ny, nz, mode):
    p = configs.dendrite_k94_params(n=nx, nz=nz, mode=mode, history_cap=64)
    p.ny = ny
    return p, configs.dendrite_k94_ic(nx, ny, nz)


def check(insts, sims, mode):
    for inst, o in zip(insts, sims):
        for f in (0, 1):
            d = np.max(np.abs(inst.download(f) - o.get_field(f)))
            assert d <= TOL, (f, d)
            if mode == abi.MODE_DBA:
                assert np.array_equal(inst.active(f)[1], o.awake(f))
        assert np.array_equal(inst.history(), o.history())


@pytest.mark.parametrize("mode", [abi.MODE_REGULAR, abi.MODE_DBA])
@pytest.mark.parametrize("sizes", [[(4, 4, 4)], [(8, 4, 12)], [(4, 8, 1)], [(36, 12, 1)], [(36, 28, 20)],
                                   [(96, 72, 64)], [(8, 8, 8), (20, 16, 12), (40, 24, 28)]],
                         ids=lambda s: "+".join("x".join(map(str, v)) for v in s))
def test_k94_blocks_match_oracle(ctx, mode, sizes):
    insts, sims = [], []
    for s in sizes:
        p, fields = make(*s, mode)
        inst, o = ctx.create(p), OracleSim(p)
        for f, v in enumerate(fields):
            inst.upload(f, v)
            o.set_field(f, v)
        insts.append(inst)
        sims.append(o)
    for n in STEPS:
        ctx.step(insts, n)
        for o in sims:
            o.step(n)
        check(insts, sims, mode)
    for inst in insts:
        inst.destroy()
