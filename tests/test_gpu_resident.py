"""GPU: resident CH steps (k_resident.h: many steps of one instance in one
cooperative launch, the fields in LDS) against the worklist path and the oracle.

Bar: bit-identical fields, awake sets, history, counters and time. The cases:
one tile and two by two (a region whose neighbours are itself), regions cut by
the grid and by partial tiles, closed boundaries, sleeping and waking tiles,
both stencils, regular mode, every tile size, the largest grids of a region
shape, runs cut into several launches, two contexts on two threads."""
import threading

import numpy as np
import pytest

from dba_amd import Context, abi, configs
from oracle.oracle import OracleSim

pytestmark = pytest.mark.gpu

PLAN = (40, 11, 12, 64)   # resident but for the 11 steps, which are too few for it


def patchy(nx, ny, tile, seed=7):
    """Noise in patches on a quiet ground: some tiles sleep, some wake again."""
    c = configs.ch_ic(nx, ny, seed=seed, cbar=0.05)
    y, x = np.mgrid[0:ny, 0:nx]
    c[((x // tile) % 7 >= 2) | ((y // tile) % 6 >= 2)] = 0.05
    return c


def run(ctx, p, c0, mode, plan=PLAN):
    """c0: one field, or the list of fields."""
    fields = c0 if isinstance(c0, list) else [c0]
    ctx.set_single_launch(mode)
    try:
        inst = ctx.create(p)
        for f, v in enumerate(fields):
            inst.upload(f, v)
        out = []
        for n in plan:
            inst.step(n, graph_chunk=16)
            info = inst.info()
            out.append((np.stack([inst.download(f) for f in range(len(fields))]),
                        np.stack([inst.active(f)[1] for f in range(len(fields))]), inst.history(), info.cell_updates,
                        info.field_updates, info.steps_done, info.sim_time))
        inst.destroy()
        return out
    finally:
        ctx.set_single_launch(1)


def same(a, b):
    for x, y in zip(a, b):
        assert np.array_equal(x[0], y[0]), np.max(np.abs(x[0] - y[0]))
        assert np.array_equal(x[1], y[1]) and np.array_equal(x[2], y[2]) and x[3:] == y[3:]


@pytest.mark.parametrize("mode", [abi.MODE_REGULAR, abi.MODE_DBA])
@pytest.mark.parametrize("nx,ny,tile,stencil,bc", [
    (32, 32, 32, 9, 0), (64, 66, 32, 5, 0), (8, 10, 8, 9, 0), (40, 24, 8, 5, 1), (70, 130, 16, 9, 1),
    (1024, 1024, 32, 9, 0), (1000, 996, 32, 9, 1), (1200, 1100, 32, 5, 0), (1534, 1310, 32, 9, 0), (514, 480, 8, 9, 0), (900, 700, 16, 5, 0)])
def test_resident_equals_worklist(ctx, mode, nx, ny, tile, stencil, bc):
    p = configs.ch_params(n=nx, ny=ny, tile=tile, mode=mode, stencil=stencil, eps=1e-3, react_gamma=0.01, cbar=0.05,
                          history_cap=128)
    p.bc_x = p.bc_y = bc
    c0 = patchy(nx, ny, tile)
    a = run(ctx, p, c0, 1)
    same(a, run(ctx, p, c0, 0))
    if mode == abi.MODE_DBA and nx > 500:
        h = a[-1][2][:, 0]
        assert 0 < h[-1] < a[-1][1].size and (np.diff(h) > 0).any() and (np.diff(h) < 0).any()  # tiles wake and sleep


def test_resident_matches_oracle(ctx):
    p = configs.ch_params(n=300, ny=260, tile=32, eps=2e-3, react_gamma=0.01, cbar=0.05)
    c0 = patchy(300, 260, 32)
    got = run(ctx, p, c0, 1, (60,))[0]
    o = OracleSim(p)
    o.set_field(0, c0)
    o.step(60)
    assert np.array_equal(got[0][0], o.get_field(0))
    assert np.array_equal(got[1][0], o.awake(0))


# K93: one tile a workgroup (256^2 at 16 x 16) and two by two (and larger grids, which
# do not fit and keep single-launch steps); closed boundaries as in its configuration, and periodic
@pytest.mark.parametrize("mode", [abi.MODE_REGULAR, abi.MODE_DBA])
@pytest.mark.parametrize("nx,ny,tile,bc", [
    (16, 16, 16, 0), (32, 34, 16, 1), (256, 256, 16, 1), (250, 310, 16, 0), (512, 512, 16, 1), (700, 1000, 16, 1),
    (40, 56, 8, 1), (514, 480, 8, 0), (32, 66, 32, 1), (500, 530, 32, 1), (900, 1024, 32, 0)])
def test_resident_k93_equals_worklist(ctx, mode, nx, ny, tile, bc):
    p = configs.dendrite_k93_params(n=nx, ny=ny, tile=tile, mode=mode, history_cap=128, bc=bc)
    seeds = [(nx // 2, ny // 3), (nx // 8, ny // 8)] if nx > 100 else [(nx // 2, ny // 2)]
    fields = list(configs.dendrite_k93_ic(nx, ny, seeds=seeds))
    a = run(ctx, p, fields, 1)
    same(a, run(ctx, p, fields, 0))
    if mode == abi.MODE_DBA and nx > 200:
        awake = a[-1][1]
        assert 0 < awake[0].sum() < awake[0].size and not np.array_equal(awake[0], awake[1])


def test_resident_two_contexts(ctx):
    """Two more contexts on two threads, each with a grid that fills the GPU: none of
    them takes resident steps while it is not alone, and the results are the same."""
    p = configs.ch_params(n=1024, tile=32, eps=1e-3, react_gamma=0.01, cbar=0.05, history_cap=256)
    c0 = [patchy(1024, 1024, 32, seed=s) for s in (3, 4)]
    want = [run(ctx, p, c, 0, (150,)) for c in c0]
    got, errs = [None, None], []

    def work(k):
        try:
            with Context(0) as own:
                got[k] = run(own, p, c0[k], 1, (50, 50, 50))
        except Exception as e:   # noqa: BLE001 - handed to the test's thread
            errs.append(e)

    ts = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not errs, errs
    for k in range(2):
        same(got[k][-1:], want[k][-1:])
