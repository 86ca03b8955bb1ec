"""GPU: Model B runs in which the march (3D) or the one-plane kernel and the block
kernels take turns: the list's length crosses the line between them many times, both
ways, as blocks fall asleep and wake.

Each path reads the potentials of sleeping blocks that the other stored (the march stops
storing part-way through a block that fires), and the block kernels run on the smaller
grid they get where the march is there. Bar: bit-identical to the block kernels alone."""
import numpy as np
import pytest

from dba_amd import abi, configs

pytestmark = pytest.mark.gpu

PLAN = ((1, 0), (9, 0), (90, 10))


def run(ctx, p, X, env, monkeypatch):
    monkeypatch.setenv("DBA_MODELB_SUPERBLOCKS", env)
    inst = ctx.create(p)
    for f, a in enumerate(X):
        inst.upload(f, a)
    snaps = []
    for n, chunk in PLAN:
        inst.step(n, graph_chunk=chunk)
        info = inst.info()
        snaps.append([inst.download(f) for f in range(4)] +
                     [inst.active(0)[1], np.array([info.cell_updates, info.sim_time, info.cons_offset])])
    h = inst.history()
    inst.destroy()
    return snaps, h


@pytest.mark.parametrize("mode", [abi.MODE_DBA, abi.MODE_CONSERVED])
@pytest.mark.parametrize("shape,line", [((100, 64, 20), 900), ((268, 132, 1), 720)])
def test_march_and_block_kernels_in_turns(ctx, mode, shape, line, monkeypatch):
    nx, ny, nz = shape
    X = list(configs.modelb_ic(nx, ny, nz)) + [0.05 * configs.uniform01(9, nx * ny * nz).reshape(nz, ny, nx)]
    for f, v in enumerate((0.2, 0.2, 0.01)):   # noise in two corners, the rest at rest
        X[f][..., nx // 4: 3 * nx // 4] = v
        X[f][:, ny // 2:] = v
    p = configs.modelb_params(n=nx, nz=nz, mode=mode, eps=1e-3, history_cap=128)
    p.ny = ny
    a, ha = run(ctx, p, X, str(line), monkeypatch)
    b, hb = run(ctx, p, X, "0", monkeypatch)
    c, _ = run(ctx, p, X, "1", monkeypatch)
    for sa, sb, sc in zip(a, b, c):
        for u, v, w in zip(sa, sb, sc):
            assert np.array_equal(u, v) and np.array_equal(w, v)
    assert np.array_equal(ha, hb)
    long = hb[:, 0] >= line
    ups, downs = (np.diff(long.astype(int)) == 1).sum(), (np.diff(long.astype(int)) == -1).sum()
    assert ups >= 2 and downs >= 2, (ups, downs)
