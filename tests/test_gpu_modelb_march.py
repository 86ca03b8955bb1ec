"""GPU: the Model B column march (modelb_march_kernel: columns of 32 x 12 cells
walked up in z) against the block kernels and the oracle, at grids whose columns
are cut in x and y, with fewer blocks than a strip is long, and with sleeping
blocks inside a column (stored potentials, blocks current in different buffers).

Bar: bit-identical to the block kernels (the same expressions per cell, change
sums in the same order), same awake sets and history; within 1e-10 of the oracle
(log and exp)."""
import numpy as np
import pytest

from dba_amd import abi, configs
from oracle.oracle import OracleSim

pytestmark = pytest.mark.gpu


def run(ctx, p, X, env, monkeypatch):
    monkeypatch.setenv("DBA_MODELB_SUPERBLOCKS", env)
    inst = ctx.create(p)
    for f, a in enumerate(X):
        inst.upload(f, a)
    snaps = []
    for chunk, graph in ((1, 0), (5, 0), (12, 4)):
        inst.step(chunk, graph_chunk=graph)
        snaps.append([inst.download(f) for f in range(3)] + [inst.active(0)[1]])
    h = inst.history()
    inst.destroy()
    return snaps, h


@pytest.mark.parametrize("mode", [abi.MODE_REGULAR, abi.MODE_DBA, abi.MODE_CONSERVED])
@pytest.mark.parametrize("shape", [(4, 4, 4), (8, 12, 4), (36, 28, 8), (64, 20, 44), (100, 64, 20)])
def test_march_matches_block_kernels(ctx, mode, shape, monkeypatch):
    nx, ny, nz = shape
    X = list(configs.modelb_ic(nx, ny, nz)) + [0.05 * configs.uniform01(9, nx * ny * nz).reshape(nz, ny, nx)]
    if nx >= 64:   # a quiet slab: sleeping blocks, waking as the noise spreads
        for f, v in enumerate((0.2, 0.2, 0.01)):
            X[f][..., nx // 4: 3 * nx // 4] = v
            X[f][:, ny // 2:] = v
    p = configs.modelb_params(n=nx, nz=nz, mode=mode, eps=1e-4, history_cap=32)
    p.ny = ny
    a, ha = run(ctx, p, X, "1", monkeypatch)
    b, hb = run(ctx, p, X, "0", monkeypatch)
    for sa, sb in zip(a, b):
        for f in range(3):
            assert np.array_equal(sa[f], sb[f]), (f, np.max(np.abs(sa[f] - sb[f])))
        assert np.array_equal(sa[3], sb[3])
    assert np.array_equal(ha, hb)
    o = OracleSim(p)
    for f, v in enumerate(X):
        o.set_field(f, v)
    o.step(18)
    for f in range(3):
        assert np.max(np.abs(a[-1][f] - o.get_field(f))) <= 1e-10, f
    if mode != abi.MODE_REGULAR:
        assert np.array_equal(a[-1][3], o.awake(0))
        if nx >= 64:
            assert ha[:, 0].min() < nx * ny * nz // 64   # some blocks slept


@pytest.mark.parametrize("shape", [(36, 28, 8)])
def test_logarithms_outside_their_domain(ctx, shape, monkeypatch):
    """Cells with a concentration of 0, below 0 or infinite, and no solvent left: the
    march's logarithms for such lanes give what the block kernels' do (NaN, infinities)."""
    nx, ny, nz = shape
    X = list(configs.modelb_ic(nx, ny, nz)) + [np.zeros((nz, ny, nx))]
    X[0][4, 5, 6] = 0.0
    X[1][1, 20, 30] = -0.01
    X[2][6, 14, 17] = np.inf
    X[0][3, 25, 2], X[1][3, 25, 2] = 0.6, 0.4 - X[2][3, 25, 2]
    p = configs.modelb_params(n=nx, nz=nz, mode=abi.MODE_REGULAR)
    p.ny = ny
    a, _ = run(ctx, p, X, "1", monkeypatch)
    b, _ = run(ctx, p, X, "0", monkeypatch)
    for sa, sb in zip(a, b):
        for f in range(3):
            assert np.array_equal(sa[f], sb[f], equal_nan=True), f
    assert np.isnan(a[0][0]).any() and np.isfinite(a[0][0]).any()
