"""GPU: the Model B step of a grid of one plane (modelb_plane_kernel, 32 x 12 cells
per workgroup) against the block kernels and the oracle, at grids whose columns are
cut in x and y, smaller than one column, and with sleeping blocks inside a column.

Bar: bit-identical to the block kernels (the same expressions per cell, change sums
in the same order), same awake sets and history; within 1e-10 of the oracle."""
import numpy as np
import pytest

from dba_amd import abi, configs
from oracle.oracle import OracleSim
from test_gpu_modelb_march import run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [abi.MODE_REGULAR, abi.MODE_DBA, abi.MODE_CONSERVED])
@pytest.mark.parametrize("shape", [(4, 4), (8, 12), (32, 24), (36, 28), (100, 64), (268, 132)])
def test_plane_matches_block_kernels(ctx, mode, shape, monkeypatch):
    nx, ny = shape
    X = list(configs.modelb_ic(nx, ny, 1)) + [0.05 * configs.uniform01(9, nx * ny).reshape(1, ny, nx)]
    if nx >= 100:   # a quiet band: sleeping blocks, waking as the noise spreads
        for f, v in enumerate((0.2, 0.2, 0.01)):
            X[f][..., nx // 5: nx // 5 + 64] = v
            X[f][:, ny // 2:] = v
    p = configs.modelb_params(n=nx, nz=1, mode=mode, eps=1e-4, history_cap=32)
    p.ny = ny
    a, ha = run(ctx, p, X, "1", monkeypatch)
    b, hb = run(ctx, p, X, "0", monkeypatch)
    c, _ = run(ctx, p, X, "", monkeypatch)   # by the list's length: both within one run
    for sa, sb, sc in zip(a, b, c):
        for f in range(3):
            assert np.array_equal(sa[f], sb[f]), (f, np.max(np.abs(sa[f] - sb[f])))
            assert np.array_equal(sc[f], sb[f]), f
        assert np.array_equal(sa[3], sb[3]) and np.array_equal(sc[3], sb[3])
    assert np.array_equal(ha, hb)
    o = OracleSim(p)
    for f, v in enumerate(X):
        o.set_field(f, v)
    o.step(18)
    for f in range(3):
        assert np.max(np.abs(a[-1][f] - o.get_field(f))) <= 1e-10, f
    if mode != abi.MODE_REGULAR:
        assert np.array_equal(a[-1][3], o.awake(0))
        if nx >= 100:
            assert ha[:, 0].min() < nx * ny // 16   # some blocks slept
