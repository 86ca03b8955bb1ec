"""GPU: Model B with r_x, r_y, r_z and 1 - z_crit that are no powers of two, so that the
quotients by them round: the march and the one-plane kernel (whose logarithms are known
to be finite in their usual branch) against the block kernels, bit for bit, and the
oracle, which divides."""
import numpy as np
import pytest

from dba_amd import abi, configs
from oracle.oracle import OracleSim
from test_gpu_modelb_march import run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [abi.MODE_DBA, abi.MODE_CONSERVED])
@pytest.mark.parametrize("shape", [(36, 28, 8), (100, 64, 1)])
@pytest.mark.parametrize("r,z_crit", [((3.0, 7.0, 10.0), 0.3), ((0.7, 1.0, 49.0), 0.05)])
def test_quotients_agree(ctx, mode, shape, r, z_crit, monkeypatch):
    nx, ny, nz = shape
    X = list(configs.modelb_ic(nx, ny, nz)) + [0.05 + 0.3 * configs.uniform01(9, nx * ny * nz).reshape(nz, ny, nx)]
    p = configs.modelb_params(n=nx, nz=nz, mode=mode, eps=1e-4, history_cap=32)
    p.ny = ny
    p.r_x, p.r_y, p.r_z = r
    p.z_crit, p.p_gel = z_crit, 0.7
    p.k_0 = 0.01   # (at 1 the reaction uses up z within two steps at these r)
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
