"""GPU: the KH step at the edges of the range its short divisions and square
roots hold in (densities and pressures in [2^-60, 2^60), velocities 0 or of
magnitude [2^-150, 2^60)), inside it and beyond, where a tile falls back to the
plain divisions, against the oracle.

Bar: bit-identical conserved fields (NaN where the oracle has NaN): both sides
round every operation correctly, whatever sequence computes it."""
import numpy as np
import pytest

from dba_amd import abi, configs
from oracle.oracle import OracleSim

pytestmark = pytest.mark.gpu


def fields(kind, n, dx, g):
    rho, u, v, p = configs.kh_primitive(configs.kh_reference_ic(n, dx=dx), g, dx * dx)
    patch = (slice(n // 4, n // 4 + 12), slice(n // 2, n // 2 + 12))   # part of several tiles
    if kind == "small":            # densities and pressures below 2^-60: every tile falls back
        rho, p = rho * 2.0 ** -70, p * 2.0 ** -70
    elif kind == "edge":           # a little above 2^-60
        rho, p = rho * 2.0 ** -58, p * 2.0 ** -58
    elif kind == "large":          # above 2^60
        rho, p = rho * 2.0 ** 62, p * 2.0 ** 62
    elif kind == "still":          # v exactly 0 in a patch, and below 2^-150 in another
        v = v.copy()
        v[patch] = 0.0
        v[n // 2:n // 2 + 9, 3:17] = 1e-60
    elif kind == "vacuum":         # a patch of almost no pressure: face values cancel to nothing and below
        p = p.copy()
        p[patch] = 1e-3
        rho = rho.copy()
        rho[patch] = 1e-2
    elif kind == "overflow":       # a cell without a finite energy
        p = p.copy()
        p[n // 3, n // 3] = np.inf
    return configs.kh_conserved(rho, u, v, p, g, dx * dx)


@pytest.mark.parametrize("dx", [1.0 / 64, 0.003])          # exact reciprocals of the spacing, and divisions by it
@pytest.mark.parametrize("tile", [8, 16])
@pytest.mark.parametrize("kind", ["plain", "small", "edge", "large", "still", "vacuum", "overflow"])
def test_kh_ranges_match_oracle(ctx, kind, tile, dx):
    n, g = 64, 5.0 / 3.0
    p = configs.kh_reference_params(n=n, tile=tile, mode=abi.MODE_DBA, dx=dx, dt=2e-4, eps=2.0, history_cap=16)
    U = fields(kind, n, dx, g)
    inst = ctx.create(p)
    o = OracleSim(p)
    for f in range(4):
        inst.upload(f, U[f])
        o.set_field(f, U[f])
    steps = 3 if kind == "overflow" else 8
    with np.errstate(all="ignore"):
        for _ in range(steps):
            inst.step(1)
            o.step(1)
            for f in range(4):
                a, b = inst.download(f), o.get_field(f)
                assert np.array_equal(a, b, equal_nan=True), (kind, f)
            assert np.array_equal(inst.active(0)[1], o.awake(0))
    inst.destroy()
