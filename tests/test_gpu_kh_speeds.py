"""GPU: the CFL time step of a KH state none of whose cells has a wave speed (pressures
below 0, or no numbers at all).

A speed that is no number does not count, as in fmax: with none left the largest speed
is 0 and the time step infinite, on every step, whatever the number of tiles (1024 fill
one segment of the end-of-step kernel to its last lane)."""
import numpy as np
import pytest

from dba_amd import abi, configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tile,n", [(8, 256), (8, 64), (16, 512), (16, 528)])
def test_no_speed_counts_as_none(ctx, tile, n):
    p = configs.kh_params(n=n, tile=tile)
    assert p.dt_mode == abi.DT_CFL
    inst = ctx.create(p)
    for f in range(4):
        inst.upload(f, np.full((n, n), np.nan))
    for _ in range(3):
        inst.step(1)
        assert inst.info().last_dt == np.inf and inst.info().sim_time == np.inf
    inst.destroy()
