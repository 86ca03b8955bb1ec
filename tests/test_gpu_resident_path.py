"""GPU: which step calls take resident steps, and the single-launch steps of the same
instances.

A call takes resident steps only if it has at least 12 steps, one CH or K93 instance
that fits the chip, no workgroup size of its own, no timing, and a context alone on its
device; the counter says so, so that a test of them cannot pass on another path. The
single-launch kernels stay the path of every other call: with resident steps off, the
long runs (replayed chunks and eager remainders) are compared with the worklist."""
import numpy as np
import pytest

from dba_amd import Context, abi, configs
from test_gpu_resident import patchy, run, same
from test_gpu_single_launch import ch_case, k93_run
from test_gpu_single_launch import run as ch_run

pytestmark = pytest.mark.gpu


@pytest.fixture
def launched_steps(ctx):
    """The session's context without resident steps."""
    ctx.set_resident(False)
    yield ctx
    ctx.set_resident(True)


def k93_fields(nx, ny):
    return list(configs.dendrite_k93_ic(nx, ny, seeds=[(nx // 2, ny // 3)]))


def ch_params(nx, ny, tile, **kw):
    return configs.ch_params(n=nx, ny=ny, tile=tile, eps=1e-3, react_gamma=0.01, cbar=0.05, history_cap=128, **kw)


# CH: the region shapes of each tile size, partial tiles, and one grid past the largest;
# K93: 512^2 is the largest on 16 x 16 tiles
@pytest.mark.parametrize("model,nx,ny,tile,fits", [
    ("ch", 64, 66, 32, True), ("ch", 1024, 1024, 32, True), ("ch", 1200, 1100, 32, True), ("ch", 1534, 1310, 32, True),
    ("ch", 900, 700, 16, True), ("ch", 514, 480, 8, True), ("ch", 1600, 1570, 32, False), ("ch", 1100, 1040, 16, False),
    ("k93", 256, 256, 16, True), ("k93", 512, 512, 16, True), ("k93", 514, 480, 8, True), ("k93", 500, 500, 32, True),
    ("k93", 700, 1000, 16, False)])
def test_calls_that_take_resident_steps(ctx, model, nx, ny, tile, fits):
    if model == "ch":
        p, fields = ch_params(nx, ny, tile), [patchy(nx, ny, tile)]
    else:
        p, fields = configs.dendrite_k93_params(n=nx, ny=ny, tile=tile, history_cap=128), k93_fields(nx, ny)
    n0 = ctx.resident_calls()
    run(ctx, p, fields, 1, (11,))
    assert ctx.resident_calls() == n0
    run(ctx, p, fields, 1, (12, 40, 3))
    assert ctx.resident_calls() == n0 + (2 if fits else 0)
    run(ctx, p, fields, 2, (30,))
    assert ctx.resident_calls() == n0 + (3 if fits else 0)


def test_calls_that_do_not(ctx):
    c0 = patchy(512, 512, 32)
    n0 = ctx.resident_calls()
    run(ctx, ch_params(512, 512, 32), c0, 0, (20,))                       # the worklist path
    run(ctx, ch_params(512, 512, 32, threads=256), c0, 1, (20,))          # a workgroup size of its own
    run(ctx, ch_params(512, 512, 32, mode=abi.MODE_CONSERVED), c0, 1, (20,))
    a, b = (ctx.create(ch_params(512, 512, 32)) for _ in range(2))
    for inst in (a, b):
        inst.upload(0, c0)
    ctx.step([a, b], 20)                                                  # two instances
    ctx.timing(True)
    a.step(20)
    ctx.timing(False)
    ctx.set_resident(False)
    a.step(20)
    ctx.set_resident(True)
    with Context(0) as other:                                             # a second context on the device
        run(other, ch_params(512, 512, 32), c0, 1, (20,))
        a.step(20)
        ctx.sync()
        assert other.resident_calls() == 0
    assert ctx.resident_calls() == n0
    a.step(20)                                                            # alone again
    assert ctx.resident_calls() == n0 + 1
    b.step(60)
    assert ctx.resident_calls() == n0 + 2
    assert np.array_equal(a.history()[:80], b.history()[:80]) and a.info().steps_done == 100
    for inst in (a, b):
        inst.destroy()


@pytest.mark.parametrize("tile,stencil,bc,mode", [
    (32, 9, "periodic", abi.MODE_DBA), (16, 5, "periodic", abi.MODE_DBA), (8, 9, "noflux", abi.MODE_DBA),
    (16, 9, "periodic", abi.MODE_REGULAR)])
def test_ch_single_launch_equals_worklist(launched_steps, tile, stencil, bc, mode):
    ctx, n0 = launched_steps, launched_steps.resident_calls()
    p, c = ch_case(16 * tile, tile, mode, stencil, bc)
    plan = [(1, 0), (7, 0), (100, 25), (37, 10), (40, 0)]
    a, b = (ch_run(ctx, p, c, single, plan) for single in (False, True))
    assert ctx.resident_calls() == n0
    for k in ("c", "hist", "work"):
        assert np.array_equal(a[k], b[k]), k
    assert all(np.array_equal(x, y) for x, y in zip(a["masks"], b["masks"]))
    assert (a["steps"], a["updates"], a["time"]) == (b["steps"], b["updates"], b["time"])


def test_ch_several_segments_single_launch_equals_worklist(launched_steps):
    p, c = ch_case(1024, 16, abi.MODE_DBA, 9, "periodic")   # 4096 tiles, four segments
    plan = [(1, 0), (6, 0), (40, 20), (30, 0)]
    a, b = (ch_run(launched_steps, p, c, single, plan) for single in (False, True))
    for k in ("c", "hist", "work"):
        assert np.array_equal(a[k], b[k]), k
    assert all(np.array_equal(x, y) for x, y in zip(a["masks"], b["masks"]))
    assert (a["steps"], a["updates"], a["time"]) == (b["steps"], b["updates"], b["time"])


# 16 x 16 tiles at the default thread count: speculative staging, for more than 100 steps
@pytest.mark.parametrize("n,tile,mode,bc", [
    (256, 16, abi.MODE_DBA, abi.BC_NOFLUX), (512, 16, abi.MODE_DBA, abi.BC_NOFLUX), (256, 8, abi.MODE_DBA, abi.BC_NOFLUX),
    (256, 32, abi.MODE_DBA, abi.BC_NOFLUX), (256, 16, abi.MODE_REGULAR, abi.BC_NOFLUX),
    (256, 16, abi.MODE_DBA, abi.BC_PERIODIC)])
def test_k93_single_launch_equals_worklist(launched_steps, n, tile, mode, bc):
    ctx, n0 = launched_steps, launched_steps.resident_calls()
    p = configs.dendrite_k93_params(n=n, tile=tile, mode=mode, history_cap=400, bc=bc)
    phi, T = configs.dendrite_k93_ic(n, n, seeds=[(90, 100), (170, 150)])
    plan = [(1, 0), (9, 0), (150, 50), (33, 10), (120, 0)]
    a, b = (k93_run(ctx, p, phi, T, single, plan) for single in (False, True))
    assert ctx.resident_calls() == n0
    for k in ("phi", "T", "hist", "work"):
        assert np.array_equal(a[k], b[k]), k
    assert all(np.array_equal(x, y) for sa, sb in zip(a["masks"], b["masks"]) for x, y in zip(sa, sb))
    assert (a["steps"], a["updates"], a["time"]) == (b["steps"], b["updates"], b["time"])


def test_resident_and_single_launch_agree(ctx):
    """The same run on both, bit for bit."""
    p, c0 = ch_params(1024, 1024, 32), patchy(1024, 1024, 32)
    a = run(ctx, p, c0, 1)
    ctx.set_resident(False)
    try:
        b = run(ctx, p, c0, 1)
    finally:
        ctx.set_resident(True)
    same(a, b)


def test_instances_of_several_region_shapes(ctx):
    """One kernel serves regions of different sizes: instances of each, stepped in turn,
    keep their resident steps (the largest LDS a launch may ask for belongs to the kernel)."""
    sizes = [(1534, 1310), (1024, 1024), (1200, 1100), (600, 1000)]   # 3 x 3, 2 x 2, 3 x 2 and single tiles
    insts = []
    for k, (nx, ny) in enumerate(sizes):
        inst = ctx.create(ch_params(nx, ny, 32))
        inst.upload(0, patchy(nx, ny, 32, seed=k))
        insts.append(inst)
    n0 = ctx.resident_calls()
    for order in (insts, insts[::-1], insts):
        for inst in order:
            inst.step(16)
    assert ctx.resident_calls() == n0 + 12
    for inst in insts:
        assert inst.info().steps_done == 48
        inst.destroy()
