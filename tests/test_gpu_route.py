"""Which solves are resident, what those do that are given up, and the wave loop at configurations
whose default is resident -- needs an MI355X with 256 CUs.

With profile_kernels a resident solve reports one launch, a solve by waves one per wave."""
import numpy as np
import pytest

import ghcm_amd as g
import oracle
from conftest import fixed_point_gap3d, ulp32
from test_gpu_parity import check

pytestmark = pytest.mark.gpu
BY_WAVES = dict(max_waves=1_000_000)
SWEEP = dict(tile_w=64, tile_h=64, kernel=g.KERNEL_SWEEP, n_active=512, inner_iter_cap=1)
TILE = {"8x8": {}, "8x8 fim": dict(kernel=g.KERNEL_FIM), "16x16": dict(tile_w=16, tile_h=16),
        "16x16 fim": dict(tile_w=16, tile_h=16, kernel=g.KERNEL_FIM), "32x8": dict(tile_w=32, tile_h=8),
        "32x32": dict(tile_w=32, tile_h=32), "sweep": SWEEP, "volume": dict(SWEEP, n_active=2048)}


def _solve(ctx, cost, seeds):
    return (ctx.solve3d if cost.ndim == 3 else ctx.solve)(cost, seeds)


def _check(t, cost, seeds, label):
    if cost.ndim == 2:
        return check(t, oracle.fmm_f32(cost, seeds), seeds, cost, label=label)
    ref = oracle.fmm3d_f64(cost, seeds)
    assert float(np.max(np.abs(t - ref))) <= 1e-4 * float(ref.max()) + 1e-5
    assert np.all(fixed_point_gap3d(t, cost, seeds) <= 4 * ulp32(t) + 2e-5)


# the most tiles that are resident (one-wave tiles: eight, six and two waves to a SIMD, less the
# work-group that watches; volumes two work-groups to a CU) and one more or one row more
ROUTES = [("8x8", (744, 704), True), ("8x8", (744, 712), False), ("8x8 fim", (744, 704), True),
          ("16x16", (944, 1664), True), ("16x16", (1248, 1264), False), ("16x16 fim", (944, 1664), True),
          ("32x8", (472, 3328), True), ("32x8", (480, 3328), False),
          ("32x32", (1280, 1632), True), ("32x32", (1312, 1632), False),
          ("sweep", (1, 1), True), ("sweep", (2048, 2048), True), ("sweep", (2049, 2049), True),
          ("sweep", (6000, 5000), True), ("volume", (64, 64, 512), True), ("volume", (24, 1368, 7), False)]


@pytest.mark.parametrize("tiles,shape,resident", ROUTES)
def test_route(tiles, shape, resident):
    cost = np.ones(shape, np.float32)
    seeds = [(0,) * len(shape)]
    print(f"case route {tiles} {shape}", flush=True)
    with g.Context(0, profile_kernels=1, **TILE[tiles]) as ctx:
        _, st = _solve(ctx, cost, seeds)
        assert (st["solve_launches"] == 1) == resident, st
        ctx.set_config(**BY_WAVES)
        if st["tiles_total"] > 1:
            assert _solve(ctx, cost, seeds)[1]["solve_launches"] > 1


@pytest.mark.parametrize("change", [dict(n_active=64), dict(launch_mode=4), dict(scheduler=g.SCHED_HOST_PQ)])
def test_configurations_that_go_by_waves(change):
    cost = np.ones((500, 500), np.float32)
    with g.Context(0, **dict(dict(SWEEP, profile_kernels=1), **change)) as ctx:
        _, st = ctx.solve(cost, [(3, 3)])
    assert st["solve_launches"] > 1


GIVEN_UP = [("8x8", (200, 300)), ("16x16 fim", (200, 300)), ("32x8", (200, 300)), ("32x32", (200, 300)),
            ("sweep", (200, 300)), ("sweep", (2300, 2100)), ("volume", (20, 40, 70))]


@pytest.mark.parametrize("n_seeds", [3, 3000])
@pytest.mark.parametrize("tiles,shape", GIVEN_UP)
def test_given_up_solves_go_by_waves(rng, tiles, shape, n_seeds):
    cost = rng.uniform(0.2, 5.0, shape).astype(np.float32)
    seeds = np.stack([rng.integers(0, n, n_seeds) for n in shape[::-1]], 1).astype(np.uint32)
    print(f"case given up {tiles} {shape}", flush=True)
    with g.Context(0, profile_kernels=1, **TILE[tiles]) as ctx:
        for refuse in (True, False, True):
            ctx.debug_refuse_resident(refuse)
            t, st = _solve(ctx, cost, seeds)
            assert st["converged"] == 1 and (st["solve_launches"] == 1) == (not refuse), st
            _check(t, cost, seeds, f"{tiles} {shape} {refuse}")


def test_given_up_batch(rng):
    costs = [rng.uniform(0.1, 10.0, (int(rng.integers(60, 300)), 200)).astype(np.float32) for _ in range(150)]
    with g.Context(0, profile_kernels=1, **dict(SWEEP, n_active=65536)) as ctx:
        dev = [(ctx.to_device(c), ctx.alloc(c.shape, np.float32)) for c in costs]
        prepared = ctx.prepare_batch([(d.ptr, t.ptr, c.shape[1], c.shape[0], [(5, 5), (190, 50)])
                                      for (d, t), c in zip(dev, costs)])
        for refuse in (True, False):
            ctx.debug_refuse_resident(refuse)
            st = ctx.solve_batch(g.FIELD_COST_F32, prepared)
            assert st["converged"] == 1 and (st["solve_launches"] == 1) == (not refuse)
            for (_, t), c in zip(dev, costs):
                seeds = [(5, 5), (190, 50)]
                check(t.download(), oracle.fmm_f32(c, seeds), seeds, c)


# The wave loop where the default route is resident: every tile kernel of launch_mode 0.
@pytest.mark.parametrize("tiles", list(TILE))
@pytest.mark.parametrize("eps", [1e-5, 0.0])
def test_by_waves(rng, tiles, eps):
    shape = (9, 41, 130) if tiles == "volume" else (129, 333)
    cost = rng.uniform(0.1, 10.0, shape).astype(np.float32)
    seeds = sorted({(0,) * len(shape), tuple(n - 1 for n in shape[::-1]), tuple(n // 2 for n in shape[::-1])})
    with g.Context(0, min_change=eps, **dict(TILE[tiles], **BY_WAVES)) as ctx:
        t, st = _solve(ctx, cost, seeds)
    assert st["converged"] == 1
    _check(t, cost, seeds, f"{tiles} by waves")
