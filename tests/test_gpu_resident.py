"""The resident solve (one launch, tiles kept in LDS, borders exchanged while sweeping) against
the oracle's FP32 FMM and against the wave loop -- needs an MI355X.

Tolerances: the oracle bar of the parity tests (1e-4 max T, identical INF pattern, fixed-point
gap within 4 ulp + 2 eps); against the wave loop (launch_mode 4), two fixed points of the same
FP32 update whose visiting orders differ: 4e-6 max T, about 32 ulp of the largest time.
"""
import threading

import numpy as np
import pytest

import ghcm_amd as g
import oracle
from conftest import fixed_point_gap3d, ulp32
from test_gpu_parity import check

pytestmark = pytest.mark.gpu
CFG = dict(tile_w=64, tile_h=64, kernel=g.KERNEL_SWEEP, n_active=512, inner_iter_cap=1)


def _field(rng, h, w, obstacles=0.1):
    cost = rng.uniform(0.1, 10.0, (h, w)).astype(np.float32)
    cost[rng.random((h, w)) < obstacles] = np.inf
    return cost


# edges of tiles (63, 64, 65), one row or column, and more tiles than resident work-groups
# (2100 x 2100 has 1,089 tiles; 70000 x 64 and 64 x 70000 have 1,094)
@pytest.mark.parametrize("shape", [(1, 1), (1, 200), (200, 1), (63, 64), (64, 65), (65, 63),
                                   (129, 200), (200, 641), (2100, 2100), (64, 70000), (70000, 64)])
def test_shapes_obstacles_and_corner_seeds(rng, shape):
    h, w = shape
    cost = _field(rng, h, w, 0.1 if min(h, w) > 1 else 0.0)
    seeds = {(0, 0), (w - 1, h - 1), (min(63, w - 1), min(63, h - 1)), (min(64, w - 1), min(64, h - 1)),
             (int(rng.integers(0, w)), int(rng.integers(0, h)))}
    seeds = sorted(seeds)
    for x, y in seeds:
        cost[y, x] = 1.0
    ref = oracle.fmm_f32(cost, seeds)
    print(f"case resident {shape}", flush=True)
    with g.Context(0, **CFG) as ctx:
        for _ in range(2):
            t, st = ctx.solve(cost, seeds)
            assert st["converged"] == 1 and st["waves"] > 0
            check(t, ref, seeds, cost, label=f"resident {shape}")
        ctx.set_config(launch_mode=4)
        tw, _ = ctx.solve(cost, seeds)
    fin = np.isfinite(tw)
    assert np.array_equal(fin, np.isfinite(t))
    assert np.max(np.abs(t[fin] - tw[fin])) <= 4e-6 * float(tw[fin].max()) + 1e-6


@pytest.mark.parametrize("kind", ["speed_f32", "speed_f16", "speed_bf16"])
def test_storage_kinds_and_epsilon_zero(kind):
    speed = g.gen_smooth_speed(333, 270, 9, 12.0, 0.2, 5.0)
    stored = {"speed_f32": speed.astype(np.float32), "speed_f16": speed.astype(np.float16),
              "speed_bf16": g.to_bf16(speed)}[kind]
    back = g.from_bf16(stored) if kind == "speed_bf16" else stored
    cost = g.cost_from_speed(back)
    seeds = g.gen_points(333, 270, 10, 5)
    print(f"case resident {kind}", flush=True)
    with g.Context(0, min_change=0.0, **CFG) as ctx:
        t, _ = ctx.solve(stored, seeds, kind=g.KINDS[kind])
    check(t, oracle.fmm_f32(cost, seeds), seeds, cost, label=kind, eps=0.0)


WAVE_TILES = [(g.KERNEL_SYSTOLIC, (8, 8)), (g.KERNEL_FIM, (8, 8)), (g.KERNEL_SYSTOLIC, (16, 16)),
              (g.KERNEL_FIM, (16, 16)), (g.KERNEL_SYSTOLIC, (32, 8)), (g.KERNEL_SYSTOLIC, (32, 32))]


# one cell, edges of tiles, and for 8x8 tiles the most that fit (8,184) and more (wave loop)
@pytest.mark.parametrize("kernel,tile", WAVE_TILES)
@pytest.mark.parametrize("shape", [(1, 1), (1, 130), (7, 9), (8, 33), (17, 64), (129, 200), (720, 720), (744, 704), (744, 712)])
def test_one_wave_tiles(rng, kernel, tile, shape):
    h, w = shape
    cost = _field(rng, h, w, 0.1 if min(h, w) > 1 else 0.0)
    seeds = sorted({(0, 0), (w - 1, h - 1), (min(7, w - 1), min(7, h - 1)), (min(8, w - 1), min(8, h - 1)),
                    (int(rng.integers(0, w)), int(rng.integers(0, h)))})
    for x, y in seeds:
        cost[y, x] = 1.0
    ref = oracle.fmm_f32(cost, seeds)
    print(f"case resident kernel={kernel} tile={tile} {shape}", flush=True)
    with g.Context(0, tile_w=tile[0], tile_h=tile[1], kernel=kernel) as ctx:
        for _ in range(2):
            t, st = ctx.solve(cost, seeds)
            assert st["converged"] == 1 and st["waves"] > 0
            check(t, ref, seeds, cost, label=f"{kernel} {tile} {shape}")


@pytest.mark.parametrize("kind", ["speed_f32", "speed_f16", "speed_bf16"])
def test_one_wave_tiles_storage_and_batch(rng, kind):
    """Several instances, stored as speed, at eps = 0; hundreds of sources in one of them."""
    speeds = [g.gen_smooth_speed(w, h, 3 + w, 8.0, 0.2, 5.0) for w, h in ((100, 90), (33, 150), (8, 8))]
    stored = [{"speed_f32": s.astype(np.float32), "speed_f16": s.astype(np.float16),
               "speed_bf16": g.to_bf16(s) if kind == "speed_bf16" else None}[kind] for s in speeds]
    costs = [g.cost_from_speed(g.from_bf16(s) if kind == "speed_bf16" else s) for s in stored]
    seeds = [[(5, 5), (99, 89)], g.gen_points(33, 150, 4, 300), [(3, 4)]]
    print(f"case resident one-wave {kind}", flush=True)
    with g.Context(0, min_change=0.0) as ctx:
        dev = [(ctx.to_device(s), ctx.alloc(s.shape, np.float32)) for s in stored]
        st = ctx.solve_batch(g.KINDS[kind], [(d.ptr, t.ptr, s.shape[1], s.shape[0], q)
                                             for (d, t), s, q in zip(dev, stored, seeds)])
        assert st["converged"] == 1
        for (d, t), c, q in zip(dev, costs, seeds):
            check(t.download(), oracle.fmm_f32(c, q), q, c, label=f"{kind} {c.shape}", eps=0.0)
            d.free()
            t.free()


# partial tiles in each axis, one cell, one tile row; 511 and 513 tiles (512 fit: above, wave loop)
@pytest.mark.parametrize("kind", ["cost", "speed_f16"])
@pytest.mark.parametrize("shape", [(1, 1, 1), (5, 3, 64), (8, 8, 65), (9, 17, 130), (30, 41, 70), (56, 584, 5), (24, 1368, 7)])
def test_volumes(rng, shape, kind):
    speed = rng.uniform(0.2, 5.0, shape)
    stored = speed.astype(np.float16) if kind == "speed_f16" else (1.0 / speed).astype(np.float32)
    cost = (1.0 / stored.astype(np.float32)).astype(np.float32) if kind == "speed_f16" else stored
    d, h, w = shape
    seeds = sorted({(0, 0, 0), (w - 1, h - 1, d - 1), (min(63, w - 1), min(7, h - 1), min(8, d - 1))})
    print(f"case resident volume {shape} {kind}", flush=True)
    ref = oracle.fmm3d_f64(cost, seeds)
    with g.Context(0, **dict(CFG, n_active=2048)) as ctx:
        for _ in range(2):
            t, st = ctx.solve3d(stored, seeds, kind=g.KINDS[kind])
            assert st["converged"] == 1
            assert np.array_equal(np.isfinite(t), np.isfinite(ref))
            # 1e-4 max T as in the 3-D parity tests, plus the least change that counts
            assert float(np.max(np.abs(t - ref))) <= 1e-4 * float(ref.max()) + 1e-5
            gap = fixed_point_gap3d(t, cost, seeds)
            assert np.all(gap <= 4 * ulp32(t) + 2e-5), gap.max()


def test_no_seeds_and_walled_off_tiles():
    cost = np.ones((300, 300), np.float32)
    with g.Context(0, **CFG) as ctx:
        t, st = ctx.solve(cost, np.zeros((0, 2), np.uint32))
        assert np.all(np.isinf(t)) and st["converged"] == 1
        cost[:, 70] = np.inf
        t, _ = ctx.solve(cost, [(3, 3)])
    assert np.all(np.isinf(t[:, 70:]))
    check(t, oracle.fmm_f32(cost, [(3, 3)]), [(3, 3)], cost)


@pytest.mark.parametrize("n_inst", [7, 160, 600, 900])
def test_uneven_batch(rng, n_inst):
    """Several instances in one resident launch; 160 of them have more tiles than work-groups
    (which scan the borders of their closed tiles), 600 about eleven tiles to each, 900 over 16
    (which are told)."""
    shapes = [(int(rng.integers(1, 300)), int(rng.integers(1, 300))) for _ in range(n_inst - 1)] + [(300, 1400)]
    if n_inst > 100:
        shapes = [(h + 100, w + 100) for h, w in shapes]
    costs = [_field(rng, h, w, 0.05) for h, w in shapes]
    seeds = []
    for c in costs:
        s = [(int(rng.integers(0, c.shape[1])), int(rng.integers(0, c.shape[0]))) for _ in range(3)]
        for x, y in s:
            c[y, x] = 1.0
        seeds.append(s)
    print(f"case resident batch {n_inst}", flush=True)
    with g.Context(0, **dict(CFG, n_active=65536)) as ctx:
        dev = [(ctx.to_device(c), ctx.alloc(c.shape, np.float32)) for c in costs]
        st = ctx.solve_batch(g.FIELD_COST_F32, [(d.ptr, t.ptr, c.shape[1], c.shape[0], s)
                                                for (d, t), c, s in zip(dev, costs, seeds)])
        assert st["converged"] == 1
        for (d, t), c, s in zip(dev, costs, seeds):
            check(t.download(), oracle.fmm_f32(c, s), s, c, label=f"batch {c.shape}")
            d.free()
            t.free()


def test_contexts_in_threads():
    """Three contexts solve 2048^2 at once, repeatedly: each wants the whole chip, so launches
    wait for one another or give way to the wave loop; every result is the same."""
    speed = g.gen_smooth_speed(2048, 2048, 3, 32.0, 0.1, 10.0)
    cost = g.cost_from_speed(speed)
    seeds = g.gen_points(2048, 2048, 4, 3)
    ref = oracle.fmm_f32(cost, seeds)
    out, errs = {}, []

    def work(i):
        try:
            with g.Context(0, **CFG) as ctx:
                for _ in range(3):
                    out[i] = ctx.solve(cost, seeds)[0]
        except Exception as e:      # noqa: BLE001
            errs.append(e)

    print("case resident threads", flush=True)
    ts = [threading.Thread(target=work, args=(i,)) for i in range(3)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not errs, errs
    for i in range(3):
        check(out[i], ref, seeds, cost, label=f"thread {i}")
