"""The work whose time matters: eikonal solves as a user of this package makes them.

``listed()`` holds fixed cases, ``draw(rng)`` makes more of the same ranges; ``prepare`` builds
what a program holds before the call (fields, sources, output buffers, a context or a server),
``run`` is one call through the public entry points, ``work`` the bytes and operations that the
call cannot do without, and ``exact`` the solution of the same discrete system in 64 bits.

A case is a dict of plain values:

    path    "solve"  Context.solve_device     one 2-D field resident in device memory
            "host"   Context.solve            one 2-D field in host memory, times back to it
            "batch"  Context.solve_batch      many uneven 2-D fields in one call
            "serve"  Server.submit_device     many requests to a running server, all awaited
            "volume" Context.solve3d_device   one 3-D field resident in device memory
    w h d   size in cells (batch and serve: lo, hi and n, the range of sides and the count)
    field   "smooth" log-normal speed in [0.1, 10], or "ring", seven walls with one gap each,
            or "mixed" (batch and serve: either, instance by instance)
    wall    speed of the ring walls
    store   "cost" (FP32 cost), "speed_f32", "speed_f16" or "speed_bf16"
    sources point sources (batch and serve: up to that many)
    tiles   "sweep" 64 x 64 tiles by fast sweeping (the configuration of the benchmark),
            "default" Config() as it stands (8 x 8 systolic tiles), "fim" 16 x 16 FIM tiles

torch is imported before the package: the solver then shares torch's HIP runtime.
"""
import functools
import math
import random

import numpy as np
import torch

import ghcm_amd as g

DEV = "cuda"
CONFIGS = {
    "sweep": dict(tile_w=64, tile_h=64, kernel=g.KERNEL_SWEEP, n_active=512, inner_iter_cap=1),
    "default": dict(),
    "fim": dict(tile_w=16, tile_h=16, kernel=g.KERNEL_FIM),
    # many instances at once: every queued tile of a wave is solved in it
    "wide": dict(tile_w=64, tile_h=64, kernel=g.KERNEL_SWEEP, n_active=65536, inner_iter_cap=1),
    "volume": dict(tile_w=64, tile_h=64, kernel=g.KERNEL_SWEEP, n_active=2048, inner_iter_cap=1),
}
DTYPES = {"cost": torch.float32, "speed_f32": torch.float32, "speed_f16": torch.float16,
          "speed_bf16": torch.bfloat16}


def listed():
    return [
        # the smallest call: one maze of ring walls, the reference's own demo size
        dict(name="ring-256", path="solve", w=256, h=256, field="ring", wall=1e-3, store="cost",
             sources=1, tiles="sweep"),
        # an ordinary grid whose sides are no multiple of anything, stored as bfloat16
        dict(name="smooth-1531x977-bf16", path="solve", w=1531, h=977, field="smooth", wall=0.0,
             store="speed_bf16", sources=3, tiles="sweep"),
        # the benchmark's headline: one large smooth field, four sources
        dict(name="smooth-4096", path="solve", w=4096, h=4096, field="smooth", wall=0.0,
             store="cost", sources=4, tiles="sweep"),
        # strong contrast: the front winds through the gaps of seven walls; half precision
        dict(name="contrast-2048-f16", path="solve", w=2048, h=2048, field="ring", wall=1e-4,
             store="speed_f16", sources=1, tiles="sweep"),
        # a caller whose fields live in host memory: in over PCIe, solved, and back
        dict(name="host-2048", path="host", w=2048, h=2048, field="smooth", wall=0.0, store="cost",
             sources=2, tiles="sweep"),
        # the drop-in caller that changes nothing: default configuration, host buffers
        dict(name="dropin-512", path="host", w=512, h=512, field="ring", wall=1e-3, store="cost",
             sources=1, tiles="default"),
        # the other reference tile algorithm at one of its usual block sizes
        dict(name="fim-640x384", path="solve", w=640, h=384, field="smooth", wall=0.0,
             store="cost", sources=2, tiles="fim"),
        # the benchmark's batch: 512 uneven instances, sides 64..2048
        dict(name="batch-512", path="batch", lo=64, hi=2048, n=512, field="mixed", wall=1e-3,
             store="cost", sources=8, tiles="wide"),
        # a small batch of small uneven instances
        dict(name="batch-48-small", path="batch", lo=64, hi=448, n=48, field="mixed", wall=1e-3,
             store="speed_f32", sources=4, tiles="wide"),
        # requests handed to a running server all at once
        dict(name="serve-64", path="serve", lo=128, hi=1536, n=64, field="mixed", wall=1e-3,
             store="cost", sources=4, tiles="wide"),
        # the 3-D benchmark volume
        dict(name="volume-256", path="volume", w=256, h=256, d=256, field="smooth", wall=0.0,
             store="cost", sources=4, tiles="volume"),
        # a small ragged volume in half precision
        dict(name="volume-150x90x61-f16", path="volume", w=150, h=90, d=61, field="smooth",
             wall=0.0, store="speed_f16", sources=2, tiles="volume"),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["solve", "solve", "solve", "host", "tiles", "batch", "serve", "volume"])
    store = rng.choice(list(DTYPES))
    field = rng.choice(["smooth", "ring"])
    wall = rng.choice([1e-3, 1e-4]) if field == "ring" else 0.0
    if path == "solve":
        return dict(path="solve", w=_log_uniform(rng, 150, 4000), h=_log_uniform(rng, 150, 4000),
                    field=field, wall=wall, store=store, sources=rng.randint(1, 8), tiles="sweep")
    if path == "host":
        return dict(path="host", w=_log_uniform(rng, 200, 2500), h=_log_uniform(rng, 200, 2500),
                    field=field, wall=wall, store="cost", sources=rng.randint(1, 4), tiles="sweep")
    if path == "tiles":
        return dict(path=rng.choice(["solve", "host"]), w=_log_uniform(rng, 100, 800),
                    h=_log_uniform(rng, 100, 800), field=field, wall=wall, store="cost",
                    sources=rng.randint(1, 4), tiles=rng.choice(["default", "fim"]))
    if path in ("batch", "serve"):
        hi = rng.randint(200, 1500)
        return dict(path=path, lo=rng.randint(40, 150), hi=hi, n=_log_uniform(rng, 8, 120),
                    field="mixed", wall=1e-3, store=store, sources=rng.randint(1, 8), tiles="wide")
    return dict(path="volume", w=_log_uniform(rng, 40, 256), h=_log_uniform(rng, 40, 220),
                d=_log_uniform(rng, 20, 200), field="smooth", wall=0.0, store=store,
                sources=rng.randint(1, 4), tiles="volume")


# ---- inputs --------------------------------------------------------------------------------

def _blur_matrix(n, sigma):
    """(n, n) Gaussian filter of `sigma` cells with a half-sample reflecting boundary."""
    radius = int(4 * sigma + 0.5)
    k = torch.arange(-radius, radius + 1, device=DEV)
    wt = torch.exp(-0.5 * (k.double() / sigma) ** 2)
    wt = (wt / wt.sum()).float()
    m = (torch.arange(n, device=DEV)[:, None] + k[None, :]) % (2 * n)
    m = torch.where(m < n, m, 2 * n - 1 - m)
    return torch.zeros(n, n, device=DEV).scatter_add_(1, m, wt.expand(n, -1).contiguous())


def _lognormal(z):
    """Speed in [0.1, 10], log-linear in z."""
    lo, hi = z.min(), z.max()
    return torch.pow(10.0, -1.0 + 2.0 * (z - lo) / (hi - lo))


def _smooth(w, h, seed, sigma=32.0):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    z = torch.randn(h, w, generator=gen, device=DEV)
    right = _blur_matrix(w, sigma).t().contiguous()
    return _lognormal(_blur_matrix(h, sigma) @ (z @ right))


def _smooth3(w, h, d, seed, sigma=8.0):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    z = torch.randn(d, h, w, generator=gen, device=DEV)
    z = (z.reshape(d * h, w) @ _blur_matrix(w, sigma).t().contiguous()).reshape(d, h, w)
    z = z.transpose(1, 2).contiguous().reshape(d * w, h) @ _blur_matrix(h, sigma).t().contiguous()
    z = z.reshape(d, w, h).transpose(1, 2).contiguous()
    z = _blur_matrix(d, sigma) @ z.reshape(d, h * w)
    return _lognormal(z.reshape(d, h, w))


def _ring(w, h, seed, wall):
    """Seven circular walls around the centre, each with one gap, on a background of speed 1."""
    rng = random.Random(seed)
    scale = min(w, h) / 256.0
    y = torch.arange(h, device=DEV, dtype=torch.float32)[:, None] - h // 2
    x = torch.arange(w, device=DEV, dtype=torch.float32)[None, :] - w // 2
    r, ang = torch.sqrt(x * x + y * y), torch.atan2(y, x)
    speed = torch.ones(h, w, device=DEV)
    for k in range(7):
        radius, theta = scale * (16.0 + k * 104.0 / 6.0), rng.uniform(-math.pi, math.pi)
        da = torch.abs(ang - theta)
        da = torch.minimum(da, 2 * math.pi - da)
        speed[(torch.abs(r - radius) < 1.5 * scale) & (da >= 3.0 * scale / radius)] = wall
    return speed


def _stored(speed, store):
    return 1.0 / speed if store == "cost" else speed.to(DTYPES[store])


def _one(case, seed):
    """(field, sources) of a single-field case."""
    rng = random.Random(seed)
    w, h, d = case["w"], case["h"], case.get("d", 0)
    if d:
        speed = _smooth3(w, h, d, seed)
        pts = [(rng.randrange(w), rng.randrange(h), rng.randrange(d)) for _ in range(case["sources"])]
    else:
        speed = _smooth(w, h, seed) if case["field"] == "smooth" else _ring(w, h, seed, case["wall"])
        pts = [(rng.randrange(w), rng.randrange(h)) for _ in range(case["sources"])]
        if case["field"] == "ring" and case["sources"] == 1:
            pts = [(w // 2, h // 2)]
    return _stored(speed, case["store"]), np.array(pts, dtype=np.uint32)


def _shapes(case):
    """Sides of a batch's or a server's instances: the case alone decides them."""
    rng = random.Random(repr(sorted((k, v) for k, v in case.items() if k != "name")))
    lo, hi = case["lo"], case["hi"]
    even = lo % 64 == 0 and hi % 64 == 0
    out = []
    for _ in range(case["n"]):
        w, h = rng.randint(lo, hi), rng.randint(lo, hi)
        if case["path"] == "serve":
            w = h = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
        out.append((-(-w // 64) * 64, -(-h // 64) * 64) if even else (w, h))
    return out


def _many(case, seed):
    """[(field, w, h, sources)] of a batch or serve case."""
    rng = random.Random(seed)
    out = []
    for i, (w, h) in enumerate(_shapes(case)):
        s = seed * 1009 + i
        speed = _ring(w, h, s, case["wall"]) if rng.random() < 0.5 else _smooth(w, h, s)
        pts = [(rng.randrange(w), rng.randrange(h)) for _ in range(rng.randint(1, case["sources"]))]
        out.append((_stored(speed, case["store"]), w, h, np.array(pts, dtype=np.uint32)))
    return out


# ---- the handles a program keeps ------------------------------------------------------------

@functools.lru_cache(maxsize=None)
def _context(tiles):
    return g.Context(0, **CONFIGS[tiles])


@functools.lru_cache(maxsize=None)
def _server(kind):
    return g.Server(0, kind=kind, hbm_budget_bytes=2 << 30, **CONFIGS["wide"])


def prepare(case, seed):
    kind, path = g.KINDS[case["store"]], case["path"]
    state = dict(case=case, kind=kind)
    if path in ("batch", "serve"):
        many = _many(case, seed)
        # the times of all instances in one allocation, each from a 256-byte boundary
        at, total = [], 0
        for _, w, h, _ in many:
            at.append(total)
            total += -(-w * h // 64) * 64
        times = torch.zeros(total, device=DEV)
        calls = [(f.data_ptr(), times.data_ptr() + 4 * o, w, h, s) for (f, w, h, s), o in zip(many, at)]
        state.update(keep=many, times=times, calls=calls)
        if path == "batch":
            state["ctx"] = _context(case["tiles"])
            state["prepared"] = state["ctx"].prepare_batch(calls)
        else:
            state["server"] = _server(kind)
    else:
        field, seeds = _one(case, seed)
        state.update(ctx=_context(case["tiles"]), seeds=seeds)
        if path == "host":
            state["field"] = field.cpu().numpy()
        else:
            state.update(field=field, times=torch.zeros(field.shape, device=DEV))
    torch.cuda.synchronize()   # the solver works on a stream of its own
    return state


def run(state):
    case, kind, path = state["case"], state["kind"], state["case"]["path"]
    if path == "batch":
        state["ctx"].solve_batch(kind, state["prepared"])
        return state["times"]
    if path == "serve":
        srv = state["server"]
        tickets = [srv.submit_device(f, w, h, s, t) for f, t, w, h, s in state["calls"]]
        for t in tickets:
            srv.wait(t)
        return state["times"]
    if path == "host":
        return state["ctx"].solve(state["field"], state["seeds"], kind)[0]
    f, t = state["field"].data_ptr(), state["times"].data_ptr()
    if path == "volume":
        state["ctx"].solve3d_device(f, kind, case["w"], case["h"], case["d"], state["seeds"], t)
    else:
        state["ctx"].solve_device(f, kind, case["w"], case["h"], state["seeds"], t)
    return state["times"]


def work(case):
    """Each field element read once, each time written once; one upwind update a cell (about 10
    operations in 2-D, 20 in 3-D)."""
    if case["path"] in ("batch", "serve"):
        cells = sum(w * h for w, h in _shapes(case))
    else:
        cells = case["w"] * case["h"] * case.get("d", 1)
    per = 2 if case["store"] in ("speed_f16", "speed_bf16") else 4
    return {"bytes": cells * (per + 4), "flops": cells * (20 if case["path"] == "volume" else 10)}


# ---- 64-bit solution ------------------------------------------------------------------------

def _fixed_point(cost, seeds):
    """The upwind discrete solution in 64 bits: every cell relaxed from its neighbours until none
    falls any more.  cost: (..., H, W) with 2 axes, or (D, H, W) with 3; seeds index the axes in
    reverse order (x, y[, z])."""
    n = cost.dim()
    c = cost.double()
    box = torch.full([s + 2 for s in c.shape], math.inf, dtype=torch.float64, device=c.device)
    mid = tuple(slice(1, -1) for _ in range(n))
    t = box[mid]
    for s in seeds:
        t[tuple(int(v) for v in reversed(s))] = 0.0

    def side(axis, lo):
        return box[tuple((slice(0, -2) if lo else slice(2, None)) if k == axis else slice(1, -1)
                         for k in range(n))]

    ends = [(side(k, True), side(k, False)) for k in range(n)]
    big = 1e300       # stands for +INF inside an update, so that no difference is a NaN
    for it in range(1, 200000):
        mins = [torch.minimum(a, b).clamp_(max=big) for a, b in ends]
        m1, m2 = torch.minimum(mins[0], mins[1]), torch.maximum(mins[0], mins[1])
        if n == 3:
            m3 = torch.maximum(m2, mins[2])
            m2 = torch.minimum(m2, mins[2])
            m1, m2 = torch.minimum(m1, m2), torch.maximum(m1, m2)
        u = torch.minimum(m2.sub_(m1), c)            # at u = c the two-axis root is m1 + c
        new = (2.0 * c * c - u * u).sqrt_().add_(u).mul_(0.5)
        if n == 3:
            v = torch.minimum(m3.sub_(m1), new)      # at v = new the three-axis root is `new`
            disc = (3.0 * c * c - u * u - v * v - (u - v) ** 2).clamp_(min=0.0)
            new = (u + v + disc.sqrt_()) / 3.0
        new.add_(m1)
        new[new >= big] = math.inf
        if it % 64 == 0:
            before = t.clone()
        torch.minimum(t, new, out=t)
        if it % 64 == 0:
            fell = before - t
            fell = torch.where(torch.isnan(fell), 0.0, fell)
            if float((fell / t.clamp(min=1e-300)).max()) <= 1e-13:
                break
    return t.clone()


def _cost64(field, store):
    return field.double() if store == "cost" else 1.0 / field.double()


def exact(case, seed):
    if case["path"] in ("batch", "serve"):
        if sum(w * h for w, h in _shapes(case)) > 12_000_000:
            return None                              # too long a relaxation, field by field
        out = []
        for f, w, h, s in _many(case, seed):
            t = _fixed_point(_cost64(f, case["store"]), s).reshape(-1)
            out.append(torch.cat([t, t.new_zeros(-len(t) % 64)]))
        return torch.cat(out)
    field, seeds = _one(case, seed)
    t = _fixed_point(_cost64(field, case["store"]), seeds)
    return t.cpu().numpy() if case["path"] == "host" else t
