"""Requests admitted to a server together: one launch initialises all of them.  Needs an MI355X."""
import numpy as np
import pytest

import ghcm_amd as g
import oracle
from test_gpu_parity import check

pytestmark = pytest.mark.gpu

CONFIGS = {"sweep": dict(tile_w=64, tile_h=64, kernel=g.KERNEL_SWEEP, n_active=512, inner_iter_cap=1),
           "systolic": dict(tile_w=16, tile_h=16, kernel=g.KERNEL_SYSTOLIC, n_active=2048)}


# one request, a few, and more than the slots (so that slots are used again); one-cell, one-row and
# ragged fields beside one of 1100 x 70
@pytest.mark.parametrize("n", [1, 5, 90])
@pytest.mark.parametrize("cfg", list(CONFIGS))
def test_burst_of_requests(rng, cfg, n):
    shapes = [(70, 1100), (1, 1), (1, 200), (65, 64), (63, 129)]
    shapes += [(int(rng.integers(1, 150)), int(rng.integers(1, 150))) for _ in range(n)]
    reqs = []
    for i, (h, w) in enumerate(shapes[:n]):
        cost = rng.uniform(0.1, 10.0, (h, w)).astype(np.float32)
        reqs.append((cost, [(int(rng.integers(0, w)), int(rng.integers(0, h))) for _ in range(1 + i % 3)]))
    print(f"case burst of {n} requests, {cfg}", flush=True)
    with g.Server(0, max_slots=64, **CONFIGS[cfg]) as srv:
        for _ in range(2):
            tickets = [srv.submit(cost, seeds) for cost, seeds in reqs]
            for (cost, seeds), ticket in zip(reqs, tickets):
                t, r = srv.wait(ticket, 60.0)
                assert r["status"] == g.OK
                check(t, oracle.fmm_f32(cost, seeds), seeds, cost, label=f"{cfg} {cost.shape}")
