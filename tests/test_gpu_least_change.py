"""A resident solve with a large least change leaves no border behind -- needs an MI355X.

The field makes one tile's border fall many times by less than the least change.  K corridors, each
longer and a little cheaper than the one before, end in one collector, whose time therefore falls
K times by 1.2 eps, one corridor after the other.  It meets a time that stays (r) in the cell q,
which as long as both count falls by less than eps each time, 14 eps in all.  q's right neighbour
lies in the next tile (A), and above it, in a third (B), the only cell that A's border feeds.

Tolerance: a settled cell does not improve by eps from its neighbours: gap <= 2 eps and 4 ulp, as
in the parity tests.
"""
import numpy as np
import pytest

import ghcm_amd as g
from conftest import fixed_point_gap, ulp32

pytestmark = pytest.mark.gpu
EPS, K = 0.125, 24


def staircase(tw, th):
    spacing = max(40, 3 * th)
    cols = -(-(2 * K + 2) // tw) * tw              # of the corridors
    w, h = cols + 3 * tw, th + spacing * (K + 1)
    cost = np.full((h, w), np.inf, np.float32)
    y = th                                         # the collector's row: the first of its tiles
    xq = cols + tw - 1                             # q: the last column of its tile
    cost[y, 0:xq] = 1e-4
    seeds = []
    r, c = 500.0, 18 * EPS
    for i in range(K):
        n = spacing * (i + 1)
        cost[y + 1:y + n, 2 * i] = (r + c - 1.2 * EPS * i) / (n - 1)
        cost[y + n, 2 * i] = 1.0
        seeds.append((2 * i, y + n))
    cost[y, xq] = c
    cost[y + 1, xq] = r                            # time r, from the source below it
    cost[y + 2, xq] = 1.0
    seeds.append((xq, y + 2))
    cost[y, xq + 1] = cost[y - 1, xq + 1] = 1.0    # A and, above it, B
    return cost, seeds, (xq + 1, y - 1)


TILES = [(g.KERNEL_SYSTOLIC, (8, 8)), (g.KERNEL_FIM, (16, 16)), (g.KERNEL_SYSTOLIC, (32, 8)),
         (g.KERNEL_FIM, (32, 32)), (g.KERNEL_SWEEP, (64, 64))]


@pytest.mark.parametrize("kernel,tile", TILES)
def test_small_drops_of_a_border_add_up(kernel, tile):
    cost, seeds, (bx, by) = staircase(*tile)
    print(f"case staircase kernel={kernel} tile={tile} {cost.shape}", flush=True)
    with g.Context(0, tile_w=tile[0], tile_h=tile[1], kernel=kernel, min_change=EPS, n_active=512) as ctx:
        t, st = ctx.solve(cost, seeds)
    assert st["converged"] == 1
    gap = fixed_point_gap(t, cost, seeds)
    print(f"  T[B]={t[by, bx]} T[A]={t[by + 1, bx]} gap {gap.max()}", flush=True)
    assert np.all(gap <= 4 * ulp32(t) + 2 * EPS), f"gap {gap.max()} at {np.unravel_index(gap.argmax(), gap.shape)}"
