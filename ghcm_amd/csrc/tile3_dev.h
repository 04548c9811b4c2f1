// tile3_dev.h -- device code shared by the 3-D tile kernels: the three-axis Godunov update and one
// round of an octant sweep over an LDS box.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "tile_dev.h"

namespace ghcm {

// Godunov upwind update in three dimensions for |grad T| = f, h = 1 (the K-axis update of
// src/eikonal.h:73-118 and data/eikonal_common.cl:221-285 at K = 3), on the three axis
// minima a, b, c in any order.  Sorted m1 <= m2 <= m3, the update is the first of
//   m1 + f                                    if it does not exceed m2,
//   the two-axis root                         if it does not exceed m3,
//   m1 + (u + v + sqrt(3 f^2 - u^2 - v^2 - (u - v)^2)) / 3, u = m2 - m1, v = m3 - m1,
// the larger root of (T-m1)^2 + (T-m2)^2 + (T-m3)^2 = f^2 with the common part m1 taken out
// of the discriminant (the reference forms it from the unshifted values).
// Evaluated without a compare or select, by clamping each added axis to where the form
// below it stops being valid (the forms meet there):
//   t2 = the two-axis form at e = min(u, f) (as godunov_raw: exactly m1 + f for u >= f),
//   m3c = min(m3, t2): for m3 >= t2 the three-axis root at v = t2 - m1 is t2 itself,
//   t3 = the three-axis form at (e, m3c - m1),
//   T = med3(t3, m3c, t2), i.e. t3 clamped to [m3c, t2].
// For m3 >= t2 that is t2 exactly; for m3 < t2 it is t3, never below m3 (the largest minimum
// it used) and never above t2.  A float32 emulation over 3 M inputs spread over the three
// branches and their boundaries gives the branch form's result bit for bit except 32
// three-axis cases (1-2 ulp, where t3 had rounded above t2), and the same count of one-ulp
// non-monotone steps.  As in two dimensions, m1 is added by one final rounding.  +INF minima
// fall through to the lower-axis forms (an INF - INF difference makes a NaN that the clamps
// and the final med3, which returns the minimum of its other operands for a NaN operand, drop);
// f = +INF yields +INF.  Every cell update and every face prediction of both 3-D kernels goes
// through this one function.
__device__ __forceinline__ float godunov3(float a, float b, float c, float f) {
    // Sorted by three-operand minimum, median and maximum (v_min3/v_med3/v_max3: the values
    // are non-negative or +INF, never NaN, so the float forms order them exactly).
    const float m1 = fminf(fminf(a, b), c);
    const float m3 = fmaxf(fmaxf(a, b), c);
    const float m2 = __builtin_amdgcn_fmed3f(a, b, c);
    const float u = m2 - m1;
    const float s2 = 1.41421356237309515f * f;
    const float e = __builtin_amdgcn_fmed3f(u, f, 0.0f);
    const float r2 = __builtin_amdgcn_sqrtf((s2 - e) * (s2 + e));
    const float t2 = __builtin_fmaf(e + __builtin_fmaxf(r2, e), 0.5f, m1);
    const float m3c = __builtin_fminf(m3, t2);
    const float v = m3c - m1, w = e - v;
    const float disc = fmaxf(3.0f * f * f - (e * e + v * v + w * w), 0.0f);
    const float t3 = m1 + (e + v + __builtin_amdgcn_sqrtf(disc)) * (1.0f / 3.0f);
    return __builtin_amdgcn_fmed3f(t3, m3c, t2);
}

// ---------------------------------------------------------------------------------------
// Three-dimensional sweep tile solver: eight wave64s per work-group relax one 64 x 8 x 8 tile
// with the eight Gauss-Seidel orders of 3-D fast sweeping (Zhao 2005), one octant per wave,
// concurrently on the same LDS box.  Lane L owns the row (y, z) = (L mod 8, L / 8) and walks
// along x (towards +x or -x with the octant); the octant's rank of the row, r = y' + z' (y'
// and z' counted in the octant's directions, 0..14), skews the walk: at step s the lane is at
// x-position (s - r) mod 64.  The rows upwind in y and z have rank r - 1, so they relaxed the
// same x one step earlier: their results arrive through a DPP row shift (y, the neighbouring
// lane) and ds_bpermute (z, eight lanes away), the upwind x value is the lane's own previous
// result, and each is merged with an LDS read of that cell (improvements of the other seven
// sweeps).  64 + 14 steps give every row one complete ordered walk, so a round of the eight
// sweeps is one full fast-sweeping iteration over the tile in 78 steps; before and after its
// walk a lane relaxes cells of the neighbouring walks instead of idling (every value involved
// is an upper bound).  Rounds repeat until no cell improves by >= eps or the round cap.
// ---------------------------------------------------------------------------------------
constexpr int kS3X = 64, kS3Y = 8, kS3Z = 8;       // tile extents
constexpr int kS3Threads = 512;                    // eight wave64s, one octant each
constexpr int kS3PX = kS3X + 2;                    // box row: x = -1 .. 64
// Box plane stride in words (>= 10 rows of 66).  A step's 64 lanes address the cells
// (z, y, x) = (z, y, c -+ y -+ z); with rows of 66 words and planes of 695 the 64 addresses
// fall in 64 different banks for half of the octants and at most two per bank for the others
// (no stride from 660 to 800 does better for all eight).
constexpr int kS3Plane = 695;
constexpr int kS3Box = (kS3Z + 2) * kS3Plane;      // words of the time box; the cost box follows
constexpr int kS3MaxRank = (kS3Y - 1) + (kS3Z - 1);
constexpr uint32_t kS3HardRounds = 64;
static_assert(kS3Y == 8 && kS3Z == 8, "lane L owns row (L mod 8, L / 8)");

__device__ __forceinline__ int s3_box(int bx, int by, int bz) { return bz * kS3Plane + by * kS3PX + bx; }

// One round of octant (DX, SY, SZ) over the LDS box (time box at shb, cost box kS3Box words
// after it), run by one wave64.
//
// With CHUNK != 0, between() is called by every lane after each CHUNK steps.
template <int DX, int SY, int SZ, int CHUNK = 0, int STEPS = kS3X + kS3MaxRank, class F = NoExchange>
__device__ __forceinline__ void sweep3_round(char* const shb, const int L, F between = F{}) {
    constexpr int PX = kS3PX, PL = kS3Plane;
    // Word offsets from the corner (x-1, y-1, z-1) of the cell's 3 x 3 x 3 neighbourhood: every
    // read and the merge are immediate offsets from one per-step address.
    constexpr int kCell = PL + PX + 1;
    constexpr int kUpX = kCell - DX;
    constexpr int kUpY = kCell - SY * PX;
    constexpr int kUpZ = kCell - SZ * PL;
    constexpr int kCost = kS3Box + kCell;
    // Rows whose upwind z neighbour is in the halo: z = 0 (7) for SZ > 0 (< 0).
    constexpr uint64_t kZHalo = SZ > 0 ? 0x00000000000000FFull : 0xFF00000000000000ull;
    // DPP row shift by one lane towards higher lanes (SY > 0: lane L reads lane L-1) or lower.
    // The rows whose upwind y neighbour is in the halo (y = 0 for SY > 0, 7 for SY < 0) either
    // have no source lane in their row of 16 or take the row y = 7 (0) of the neighbouring z:
    // those rows (kYLast) hand on +INF instead of their result, so every halo row's y value is
    // its LDS read alone.
    constexpr int kDppY = SY > 0 ? 0x111 : 0x101;
    constexpr uint64_t kYLast = SY > 0 ? 0x8080808080808080ull : 0x0101010101010101ull;
    const int y = L & 7, z = L >> 3;
    const int rank = (SY > 0 ? y : kS3Y - 1 - y) + (SZ > 0 ? z : kS3Z - 1 - z);
    const int zsrc = 4 * ((L - 8 * SZ) & 63);           // ds_bpermute byte address of the z-upwind lane
    const int x0 = DX > 0 ? 0 : kS3X - 1;
    const int rs = 4 * (z * PL + y * PX + x0);           // the walk's first cell (corner-relative)
    // The first load steps to x-position (0 - rank) mod 64, or to rs where that is 0.
    int bb = rs + 4 * DX * (kS3X - 1 - rank);
    // 78 steps complete every walk; the loop runs 80 (four per iteration, never unrolled further).
    constexpr int SE = (STEPS + 3) & ~3;
    struct Nb {
        float ux, uy, uz, cc;
        int b;
        bool first;
    };
    // Single-word loads at immediate offsets from the step's address (relaxed atomic loads are
    // not paired into ds_read2, which would need a second address register per step).
    auto at = [&](int b, int word) -> float {
        return __uint_as_float(__hip_atomic_load(reinterpret_cast<const uint32_t*>(shb + b + 4 * word),
                                                 __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
    };
    // Step s: lanes with rank == s mod 64 are at x-position 0 (their walk restarts at rs).  The
    // test for the next step is made one load ahead, so the select does not wait on the
    // compare's lane mask.
    bool first_next = rank == 0;
    auto load = [&](Nb& o, int st) {
        o.first = first_next;
        bb = o.first ? rs : bb + 4 * DX;
        o.b = bb;
        o.ux = at(bb, kUpX);
        o.uy = at(bb, kUpY);
        o.uz = at(bb, kUpZ);
        o.cc = at(bb, kCost);
        first_next = rank == ((st + 1) & 63);
    };
    auto umin = [](float u, float v) {
        return __uint_as_float(min(__float_as_uint(u), __float_as_uint(v)));
    };
    const float inf = __builtin_inff();
    // The previous step's result of this lane (upwind x), of the y-upwind lane (a DPP row shift
    // folded into the minimum: its `old` is the minimum's identity and its bound control is
    // off, so a lane without a source lane keeps its LDS read) and of the z-upwind lane
    // (ds_bpermute, issued as soon as the result exists, ahead of the next step's LDS reads).
    float prev = inf, ysend = inf, zv = inf;
    auto step = [&](const Nb& n) {
        const float ax = umin(n.ux, n.first ? inf : prev);
        const float ay = __uint_as_float(
            min(__float_as_uint(n.uy),
                (uint32_t)__builtin_amdgcn_update_dpp(-1, __float_as_int(ysend), kDppY, 0xF, 0xF, false)));
        const float az = umin(n.uz, __builtin_amdgcn_inverse_ballot_w64(kZHalo) ? inf : zv);
        const float t = godunov3(ax, ay, az, n.cc);
        __hip_atomic_fetch_min(reinterpret_cast<uint32_t*>(shb + n.b + 4 * kCell), __float_as_uint(t),
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        prev = t;
        zv = __int_as_float(__builtin_amdgcn_ds_bpermute(zsrc, __float_as_int(t)));
        ysend = __builtin_amdgcn_inverse_ballot_w64(kYLast) ? inf : t;
    };
    // Loads of step s+1 are issued before step s is computed: their cells are upper bounds
    // whatever the interleaving, and the values step s produces reach step s+1 through registers.
    // Four register sets in rotation, so that the loads do not wait for those step s-1 still uses
    // (two -> four: 256^3 by waves 3,920 -> 3,830 us, 70 x 200 x 60 resident 500 -> 492).
    Nb X[4];
    load(X[0], 0);
    auto four = [&](int st) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            load(X[(i + 1) & 3], st + i + 1);
            __builtin_amdgcn_sched_barrier(0);
            step(X[i]);
        }
    };
    if constexpr (CHUNK == 0) {
#pragma clang loop unroll(disable)
        for (int st = 0; st < SE; st += 4) four(st);
    } else {
        static_assert(CHUNK % 4 == 0 && SE % CHUNK == 0, "whole chunks");
        for (int s0 = 0; s0 < SE; s0 += CHUNK) {
            for (int st = s0; st < s0 + CHUNK; st += 4) four(st);
            between();
        }
    }
}

}  // namespace ghcm
