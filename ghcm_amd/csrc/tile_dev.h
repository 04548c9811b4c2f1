// tile_dev.h -- device code shared by the tile kernels: field loads, the Godunov update, wave
// reductions and one round of a fast-sweeping order over an LDS tile.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "ghcm_dev.h"
#include "tile_geom.h"

namespace ghcm {

// Pointers read out of device memory (the instance records) are generic to the compiler,
// which then emits flat accesses (64-bit lane addresses, both wait counters).  They always
// address global memory; the cast lets it emit global loads and stores with a scalar base.
template <typename T>
__device__ __forceinline__ __attribute__((address_space(1))) T* gmem(T* p) {
    return (__attribute__((address_space(1))) T*)p;
}

// Bytes per field element of a field kind (FP32 cost or speed, FP16 or BF16 speed).
template <int KIND>
constexpr uint32_t field_bytes() { return KIND <= 1 ? 4u : 2u; }

// Cost of the field element at byte address p.
template <int KIND>
__device__ __forceinline__ float load_cost_at(const char* p) {
    if constexpr (KIND == 0) {
        return *gmem(reinterpret_cast<const float*>(p));
    } else if constexpr (KIND == 1) {
        return 1.0f / *gmem(reinterpret_cast<const float*>(p));
    } else if constexpr (KIND == 2) {
        return 1.0f / static_cast<float>(*gmem(reinterpret_cast<const _Float16*>(p)));
    } else {
        uint32_t b = static_cast<uint32_t>(*gmem(reinterpret_cast<const uint16_t*>(p))) << 16;
        return 1.0f / __uint_as_float(b);
    }
}

// Godunov upwind update for |grad T| = c with h = 1, cancellation-safe form, without the
// final min against the old time.  m = min(a,b) is passed in and d = |a-b|; if c < d the 1-D
// update m + c applies (data/eikonal_common.cl:296-297); otherwise T = m + d/2 +
// sqrt((sqrt2 c - d)(sqrt2 c + d))/2, the root of (T-a)^2 + (T-b)^2 = c^2 (:299-300) with
// the discriminant factored and the large common part m added outside the root.
// Branch-free, without a select: the two-axis form is evaluated at e = min(d, c), as
// m + (e + max(root, e))/2.  For d <= c that is the form itself (root >= d there, exactly;
// the max matters only within an ulp of d = c, where it gives m + d = max(a,b), the exact
// value).  For d > c, e = c and the rounded root never exceeds c (sqrt2 rounds down to the
// float constant), so the max yields c and the result is m + c rounded once: the 1-D update,
// bit for bit.  The result therefore never falls as d crosses c (the 1-D value is not below
// the two-axis values next to it), which the border checks rely on: they predict a
// neighbour's update from a subset of the inputs its own solve sees, and a prediction an ulp
// below what the solve then computes would re-activate the pair without end at eps = 0.
// The discriminant lies in [c^2, 2c^2] on every lane, so the square root (the hardware
// v_sqrt_f32, 1 ulp) never sees a negative argument.  e is a v_med3 against 0 (d and c are
// non-negative); when d is NaN (a = b = +INF) the med3 yields the minimum of the other two
// operands, 0, and the result is m + (a finite value) = +INF.
// The large common part m is added by one final rounding of m + (e + root)/2, the
// parenthesis formed at the scale of c: the result then never rounds below max(a,b) where
// the exact root equals it (c = d), so a cell never drops below a neighbour it was computed
// from.  (Rounding m + e/2 first and adding root/2 after breaks that: two cells can then
// lower each other by an ulp at a time without end.)  The final step is
// fma(e + max(root, e), 1/2, m): halving is exact for normal numbers, so it equals m + (the
// rounded half-sum) with one rounding.
// Every update of a cell and every border prediction of a neighbour's update goes through
// this one function.
__device__ __forceinline__ float godunov_raw(float ax, float ay, float m, float c) {
    const float d = fabsf(ax - ay);                // NaN when both are +INF
    const float e = __builtin_amdgcn_fmed3f(d, c, 0.0f);
    const float s = 1.41421356237309515f * c;
    const float root = __builtin_amdgcn_sqrtf((s - e) * (s + e));
    return __builtin_fmaf(e + __builtin_fmaxf(root, e), 0.5f, m);
}

// The update min'ed with the old time t (:305-308).
__device__ __forceinline__ float godunov(float ax, float ay, float c, float t) {
    return fminf(t, godunov_raw(ax, ay, fminf(ax, ay), c));
}

// Wave reductions: a DPP butterfly inside each row of 16 lanes (quad_perm [1,0,3,2] and
// [2,3,0,1], then row_half_mirror and row_mirror, after which every lane of a row holds its
// row's result), then the four rows' results read into scalar registers and combined there.
// No LDS round trip (a __shfl_xor butterfly is six dependent ds_bpermute).  Every lane must be
// active, as at every call site; the result is wave-uniform.
template <int CTRL>
__device__ __forceinline__ uint32_t dpp_u32(uint32_t x) {
    return (uint32_t)__builtin_amdgcn_update_dpp((int)x, (int)x, CTRL, 0xF, 0xF, false);
}

template <typename Op>
__device__ __forceinline__ uint32_t wave_reduce_u32(uint32_t v, Op op) {
    v = op(v, dpp_u32<0xB1>(v));
    v = op(v, dpp_u32<0x4E>(v));
    v = op(v, dpp_u32<0x141>(v));
    v = op(v, dpp_u32<0x140>(v));
    const uint32_t r0 = (uint32_t)__builtin_amdgcn_readlane((int)v, 0);
    const uint32_t r1 = (uint32_t)__builtin_amdgcn_readlane((int)v, 16);
    const uint32_t r2 = (uint32_t)__builtin_amdgcn_readlane((int)v, 32);
    const uint32_t r3 = (uint32_t)__builtin_amdgcn_readlane((int)v, 48);
    return op(op(r0, r1), op(r2, r3));
}

// Minimum of times or keys: non-negative or +INF, so their bit patterns order like the values.
__device__ __forceinline__ float wave_min(float v) {
    return __uint_as_float(wave_reduce_u32(__float_as_uint(v), [](uint32_t x, uint32_t y) { return min(x, y); }));
}

__device__ __forceinline__ uint32_t wave_sum(uint32_t v) {
    return wave_reduce_u32(v, [](uint32_t x, uint32_t y) { return x + y; });
}

// Stores to mapped host memory: system scope, relaxed (each word is read on its own).
__device__ __forceinline__ void sys_store(uint32_t* p, uint32_t v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
__device__ __forceinline__ void sys_store64(unsigned long long* p, unsigned long long v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// An instance record as wave-uniform register values.  The record is the same for every
// lane of a work-group; passing each word through readfirstlane puts it in scalar registers,
// so the tile's loads take a scalar base and carry no dependency on the vector load that
// fetched the record (which would otherwise make every conditional staging load wait for
// all loads before it).
__device__ __forceinline__ GhcmInst uniform_inst(const GhcmInst& m) {
    auto u64 = [](const void* p) {
        const uint64_t v = reinterpret_cast<uint64_t>(p);
        const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
        const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
        return ((uint64_t)hi << 32) | lo;
    };
    GhcmInst r;
    r.field = reinterpret_cast<const void*>(u64(m.field));
    r.time = reinterpret_cast<float*>(u64(m.time));
    r.w = __builtin_amdgcn_readfirstlane(m.w);
    r.h = __builtin_amdgcn_readfirstlane(m.h);
    r.tiles_x = __builtin_amdgcn_readfirstlane(m.tiles_x);
    r.tiles_y = __builtin_amdgcn_readfirstlane(m.tiles_y);
    r.tile_base = __builtin_amdgcn_readfirstlane(m.tile_base);
    r.d = __builtin_amdgcn_readfirstlane(m.d);
    r.tiles_z = __builtin_amdgcn_readfirstlane(m.tiles_z);
    r.pad = 0u;
    return r;
}

// Threads of a sweep work-group: four wave64s, one per sweep order.
constexpr int kSweepThreads = 256;

// min(u, lane L-1's v) on time bits, with lane 0 (no source lane) taking u.  The DPP move's
// `old` is the minimum's identity (all ones) and its bound control is off, so the compiler
// folds the move into the minimum as one v_min_u32 with a wave_shr:1 DPP operand, whose
// lane 0 keeps u.
__device__ __forceinline__ float umin_from_lower_lane(float u, float v) {
    const uint32_t w = (uint32_t)__builtin_amdgcn_update_dpp(-1, __float_as_int(v), 0x138, 0xF, 0xF, false);
    return __uint_as_float(min(__float_as_uint(u), w));
}

// LDS words of a sweep tile: time box, a sink word, cost box.
template <int TW, int TH>
constexpr int sweep_lds_words() { return 2 * (TW + 2) * (TH + 2) + 1; }

// One round of one sweep order over the LDS tile (time box at shb, cost box CB words after it),
// run by one wave64.  DX > 0: lane L owns column x = L, sweeping towards +x; DX < 0: column
// TW-1-L, towards -x.  DOWN: rows ascending.  Wrapped skew: at step s lane L relaxes pass
// position (s - L) mod TH of its column (row p of a downward pass, TH-1-p of an upward one),
// so lane L reaches the first row of its ordered pass at step L, one step after lane L-1, and
// the lanes' ordered passes form one anti-diagonal front; TW + TH - 1 steps give every column
// one complete ordered pass, and before and after it a lane relaxes cells of the neighbouring
// passes instead of idling (every value involved is an upper bound).
//
// A step reads only the cell's two upwind neighbours and its cost: the sweep towards +x and +y
// updates a cell from its -x and -y neighbours.  The other two sweeps' updates cover the +x and
// +y neighbours, and the minimum of the four one-sided updates is the two-sided Godunov update
// (it is monotone in both axis values), so the four sweeps together have the same fixed point
// as sweeps that read all four neighbours.  The upwind values just computed arrive through
// `prev` (this lane's previous cell, the upwind row) and a wave_shr:1 DPP move of lane L-1's
// `prev` (the upwind column); each is merged with this lane's own LDS read of that cell, so
// improvements made by the other three sweeps are used as soon as they land.  Lane 0 has no
// source lane: its upwind column is the halo read from LDS alone.
// Results are merged into the tile with an LDS atomic minimum (no return value waited for).
//
// With CHUNK != 0, between() is called by every lane after each CHUNK steps.
struct NoExchange {
    __device__ void operator()() const {}
};
template <int TW, int TH, int DX, bool DOWN, int CHUNK = 0, int STEPS = TW + TH - 1, class F = NoExchange>
__device__ __forceinline__ void sweep_round(char* const shb, const int L, F between = F{}) {
    constexpr int PW = TW + 2;
    constexpr int PH = TH + 2;
    constexpr int CB = PW * PH + 1;
    static_assert((TH & (TH - 1)) == 0, "TH must be a power of two");
    const bool lane_on = L < TW;
    // Lanes past the tile width (TW < 64) shadow the last column and never store.
    const int xc = lane_on ? (DX > 0 ? L : TW - 1 - L) : (DX > 0 ? TW - 1 : 0);
    // Word offsets from the corner (r, xc) of the 3 x 3 box around the cell, which sits at
    // padded position (r + 1, xc + 1): every read and the store are immediate offsets from one
    // per-step address.
    constexpr int kUpRow = DOWN ? 1 : 2 * PW + 1;
    constexpr int kUpCol = DX > 0 ? PW : PW + 2;
    constexpr int kCell = PW + 1;
    constexpr int kCost = CB + PW + 1;
    constexpr int b_step = DOWN ? 4 * PW : -4 * PW;
    constexpr int r_first = DOWN ? 0 : TH - 1;
    const int p0 = (-L) & (TH - 1);
    const int r_start = DOWN ? p0 : TH - 1 - p0;
    const int b_first = r_first * (4 * PW) + 4 * xc;
    const int b_start = r_start * (4 * PW) + 4 * xc;
    // Lane L is at the first row of its pass at the steps s with s = L (mod TH): a scalar
    // one-hot pattern shifted by s & (TH-1) marks those lanes, and the row's byte offset
    // advances by one row per step, back to the first row exactly there (the wrap of the row
    // index coincides with the pass start).
    constexpr uint64_t kFirstPat = TH >= 64 ? 1ull : ~0ull / ((1ull << (TH & 63)) - 1ull);
    constexpr int SE = (STEPS + 3) & ~3;
    int bb = b_start - b_step;
    uint32_t jl = 0;
    struct Nb {
        float ur, uc, cc;
        int b;
        bool first;
    };
    auto at = [&](int b, int word) -> float { return *reinterpret_cast<const float*>(shb + b + 4 * word); };
    // LDS reads of step s+1 are issued before step s is computed: their cells are upper bounds
    // whatever the interleaving, and the fresh upwind values arrive through DPP and `prev`, so the
    // dependent chain per step is DPP + update.  Four register sets in rotation: with two, the reads
    // of step s+1 wait for the registers that step s-1 still uses (whole resident solves with two ->
    // four: 256^2 rings 232 -> 219 us, 1531 x 977 smooth 337 -> 315, 2048^2 contrast 1,750 -> 1,600;
    // reads two or three steps ahead are no faster, 320 and 1,660 us, and slower where the CU is full).
    auto load = [&](Nb& o) {
        o.first = __builtin_amdgcn_inverse_ballot_w64(kFirstPat << (jl & (TH - 1)));
        ++jl;
        bb = o.first ? b_first : bb + b_step;
        o.b = bb;
        o.ur = at(o.b, kUpRow);
        o.uc = at(o.b, kUpCol);
        o.cc = at(o.b, kCost);
    };
    // Times are non-negative or +INF, so their bit patterns order like the values: the axis
    // minima and the merge use integer minimum (no NaN canonicalisation needed).
    auto umin = [](float u, float v) {
        return __uint_as_float(min(__float_as_uint(u), __float_as_uint(v)));
    };
    float prev = __builtin_inff();
    auto step = [&](const Nb& n) {
        // Lane L-1's fresh value of the upwind column cell.
        const float ax = umin_from_lower_lane(n.uc, prev);
        const float ay = umin(n.ur, n.first ? __builtin_inff() : prev);
        const float t = godunov_raw(ax, ay, umin(ax, ay), n.cc);
        if (TW == 64 || lane_on)
            __hip_atomic_fetch_min(reinterpret_cast<uint32_t*>(shb + n.b + 4 * kCell),
                                   __float_as_uint(t), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        // The raw result is handed on, not min(t, old): both consumers take the minimum with
        // their own LDS read of the cell.
        prev = t;
    };
    Nb X[4];
    load(X[0]);
    auto four = [&]() {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            load(X[(i + 1) & 3]);
            __builtin_amdgcn_sched_barrier(0);
            step(X[i]);
        }
    };
    if constexpr (CHUNK == 0) {
        for (int st = 0; st < SE; st += 4) four();
    } else {
        static_assert(SE % CHUNK == 0 && CHUNK % 4 == 0, "whole chunks");
        for (int ch = 0; ch < SE / CHUNK; ++ch) {
            for (int st = 0; st < CHUNK; st += 4) four();
            between();
        }
    }
}

// t improves on t0 by at least eps (strictly): times are compared as bits, so a NaN or a
// negative value never counts.
__device__ __forceinline__ bool improves(float t, float t0, float eps) {
    return __float_as_uint(t) < __float_as_uint(t0) && t0 - t >= eps;
}

__device__ __forceinline__ float umin_bits(float u, float v) {
    return __uint_as_float(min(__float_as_uint(u), __float_as_uint(v)));
}

// Whether a cell of this lane's part of the LDS tile would improve from its four neighbours by at
// least eps; on no lane of the four waves: the tile is settled with respect to its halo.  Wave w
// checks a quarter of the rows, lane L column L; the rows roll through registers and the left and
// right neighbours come by DPP, so a cell costs three LDS reads (its lower neighbour, its cost and
// the halo cell for the outer lanes).
template <int TW, int TH>
__device__ __forceinline__ bool tile_unsettled(const float* t_s, const float* c_s, int w, int L, float eps) {
    constexpr int PW = TW + 2, RW = TH / 4;
    static_assert(TW == 64, "one lane per column");
    const int r0 = w * RW;
    const float* const col = t_s + (r0 + 1) * PW + L + 1;
    const float* const cst = c_s + (r0 + 1) * PW + L + 1;
    const float* const hal = t_s + (r0 + 1) * PW + (L < 32 ? 0 : PW - 1);
    float up = col[-PW], mid = col[0];
    bool res = false;
#pragma unroll
    for (int k = 0; k < RW; ++k) {
        const float down = col[(k + 1) * PW], h = hal[k * PW], c = cst[k * PW];
        // lanes 0 and 63 have no source lane and keep their halo cell
        const float l = __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(h), __float_as_int(mid), 0x138, 0xF, 0xF, false));
        const float r = __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(h), __float_as_int(mid), 0x130, 0xF, 0xF, false));
        const float ax = umin_bits(l, r), ay = umin_bits(up, down);
        res |= improves(godunov_raw(ax, ay, umin_bits(ax, ay), c), mid, eps);
        up = mid;
        mid = down;
    }
    return res;
}

}  // namespace ghcm
