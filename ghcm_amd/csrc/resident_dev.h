// resident_dev.h -- device code shared by the resident solves: agent-scope access, joining and
// leaving, tile records and the launch that prepares a solve.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "ghcm_dev.h"
#include "resident.h"
#include "tile_dev.h"
#include "tile_geom.h"

namespace ghcm {

constexpr uint32_t kCmdDone = 0xFFFFFFFFu;
constexpr uint32_t kCmdAbort = 0xFFFFFFFEu;
constexpr uint64_t kJoinTicks = 20000;               // 200 us of the 100 MHz counter
constexpr uint64_t kLimitTicks = 2000000000ull;      // 20 s
// Issue priority of a wave that sweeps or relaxes a tile, over the 0 of those that look, wait, open
// or write back: a step's chain of dependent instructions then never stands behind the polling of
// the idle tiles on its SIMD.  All waves at 0 against this: 4096^2 1,080 -> 993 us, 2048^2 contrast
// 1,541 -> 1,474, batch of 512 11.7 -> 10.6 ms, 512^2 in 8x8 systolic tiles 1,433 -> 1,391; one tile
// or less to a SIMD (256^2, 1531 x 977, small volumes) equal.
constexpr int kWorkPriority = 2;

__device__ __forceinline__ uint32_t ld_agent(const uint32_t* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_agent(uint32_t* p, uint32_t v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned long long ld_agent64(const unsigned long long* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_agent64(unsigned long long* p, unsigned long long v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Every vector memory operation of this wave so far is complete (stores: visible at the scope
// they were made).
__device__ __forceinline__ void wait_stores() { __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

__device__ __forceinline__ uint64_t now_ticks() { return __builtin_amdgcn_s_memrealtime(); }

// The tiles' order: row by row, row ty rotated by ty times shear tiles, so that a front along a
// column of tiles meets as many different work-groups (and XCDs) as one along a row.
__device__ __forceinline__ uint32_t shear(uint32_t tiles_x) { return (tiles_x * 3u / 8u) | 1u; }
__device__ __forceinline__ uint32_t resident_rank(const GhcmInst& in, uint32_t tx, uint32_t ty) {
    const uint32_t rot = (uint32_t)(((uint64_t)ty * shear(in.tiles_x)) % in.tiles_x);
    const uint32_t x = tx + rot;
    return in.tile_base + ty * in.tiles_x + (x >= in.tiles_x ? x - in.tiles_x : x);
}
__device__ __forceinline__ void resident_tile(const GhcmInst& in, uint32_t rank, int& tx, int& ty) {
    const uint32_t lr = rank - in.tile_base, y = lr / in.tiles_x, x = lr - y * in.tiles_x;
    const uint32_t rot = (uint32_t)(((uint64_t)y * shear(in.tiles_x)) % in.tiles_x);
    tx = (int)(x >= rot ? x - rot : x + in.tiles_x - rot);
    ty = (int)y;
}

// A tile's record as wave-uniform values.
template <typename Tile>
__device__ __forceinline__ Tile uniform_tile(const Tile* p) {
    static_assert(sizeof(Tile) % 16 == 0, "whole vectors");
    Tile d;
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    u32x4 v[sizeof(Tile) / 16];
    uint32_t* const o = reinterpret_cast<uint32_t*>(&d);
#pragma unroll
    for (size_t i = 0; i < sizeof(Tile) / 16; ++i) v[i] = gmem(reinterpret_cast<const u32x4*>(p))[i];
#pragma unroll
    for (size_t i = 0; i < sizeof(Tile) / 16; ++i) {
        o[4 * i] = __builtin_amdgcn_readfirstlane(v[i].x);
        o[4 * i + 1] = __builtin_amdgcn_readfirstlane(v[i].y);
        o[4 * i + 2] = __builtin_amdgcn_readfirstlane(v[i].z);
        o[4 * i + 3] = __builtin_amdgcn_readfirstlane(v[i].w);
    }
    return d;
}

// Whether the caller is the last of N to come to the counter at ctl[which]: one counter for the
// work-groups b with equal b % kResSpread, and one for the last of each, each on its own line.
__device__ __forceinline__ bool last_in(uint32_t* ctl, uint32_t which, uint32_t b, uint32_t N) {
    const uint32_t j = b % kResSpread, members = (N - j + kResSpread - 1u) / kResSpread;
    uint32_t* const c = ctl + which;
    if (__hip_atomic_fetch_add(c + (1u + j) * kCounterStride, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1u != members)
        return false;
    return __hip_atomic_fetch_add(c, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1u == min(N, kResSpread);
}

__device__ __forceinline__ bool decide(uint32_t* ctl, uint32_t what) {
    uint32_t expect = 0u;
    return __hip_atomic_compare_exchange_strong(&ctl[kResDecision], &expect, what, __ATOMIC_RELAXED,
                                                __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// 1 once every work-group is running; 2, the solve given up, if that takes kJoinTicks.
__device__ __forceinline__ uint32_t await_decision(uint32_t* ctl, uint64_t t_start) {
    uint32_t d;
    while ((d = ld_agent(&ctl[kResDecision])) == 0u) {
        if (now_ticks() - t_start > kJoinTicks) (void)decide(ctl, 2u);
        __builtin_amdgcn_s_sleep(4);
    }
    return d;
}

// Every 1,024 rounds a busy work-group asks whether to stop: told so, or out of time, in which case
// it tells the others (N command words) and fails the solve.  Sweeps end by themselves (every round
// but the last lowers a cell); this bounds them whatever the field holds.
__device__ __forceinline__ bool must_stop(uint32_t* ctl, uint32_t* cmd, uint32_t own, uint32_t N, uint64_t t_start) {
    if (ld_agent(&cmd[own]) == kCmdAbort) return true;
    if (now_ticks() - t_start <= kLimitTicks) return false;
    st_agent(&ctl[kResFailed], 1u);
    for (uint32_t i = 0; i < N; ++i) st_agent(&cmd[i], kCmdAbort);
    return true;
}

// The totals for the host, by one thread; the tag last.  failed: the solve was given up.
template <typename Args>
__device__ __forceinline__ void report_totals(const Args& a, unsigned long long visits,
                                              unsigned long long passes, unsigned long long cells, uint32_t most,
                                              bool failed) {
    sys_store64(&a.rec->totals[0], visits);
    sys_store64(&a.rec->totals[1], passes);
    sys_store64(&a.rec->totals[2], cells);
    sys_store(&a.rec->wave, failed ? 1u : 0u);
    sys_store(&a.rec->busy_waves, most);
    wait_stores();
    sys_store(&a.rec->totals_tag, a.tag);
}

// With many sources, a.seeds: whether cell `i` of the tile of this rank is one (row by row, of CELLS),
// whether the tile holds one, and the marks made and cleared (by all threads of a grid).
template <uint32_t CELLS, typename Args>
__device__ __forceinline__ bool is_source(const Args& a, uint32_t rank, uint32_t i) {
    return ((a.seeds[(size_t)rank * (CELLS / 32u) + (i >> 5)] >> (i & 31u)) & 1u) != 0u;
}
template <uint32_t CELLS, typename Args>
__device__ __forceinline__ uint32_t& holds_source(const Args& a, uint32_t rank) {
    return a.seeds[(size_t)a.tiles * (CELLS / 32u) + rank];
}
template <uint32_t CELLS, typename Args>
__device__ __forceinline__ void mark_source(const Args& a, uint32_t rank, uint32_t i) {
    atomicOr(&a.seeds[(size_t)rank * (CELLS / 32u) + (i >> 5)], 1u << (i & 31u));
    holds_source<CELLS>(a, rank) = 1u;
}
template <uint32_t CELLS, typename Args>
__device__ __forceinline__ void clear_sources(const Args& a, size_t i0, size_t stride) {
    for (size_t i = i0; i < (size_t)a.tiles * (CELLS / 32u + 1u); i += stride) a.seeds[i] = 0u;
}

// The state of a resident solve, in one launch: the tiles' records and the sources (few: with the
// rank of their tile; many: k_resident_sources follows) from the mapped host tables, borders at
// +INF, every work-group busy.
// N: work-groups the tiles are dealt out to; words: of a tile's borders; states: counters; d_inst:
// with many sources, the instances for k_resident_sources.
template <int TW, int TH, int FB>
__global__ void k_resident_init(ResidentArgs a, const GhcmInst* h_inst, GhcmInst* d_inst, const uint32_t* h_seeds,
                                uint32_t N, uint32_t words, uint32_t states) {
    const size_t i0 = (size_t)blockIdx.x * blockDim.x + threadIdx.x, stride = (size_t)gridDim.x * blockDim.x;
    const uint4 inf4 = make_uint4(kInfBits, kInfBits, kInfBits, kInfBits);
    uint4* const e4 = reinterpret_cast<uint4*>(a.edges);
    uint4* const s4 = reinterpret_cast<uint4*>(a.seen);
    for (size_t i = i0; i < (size_t)a.tiles * words / 4; i += stride) {
        e4[i] = inf4;
        if (a.seen) s4[i] = inf4;
    }
    if (a.want)
        for (size_t i = i0; i < (size_t)kResMaxGroups * a.want_stride; i += stride) a.want[i] = kInfBits;
    for (size_t i = i0; i < states; i += stride) {
        a.state[i] = 1ull;
        a.cmd[i] = 0u;
    }
    for (size_t i = i0; i < kResCtlWords; i += stride) a.ctl[i] = 0u;
    if (many_sources(a.n_seeds)) {
        clear_sources<TW * TH>(a, i0, stride);
        for (size_t j = i0; j < a.n_inst; j += stride) d_inst[j] = h_inst[j];
    }
    for (size_t i = i0; i < (many_sources(a.n_seeds) ? 0u : a.n_seeds); i += stride) {
        const uint32_t x = h_seeds[3 * i], y = h_seeds[3 * i + 1], j = h_seeds[3 * i + 2];
        const GhcmInst in = h_inst[j];
        a.seeds[4 * i] = x;
        a.seeds[4 * i + 1] = y;
        a.seeds[4 * i + 2] = j;
        a.seeds[4 * i + 3] = resident_rank(in, x / TW, y / TH);
    }
    // Tile records: with few instances several blocks share one.
    const uint32_t share = gridDim.x > a.n_inst ? gridDim.x / a.n_inst : 1u;
    for (uint32_t j = blockIdx.x / share; j < a.n_inst; j += gridDim.x / share) {
        if (blockIdx.x / share >= gridDim.x / share) break;
        const GhcmInst in = h_inst[j];
        const uint32_t nt = in.tiles_x * in.tiles_y;
        for (uint32_t t = (blockIdx.x % share) * blockDim.x + threadIdx.x; t < nt; t += share * blockDim.x) {
            int tx, ty;
            resident_tile(in, in.tile_base + t, tx, ty);
            ResTile d;
            d.g = in.tile_base + (uint32_t)ty * in.tiles_x + (uint32_t)tx;
            d.inst = j;
            d.w = in.w;
            d.x0 = (uint32_t)tx * TW;
            d.y0 = (uint32_t)ty * TH;
            const size_t org = (size_t)d.y0 * in.w + d.x0;
            d.field = static_cast<const char*>(in.field) + org * FB;
            d.time = in.time + org;
            d.ext = (uint32_t)tile_extent((int)in.w, (int)d.x0, TW) | (uint32_t)tile_extent((int)in.h, (int)d.y0, TH) << 8;
            for (int s = 0; s < 4; ++s) {
                const uint32_t nb = tile_neighbour(in.tile_base, in.tiles_x, in.tiles_y, tx, ty, s);
                d.face[s] = nb == kNoTile ? kNoTile : nb * 4u + (uint32_t)(s ^ 2);
                const uint32_t r = nb == kNoTile ? 0u : resident_rank(in, (uint32_t)(tx + side_dx(s)), (uint32_t)(ty + side_dy(s)));
                d.call[s] = (r % N) * a.want_stride + r / N;
            }
            d.pace = 1.0f / (float)(in.tiles_x + in.tiles_y);
            d.pad = 0u;
            a.rtile[in.tile_base + t] = d;
        }
    }
}

// With many sources: each one's cell marked in its tile's bits, so that a tile reads only its own.
// With every tile reading the whole list, 10^6 sources in 4096^2 took 7,980 us against 2,840 in the
// wave loop and 512 in each of 200 fields 3,450 against 1,560; with marks 1,200 and 1,640.  The line
// at kResFewSources (listed against marked): 1,024 sources in 256^2 81 and 84 us, in 1024^2 90 and 94,
// in 512^2 of 8x8 tiles 82 and 82; 4,096 of them 89 and 86, 98 and 97, 87 and 72.
template <int TW, int TH>
__global__ void k_resident_sources(ResidentArgs a, const GhcmInst* d_inst, const uint32_t* h_seeds) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < a.n_seeds; i += (size_t)gridDim.x * blockDim.x) {
        const uint32_t x = h_seeds[3 * i], y = h_seeds[3 * i + 1], j = h_seeds[3 * i + 2];
        mark_source<TW * TH>(a, resident_rank(d_inst[j], x / TW, y / TH), y % TH * TW + x % TW);
    }
}
inline dim3 sources_grid(uint32_t n) { return dim3(n < 256u * 4096u ? (n + 255u) / 256u : 4096u); }

template <int TW, int TH>
static hipError_t launch_init(const ResidentArgs& a, const GhcmInst* h_inst, GhcmInst* d_inst, const uint32_t* h_seeds,
                              uint32_t groups, uint32_t words, uint32_t states, int kind, hipStream_t s) {
    const dim3 grid(a.tiles < 1024u ? a.tiles : 1024u), block(256);
    if (kind <= 1)
        hipLaunchKernelGGL((k_resident_init<TW, TH, 4>), grid, block, 0, s, a, h_inst, d_inst, h_seeds, groups, words,
                           states);
    else
        hipLaunchKernelGGL((k_resident_init<TW, TH, 2>), grid, block, 0, s, a, h_inst, d_inst, h_seeds, groups, words,
                           states);
    if (many_sources(a.n_seeds))
        hipLaunchKernelGGL((k_resident_sources<TW, TH>), sources_grid(a.n_seeds), block, 0, s, a, d_inst, h_seeds);
    return hipGetLastError();
}

}  // namespace ghcm
