// resident.hip -- the 2-D sweep solve without waves: one launch runs the whole solve.
//
// What bounds a plain solve is not bytes but the number of tiles a front crosses one after the
// other times the time of one crossing.  The wave loop pays per crossing a tile launch (control
// words, claim, staging from HBM, one sweep round of 127 dependent steps, commit), a boundary
// launch and two kernel gaps, 20-26 us, of which the sweep is 9.6 us, and a tile's new border
// reaches its neighbour only after all of it.  Here every work-group keeps its tile (time and
// cost) in LDS, work-groups meet only through the tiles' border cells in HBM, and a neighbour's
// new values enter a sweep that is already running.
//
//   borders    edges[tile][side][64]: a tile's border cells, stored with agent-scope (write
//              through) stores by the one work-group that owns the tile and read with
//              agent-scope loads by the owner of the neighbour.  Times only ever fall, so any
//              value read is a valid upper bound, a border needs no lock or flag, and new data
//              is its own message.  A cell is published only if it is below the neighbour's
//              adjacent cell (it cannot matter otherwise).
//   exchange   while a tile is swept, wave w looks after side w every kChunk steps: the
//              neighbour's border (loaded kChunk steps before, so no wait) goes into the halo in
//              LDS and the own border goes out.  A front crosses from tile to tile without
//              waiting for rounds to end.
//   settled    when kSweepRound steps brought no new halo value, every cell is checked once
//              against its four neighbours (0.9 us; another round of sweeps to see that nothing
//              changes takes 9.6 us).  Once nothing improves by eps the work-group only watches.
//   owners     with more tiles than resident work-groups (4 per CU: the LDS box is 34.9 KB),
//              tile r (in an order that shears the rows, so that a front in any direction meets
//              many work-groups) belongs to work-group r mod N, which has one of its tiles open
//              at a time and opens next the one with the smallest new border value.  A closed
//              tile lives in the time field; seen[] is what its neighbours' borders were.  Only
//              the owner touches a tile, so its times need no agent-scope access.
//   end        a work-group publishes a counter that is odd while it works: odd before its
//              first border store is issued, even after its last one is visible.  Work-group 0,
//              when idle, reads all counters; if all are even it sends an epoch, which a
//              work-group acknowledges after a complete look at its neighbours' borders, begun
//              after it saw the epoch, that found nothing new; if all acknowledge and no counter
//              moved, nothing is in flight: all borders were visible before the epoch and all
//              were seen.
//   residency  no work-group works before all N are running (they count themselves in); if that
//              takes over 200 us (other work holds the CUs) all leave at once and the caller runs
//              the wave loop.  Every wait ends: on the decision, on the end or on a 20 s limit.
//
// Measured (MI355X, whole calls, wave loop -> this): 256^2 rings 452 -> 231 us, 1531 x 977 smooth
// 813 -> 339, 2048^2 rings of contrast 1e4 4300 -> 1745, 2048^2 smooth 1020 -> 540, 4096^2
// smooth 1774 -> 1050, a batch of 48 uneven fields (1,123 tiles) 845 -> 400.
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "ghcm_dev.h"
#include "resident.h"
#include "tile_dev.h"
#include "tile_geom.h"

namespace ghcm {

namespace {

constexpr uint32_t kCmdDone = 0xFFFFFFFFu;
constexpr uint32_t kCmdAbort = 0xFFFFFFFEu;
// Sweep steps between two exchanges: 8 against 16 and 32, 4096^2 1,050 against 1,100 and 1,430 us,
// 2048^2 contrast 1,800 against 1,870 and 2,400 us, smaller grids equal.
constexpr int kChunk = 8;
// Sweep steps of a round: one ordered pass of all lanes (127) rounded up to the period of the
// wrapped skew, so that the next round takes up where this one ended.
constexpr int kSweepRound = 128;
constexpr uint64_t kJoinTicks = 20000;               // 200 us of the 100 MHz counter
constexpr uint64_t kLimitTicks = 2000000000ull;      // 20 s

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

// t improves on t0 by at least eps (strictly): times are compared as bits, so a NaN or a
// negative value never counts.
__device__ __forceinline__ bool improves(float t, float t0, float eps) {
    return __float_as_uint(t) < __float_as_uint(t0) && t0 - t >= eps;
}

__device__ __forceinline__ float umin_bits(float u, float v) {
    return __uint_as_float(min(__float_as_uint(u), __float_as_uint(v)));
}

// OR of `bits` over the four waves; one barrier.  Consecutive calls use different buffers.
__device__ __forceinline__ uint32_t wg_or(uint32_t bits, uint32_t* buf, int w, int L) {
    if (L == 0) buf[w] = bits;
    __syncthreads();
    return buf[0] | buf[1] | buf[2] | buf[3];
}

// Row y of an instance's tiles is rotated by y times this many tiles before the tiles are dealt
// out to the work-groups, so that a front along a column of tiles meets as many different
// work-groups (and XCDs) as one along a row.
__host__ __device__ __forceinline__ uint32_t resident_shear(uint32_t tiles_x) {
    return (tiles_x * 3u / 8u) | 1u;
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

// Whether some cell of the LDS tile would still improve from its four neighbours.
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

}  // namespace

template <int TW, int TH, int KIND>
__global__ __launch_bounds__(kSweepThreads) __attribute__((amdgpu_waves_per_eu(4)))
void k_resident_sweep(ResidentArgs a) {
    constexpr int PW = TW + 2, PH = TH + 2, PP = PW * PH, CB = PP + 1;
    constexpr int CPT = TW * TH / kSweepThreads;
    __shared__ float sh[sweep_lds_words<TW, TH>()];
    __shared__ uint32_t s_or[3][4];
    __shared__ uint32_t s_cmd[2];
    __shared__ uint32_t s_pub;
    __shared__ uint32_t s_seeded;                      // bit k: owned tile k holds a source
    __shared__ uint32_t s_key[kResMaxOwned];           // smallest new border value of an owned tile
    __shared__ uint32_t s_tile[kResMaxOwned];          // its id
    __shared__ uint32_t s_from[kResMaxOwned][4];       // its neighbours' facing borders (words of a.edges)
    float* const t_s = sh;
    float* const c_s = sh + CB;
    char* const shb = reinterpret_cast<char*>(sh);
    const int tid = threadIdx.x, L = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t b = blockIdx.x, N = gridDim.x, T = a.tiles;
    const float eps = a.eps;

    if (tid == 0) {
        if (last_in(a.ctl, kResArrived, b, N)) {
            uint32_t expect = 0u;
            __hip_atomic_compare_exchange_strong(&a.ctl[kResDecision], &expect, 1u, __ATOMIC_RELAXED,
                                                 __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        s_pub = 0u;
        s_seeded = 0u;
    }
    const uint64_t t_start = now_ticks();

    // ---- the tiles of this work-group ----
    const uint32_t m = (T - b + N - 1) / N;            // b < N <= T
    if (tid < (int)m) {
        const uint32_t r = b + (uint32_t)tid * N;
        const GhcmInst in = a.inst[a.n_inst == 1 ? 0u : a.tinst[r]];
        const uint32_t lr = r - in.tile_base, ty = lr / in.tiles_x;
        const uint32_t rot = (uint32_t)(((uint64_t)ty * resident_shear(in.tiles_x)) % in.tiles_x);
        uint32_t tx = lr - ty * in.tiles_x;
        tx = tx >= rot ? tx - rot : tx + in.tiles_x - rot;
        const uint32_t g = in.tile_base + ty * in.tiles_x + tx;
        s_tile[tid] = g;
        for (int s = 0; s < 4; ++s) {
            const uint32_t nb = tile_neighbour(in.tile_base, in.tiles_x, in.tiles_y, (int)tx, (int)ty, s);
            s_from[tid][s] = nb == kNoTile ? kNoTile : nb * 256u + (uint32_t)(s ^ 2) * 64u;
        }
        s_key[tid] = kInfBits;
    }
    // halo ring of the time box (the interior is staged whole)
    for (int i = tid; i < PW; i += kSweepThreads) {
        t_s[i] = __builtin_inff();
        t_s[(PH - 1) * PW + i] = __builtin_inff();
    }
    for (int i = tid; i < TH; i += kSweepThreads) {
        t_s[(i + 1) * PW] = __builtin_inff();
        t_s[(i + 1) * PW + PW - 1] = __builtin_inff();
    }

    __syncthreads();
    for (uint32_t i = tid; i < a.n_seeds; i += kSweepThreads) {
        const uint32_t x = a.seeds[3 * i], y = a.seeds[3 * i + 1];
        const GhcmInst in = a.inst[a.seeds[3 * i + 2]];
        const uint32_t g = tile_of_cell(in.tile_base, in.tiles_x, x, y, TW, TH);
        for (uint32_t k = 0; k < m; ++k)
            if (s_tile[k] == g) {
                s_key[k] = 0u;
                atomicOr(&s_seeded, 1u << k);
            }
    }
    __syncthreads();

    // ---- the open tile: in LDS, wave w keeping its side w ----
    uint32_t cur = kNoTile, cg = 0u, rounds = 0u, reached = 0u, opened = 0u;
    const uint32_t seeded = __builtin_amdgcn_readfirstlane(s_seeded);
    int sx = 0, sy = 0, W = 0;
    char* tb = nullptr;
    bool act = false;
    int q_own = PW + 1, q_halo = 0;
    const uint32_t* from = a.edges;
    uint32_t* to = a.edges;
    float halo = __builtin_inff();      // the neighbour's border cell, as last read
    float sent = __builtin_inff();      // this tile's border cell, as last published

    // Write the open tile back.
    auto commit = [&]() {
#pragma unroll
        for (int k = 0; k < CPT; ++k) {
            const int r = (tid + kSweepThreads * k) / TW, c = tid % TW;
            if (c < sx && r < sy) {
                const float t = t_s[(r + 1) * PW + c + 1];
                *gmem(reinterpret_cast<float*>(tb + ((uint32_t)r * (uint32_t)W + (uint32_t)c) * 4u)) = t;
                reached += __float_as_uint(t) < kInfBits ? 1u : 0u;
            }
        }
    };
    // Read owned tile k into LDS; its halo and its published borders go to registers.
    auto open = [&](uint32_t k) {
        cur = k;
        cg = __builtin_amdgcn_readfirstlane(s_tile[k]);
        const uint32_t ii = a.n_inst == 1 ? 0u : __builtin_amdgcn_readfirstlane(a.tinst[cg]);
        const GhcmInst in = uniform_inst(a.inst[ii]);
        // A tile opened for the first time is +INF but for its sources: nothing is read.
        const bool fresh = ((opened >> k) & 1u) == 0u;
        opened |= 1u << k;
        int tx, ty;
        tile_xy(cg - in.tile_base, in.tiles_x, tx, ty);
        const int ox = tx * TW, oy = ty * TH;
        W = (int)in.w;
        sx = tile_extent(W, ox, TW);
        sy = tile_extent((int)in.h, oy, TH);
        tb = reinterpret_cast<char*>(in.time) + ((int64_t)oy * W + ox) * 4;
        const char* const fb = static_cast<const char*>(in.field) + ((int64_t)oy * W + ox) * (int64_t)field_bytes<KIND>();
        const int len = (w & 1) ? sx : sy;
        const uint32_t fo = __builtin_amdgcn_readfirstlane(s_from[k][w]);
        act = fo != kNoTile && L < len;
        from = a.edges + (fo == kNoTile ? 0u : fo) + L;
        to = a.edges + (size_t)cg * 256 + (size_t)w * 64 + L;
        // box words of lane L's border cell and of the halo cell across this side
        const int Lc = min(L, len - 1);
        q_own = w == 0 ? (Lc + 1) * PW + 1 : w == 2 ? (Lc + 1) * PW + sx : w == 1 ? PW + Lc + 1 : sy * PW + Lc + 1;
        q_halo = w == 0 ? q_own - 1 : w == 2 ? q_own + 1 : w == 1 ? q_own - PW : q_own + PW;
        halo = act ? __uint_as_float(ld_agent(from)) : __builtin_inff();
        sent = act ? __uint_as_float(ld_agent(to)) : __builtin_inff();
        // Cells past the grid read the tile's first cell and become +INF (no load waits on a branch).
        constexpr int kBatch = CPT / 2;
#pragma unroll 1
        for (int k0 = 0; k0 < CPT; k0 += kBatch) {
            float tv[kBatch], cv[kBatch];
            const int c = tid % TW, r0 = tid / TW + (kSweepThreads / TW) * k0;
#pragma unroll
            for (int j = 0; j < kBatch; ++j) {
                const int r = r0 + (kSweepThreads / TW) * j;
                const uint32_t off = c < sx && r < sy ? (uint32_t)r * (uint32_t)W + (uint32_t)c : 0u;
                cv[j] = load_cost_at<KIND>(fb + off * field_bytes<KIND>());
                tv[j] = __builtin_inff();
            }
            if (!fresh) {
#pragma unroll
                for (int j = 0; j < kBatch; ++j) {
                    const int r = r0 + (kSweepThreads / TW) * j;
                    const uint32_t off = c < sx && r < sy ? (uint32_t)r * (uint32_t)W + (uint32_t)c : 0u;
                    tv[j] = *gmem(reinterpret_cast<const float*>(tb + off * 4u));
                }
            }
#pragma unroll
            for (int j = 0; j < kBatch; ++j) {
                const int r = r0 + (kSweepThreads / TW) * j;
                const bool in_grid = c < sx && r < sy;
                t_s[(r + 1) * PW + c + 1] = in_grid ? tv[j] : __builtin_inff();
                c_s[(r + 1) * PW + c + 1] = in_grid ? cv[j] : __builtin_inff();
            }
        }
        // A partial tile's last column or row has no neighbour; its far halo stays +INF.
        if (act) t_s[q_halo] = halo;
        else if (L < ((w & 1) ? TW : TH))
            t_s[w == 0 ? (L + 1) * PW : w == 2 ? (L + 1) * PW + PW - 1 : w == 1 ? L + 1 : (PH - 1) * PW + L + 1] = __builtin_inff();
        if (fresh && ((seeded >> k) & 1u)) {
            __syncthreads();
            for (uint32_t i = tid; i < a.n_seeds; i += kSweepThreads) {
                const int x = (int)a.seeds[3 * i] - ox, y = (int)a.seeds[3 * i + 1] - oy;
                if (a.seeds[3 * i + 2] == ii && x >= 0 && x < sx && y >= 0 && y < sy) t_s[(y + 1) * PW + x + 1] = 0.0f;
            }
        }
    };
    if (m == 1u) open(0u);

    // ---- every work-group is running, or none goes on ----
    if (tid == 0) {
        uint32_t d;
        while ((d = ld_agent(&a.ctl[kResDecision])) == 0u) {
            if (now_ticks() - t_start > kJoinTicks) {
                uint32_t expect = 0u;
                if (__hip_atomic_compare_exchange_strong(&a.ctl[kResDecision], &expect, 2u, __ATOMIC_RELAXED,
                                                         __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
                    st_agent(&a.ctl[kResFailed], 1u);
            }
            __builtin_amdgcn_s_sleep(4);
        }
        s_cmd[0] = d;
    }
    __syncthreads();
    const bool go = s_cmd[0] != 2u;
    __syncthreads();

    // Whether lane L's border cell would improve, given the whole box.
    auto border_improves = [&]() -> bool {
        if (!act) return false;
        const float ax = umin_bits(t_s[q_own - 1], t_s[q_own + 1]);
        const float ay = umin_bits(t_s[q_own - PW], t_s[q_own + PW]);
        return improves(godunov_raw(ax, ay, umin_bits(ax, ay), c_s[q_own]), t_s[q_own], eps);
    };

    uint32_t st = 1u, acked = 0u, pend = 0u, cmd = 0u;
    int ob = 0;
    auto any4 = [&](uint32_t bits) -> uint32_t {
        const uint32_t r = wg_or(bits, s_or[ob], w, L);
        ob = ob == 2 ? 0 : ob + 1;
        return r;
    };
    // watcher (work-group 0)
    uint32_t phase = 0u, epoch = 0u, ver[kResMaxGroups / kSweepThreads];
#pragma unroll
    for (uint32_t k = 0; k < kResMaxGroups / kSweepThreads; ++k) ver[k] = 0u;
    uint32_t poll = 0;
    // The open tile has cells that would improve.
    bool work = m == 1u && seeded != 0u;
    while (go) {
        if (work) {
            if (!(st & 1u)) {
                ++st;
                if (tid == 0) st_agent64(&a.state[b], ((unsigned long long)acked << 32) | st);
            }
            bool more, pub = false;
            float ahead = __builtin_inff();        // the neighbour's border cell, being loaded
            if (act) ahead = __uint_as_float(ld_agent(from));
            bool ch = false;
            auto publish = [&]() {
                const float mine = t_s[q_own];
                if (act && __float_as_uint(mine) < __float_as_uint(sent) && __float_as_uint(mine) < __float_as_uint(halo)) {
                    st_agent(to, __float_as_uint(mine));
                    sent = mine;
                }
            };
            auto exchange = [&]() {
                if (__float_as_uint(ahead) < __float_as_uint(halo)) {
                    halo = ahead;
                    t_s[q_halo] = ahead;
                    ch = true;
                }
                if (!pub) {
                    if (w == 0) {
                        wait_stores();              // busy is visible before any border store
                        pub = true;
                        if (L == 0) __hip_atomic_store(&s_pub, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                    } else {
                        pub = __hip_atomic_load(&s_pub, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) != 0u;
                    }
                }
                if (pub) publish();
                if (act) ahead = __uint_as_float(ld_agent(from));
            };
            // Rounds go on while they bring new halo values; after one that brought none, the
            // box is checked cell by cell.
            do {
                ch = false;
                switch (w) {
                    case 0: sweep_round<TW, TH, 1, true, kChunk, kSweepRound>(shb, L, exchange); break;
                    case 1: sweep_round<TW, TH, -1, true, kChunk, kSweepRound>(shb, L, exchange); break;
                    case 2: sweep_round<TW, TH, 1, false, kChunk, kSweepRound>(shb, L, exchange); break;
                    default: sweep_round<TW, TH, -1, false, kChunk, kSweepRound>(shb, L, exchange); break;
                }
                ++rounds;
                const bool stop = (rounds & 1023u) == 0u && ld_agent(&a.cmd[b]) == kCmdAbort;
                uint32_t r = any4((__ballot(ch) ? 1u : 0u) | (__ballot(stop) ? 4u : 0u));
                if (!(r & 1u)) {
                    pub = true;
                    publish();
                    const bool fresh = __float_as_uint(ahead) < __float_as_uint(halo);
                    if (fresh) {
                        halo = ahead;
                        t_s[q_halo] = ahead;
                    }
                    if (act) ahead = __uint_as_float(ld_agent(from));
                    const bool res = tile_unsettled<TW, TH>(t_s, c_s, w, L, eps);
                    r |= any4((__ballot(res) ? 1u : 0u) | (__ballot(fresh) ? 2u : 0u));
                    if ((r & 3u) == 2u) r |= any4(__ballot(border_improves()) ? 1u : 0u);
                    more = (r & 5u) == 1u;
                } else {
                    more = (r & 4u) == 0u;
                }
            } while (more);
            work = false;
        }
        // ---- look at every owned tile's neighbours ----
        bool idle = false;
        for (;;) {
            ++poll;
            float v = __builtin_inff();
            if (act) v = __uint_as_float(ld_agent(from));
            uint32_t c = 0u;
            if (w == 0) c = ld_agent(&a.cmd[b]);
            uint32_t bits = 0u;
            if (b == 0 && idle) {
                bool busy = false, differs = false, unacked = false;
#pragma unroll
                for (uint32_t k = 0; k < kResMaxGroups / kSweepThreads; ++k) {
                    const uint32_t i = (uint32_t)tid + kSweepThreads * k;
                    if (i < N) {
                        const unsigned long long s = ld_agent64(&a.state[i]);
                        busy |= ((uint32_t)s & 1u) != 0u;
                        differs |= (uint32_t)s != ver[k];
                        unacked |= (uint32_t)(s >> 32) != epoch;
                        if (phase == 0u) ver[k] = (uint32_t)s;
                    }
                }
                bits = (__ballot(busy) ? 4u : 0u) | (__ballot(differs) ? 8u : 0u) | (__ballot(unacked) ? 16u : 0u);
            }
            if (m > 1u) {
                // four tiles' loads at a time
                for (uint32_t k0 = 0; k0 < m; k0 += 4) {
                    float nv[4], sv[4];
#pragma unroll
                    for (uint32_t j = 0; j < 4; ++j) {
                        const uint32_t k = min(k0 + j, m - 1u);
                        const uint32_t fo = __builtin_amdgcn_readfirstlane(s_from[k][w]);
                        nv[j] = sv[j] = __builtin_inff();
                        // (cells past a partial tile's extent are never published and stay +INF)
                        if (k0 + j < m && k != cur && fo != kNoTile) {
                            nv[j] = __uint_as_float(ld_agent(a.edges + fo + L));
                            sv[j] = __uint_as_float(a.seen[(size_t)__builtin_amdgcn_readfirstlane(s_tile[k]) * 256 + w * 64 + L]);
                        }
                    }
#pragma unroll
                    for (uint32_t j = 0; j < 4; ++j) {
                        const bool lower = __float_as_uint(nv[j]) < __float_as_uint(sv[j]);
                        if (__ballot(lower)) {
                            const float key = wave_min(lower ? nv[j] : __builtin_inff());
                            if (L == 0)
                                __hip_atomic_fetch_min(&s_key[k0 + j], __float_as_uint(key), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                        }
                    }
                }
            }
            const bool ch = __float_as_uint(v) < __float_as_uint(halo);
            if (ch) {
                halo = v;
                t_s[q_halo] = v;
            }
            if (tid == 0) s_cmd[poll & 1u] = c;
            const uint32_t r = any4(bits | (__ballot(ch) ? 2u : 0u));
            cmd = s_cmd[poll & 1u];
            if (cmd == kCmdDone || cmd == kCmdAbort) break;
            if (r & 2u) {
                if (any4(__ballot(border_improves()) ? 1u : 0u)) {
                    work = true;
                    break;
                }
                continue;
            }
            if (m > 1u) {
                // the owned tile with the smallest new value, if any has one
                uint32_t best = kInfBits, bk = 0u;
                for (uint32_t k = 0; k < m; ++k) {
                    const uint32_t key = s_key[k];
                    if (key < best) { best = key; bk = k; }
                }
                best = __builtin_amdgcn_readfirstlane(best);
                bk = __builtin_amdgcn_readfirstlane(bk);
                __syncthreads();        // every wave has read the keys
                if (best != kInfBits) {
                    if (tid == 0) s_key[bk] = kInfBits;
                    // The visit counter turns odd before anything of the new tile is published.
                    if (!(st & 1u)) {
                        ++st;
                        if (tid == 0) st_agent64(&a.state[b], ((unsigned long long)acked << 32) | st);
                    }
                    if (cur != kNoTile) {
                        commit();
                        a.seen[(size_t)cg * 256 + w * 64 + L] = __float_as_uint(halo);
                    }
                    wait_stores();
                    __syncthreads();
                    open(bk);
                    __syncthreads();
                    idle = false;
                    if (any4(__ballot(best == 0u || border_improves()) ? 1u : 0u)) {
                        work = true;
                        break;
                    }
                    continue;
                }
            }
            if (!idle) {
                // Nothing left here: every border published so far is visible, then idle is.
                idle = true;
                if (st & 1u) {
                    wait_stores();
                    __syncthreads();
                    if (tid == 0) s_pub = 0u;
                    ++st;
                    if (tid == 0) st_agent64(&a.state[b], ((unsigned long long)acked << 32) | st);
                }
                phase = 0u;
                continue;
            }
            if (cmd != acked) {
                if (cmd == pend) {
                    acked = cmd;
                    if (tid == 0) st_agent64(&a.state[b], ((unsigned long long)acked << 32) | st);
                }
                pend = cmd;
            }
            if (b == 0) {
                uint32_t send = 0u;
                if (phase == 0u) {
                    if (!(r & 4u)) {
                        send = ++epoch;
                        phase = 1u;
                    }
                } else if (r & (4u | 8u)) {
                    phase = 0u;
                } else if (phase == 1u) {
                    if (!(r & 16u)) phase = 2u;
                } else {
                    send = kCmdDone;
                }
                if (send != kCmdDone && now_ticks() - t_start > kLimitTicks) {
                    send = kCmdAbort;
                    if (tid == 0) st_agent(&a.ctl[kResFailed], 1u);
                }
                if (send)
                    for (uint32_t i = tid; i < N; i += kSweepThreads) st_agent(&a.cmd[i], send);
            }
            __builtin_amdgcn_s_sleep(2);
        }
        if (!work) break;
    }
    if (go) {
        if (cur != kNoTile) commit();
        // Tiles that no front reached.
        for (uint32_t k = 0; k < m; ++k) {
            if ((opened >> k) & 1u) continue;
            const uint32_t g = s_tile[k];
            const GhcmInst in = uniform_inst(a.inst[a.n_inst == 1 ? 0u : a.tinst[g]]);
            int tx, ty;
            tile_xy(g - in.tile_base, in.tiles_x, tx, ty);
            const int ox = tx * TW, oy = ty * TH;
            for (int i = tid; i < TW * TH; i += kSweepThreads) {
                const int x = ox + i % TW, y = oy + i / TW;
                if (x < (int)in.w && y < (int)in.h) gmem(in.time)[(size_t)y * in.w + x] = __builtin_inff();
            }
        }
    }
    // ---- leave: the last work-group out reports the solve ----
    reached = wave_sum(reached);
    if (L == 0) s_or[0][w] = reached;
    __syncthreads();
    if (tid == 0) {
        const uint32_t n = s_or[0][0] + s_or[0][1] + s_or[0][2] + s_or[0][3];
        st_agent64(&a.report[b], ((unsigned long long)n << 32) | rounds);
        wait_stores();
        s_cmd[0] = last_in(a.ctl, kResLeft, b, N) ? 1u : 0u;
    }
    __syncthreads();
    if (s_cmd[0] == 0u) return;
    unsigned long long sum_rounds = 0, sum_cells = 0;
    uint32_t most = 0;
    for (uint32_t i = tid; i < N; i += kSweepThreads) {
        const unsigned long long v = ld_agent64(&a.report[i]);
        sum_rounds += (uint32_t)v;
        sum_cells += v >> 32;
        most = max(most, (uint32_t)v);
    }
    unsigned long long* const red = reinterpret_cast<unsigned long long*>(sh);
    red[tid] = sum_rounds;
    red[kSweepThreads + tid] = sum_cells;
    red[2 * kSweepThreads + tid] = most;
    __syncthreads();
    if (tid == 0) {
        for (int i = 1; i < kSweepThreads; ++i) {
            sum_rounds += red[i];
            sum_cells += red[kSweepThreads + i];
            most = max(most, (uint32_t)red[2 * kSweepThreads + i]);
        }
        sys_store64(&a.rec->totals[0], sum_rounds);
        sys_store64(&a.rec->totals[1], sum_rounds);
        sys_store64(&a.rec->totals[2], sum_cells);
        sys_store(&a.rec->wave, ld_agent(&a.ctl[kResFailed]));
        sys_store(&a.rec->busy_waves, most);
        __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
        sys_store(&a.rec->totals_tag, a.tag);
    }
}

// The state of a resident solve, in one launch: instance table, tile map and sources copied
// from mapped host memory, borders at +INF, every work-group counted as busy.
__global__ void k_resident_init(ResidentArgs a, const GhcmInst* h_inst, const uint32_t* h_seeds) {
    const size_t i0 = (size_t)blockIdx.x * blockDim.x + threadIdx.x, stride = (size_t)gridDim.x * blockDim.x;
    const uint4 inf4 = make_uint4(kInfBits, kInfBits, kInfBits, kInfBits);
    uint4* const e4 = reinterpret_cast<uint4*>(a.edges);
    uint4* const s4 = reinterpret_cast<uint4*>(a.seen);
    for (size_t i = i0; i < (size_t)a.tiles * 64; i += stride) {
        e4[i] = inf4;
        s4[i] = inf4;
    }
    for (size_t i = i0; i < kResMaxGroups; i += stride) {
        a.state[i] = 1ull;
        a.cmd[i] = 0u;
    }
    for (size_t i = i0; i < kResCtlWords; i += stride) a.ctl[i] = 0u;
    for (size_t i = i0; i < 3ull * a.n_seeds; i += stride) const_cast<uint32_t*>(a.seeds)[i] = h_seeds[i];
    for (uint32_t j = blockIdx.x; j < a.n_inst; j += gridDim.x) {
        const GhcmInst in = h_inst[j];
        if (threadIdx.x == 0) const_cast<GhcmInst*>(a.inst)[j] = in;
        if (a.tinst)
            for (uint32_t t = threadIdx.x; t < inst_tiles(in); t += blockDim.x)
                const_cast<uint32_t*>(a.tinst)[in.tile_base + t] = j;
    }
}

template <int TW, int TH, int KIND>
static hipError_t launch_resident_t(const ResidentArgs& a, uint32_t groups, hipStream_t s, hipEvent_t ev0, hipEvent_t ev1) {
    if (groups == 0 || groups > a.tiles || groups > kResMaxGroups || a.tiles > groups * kResMaxOwned)
        return hipErrorInvalidValue;
    if (ev0 && ev1)
        hipExtLaunchKernelGGL((k_resident_sweep<TW, TH, KIND>), dim3(groups), dim3(kSweepThreads), 0, s, ev0, ev1, 0, a);
    else
        hipLaunchKernelGGL((k_resident_sweep<TW, TH, KIND>), dim3(groups), dim3(kSweepThreads), 0, s, a);
    return hipGetLastError();
}

template <int TW, int TH, int KIND>
static int occ_resident_t() {
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k_resident_sweep<TW, TH, KIND>, kSweepThreads, 0) != hipSuccess)
        return 0;
    return nb;
}

ResidentKernel get_resident_kernel(int tw, int th, int kind, int mode) {
    if (mode != 2 || tw != 64 || th != 64) return {nullptr, nullptr};
    switch (kind) {
        case 0: return {&launch_resident_t<64, 64, 0>, &occ_resident_t<64, 64, 0>};
        case 1: return {&launch_resident_t<64, 64, 1>, &occ_resident_t<64, 64, 1>};
        case 2: return {&launch_resident_t<64, 64, 2>, &occ_resident_t<64, 64, 2>};
        case 3: return {&launch_resident_t<64, 64, 3>, &occ_resident_t<64, 64, 3>};
    }
    return {nullptr, nullptr};
}

hipError_t launch_resident_init(const ResidentArgs& a, const GhcmInst* h_inst, const uint32_t* h_seeds,
                                hipStream_t s) {
    const uint32_t blocks = a.tiles < 1024u ? a.tiles : 1024u;
    hipLaunchKernelGGL(k_resident_init, dim3(blocks), dim3(256), 0, s, a, h_inst, h_seeds);
    return hipGetLastError();
}

}  // namespace ghcm
