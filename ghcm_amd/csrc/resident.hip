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
//              tile lives in the time field.  Only the owner touches a tile, so its times need
//              no agent-scope access.  With few tiles the owner scans the borders that face its
//              closed tiles against seen[], what they were when it closed them; with many, who
//              publishes a border then lowers want[] of the tile across, which the owner reads
//              in one load for all its tiles and withdraws before it reads the borders: what is
//              announced after that the looks at the then open tile see.  Wants are times over
//              the tiles across the grid, so that the small and the large instances of a batch
//              advance alike (a batch of 512 12.1 -> 11.8 ms; the largest instances first, which
//              would shorten the end, 14.7 ms: tiles are then opened before all of a front is in).
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
// Measured (MI355X, whole calls, wave loop -> this): 256^2 rings 452 -> 217 us, 1531 x 977 smooth
// 813 -> 315, 2048^2 rings of contrast 1e4 4300 -> 1600, 2048^2 smooth 1020 -> 520, 4096^2
// smooth 1774 -> 950, a batch of 48 uneven fields (1,123 tiles) 845 -> 390, a batch of 512 (147 k
// tiles) 20.6 -> 10.3 ms.  There each SIMD has the sweeps of four work-groups to issue (15 vector
// instructions and a square root a step): vector issue takes 0.93 of the SIMDs' cycles.  Taken back:
// sweeping only the directions that the new border values or the unsettled cells ask for (12 %
// more rounds, and each as long as the latency of its steps, 12.4 against 11.9 ms).
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "ghcm_dev.h"
#include "resident.h"
#include "resident_dev.h"
#include "tile_dev.h"
#include "tile_geom.h"

namespace ghcm {

namespace {

// How a work-group learns that a closed tile of its own has new halo values: it has one tile
// (never closed), it scans the borders that face them all, or their neighbours' owners tell it.
enum : int { kOwnOne = 0, kOwnScan = 1, kOwnWant = 2 };

// Sweep steps between two exchanges: 8 against 16 and 32, 2048^2 contrast 1,800 against 1,870 and
// 2,400 us, smaller grids equal.
constexpr int kChunk = 8;
// With several tiles to a work-group the CUs are busy and a front is no longer waited for: 4096^2
// (four tiles each) 1,020 us at 16, 1,140 at 8, 1,280 at 32; a batch of 512 uneven fields (143)
// 11.8 ms at 16 and 32, 12.3 at 8.
constexpr int kChunkMany = 16;
// Sweep steps of a round: one ordered pass of all lanes (127) rounded up to the period of the
// wrapped skew, so that the next round takes up where this one ended.
constexpr int kSweepRound = 128;
// With several tiles to a work-group only the first round on a tile's new borders is that long and
// those after it half as long, one period of the skew: what is left to lower is little, and the
// sweeps of all the CU's work-groups share its issue slots.  Whole against half later rounds: 4096^2
// 1,130 against 1,020 us, 40 fields of up to 1200^2 1,910 against 1,700, the batch of 512 13.0
// against 11.9 ms; all rounds half 12.1 ms, and with one tile each 1531 x 977 355 against 338 us.
constexpr int kManyParts = 2;
// The largest `want` of a tile that is wanted (a product of finite times may overflow).
constexpr float kLatest = 3e38f;

// OR of `bits` over the four waves; one barrier.  Consecutive calls use different buffers.
__device__ __forceinline__ uint32_t wg_or(uint32_t bits, uint32_t* buf, int w, int L) {
    if (L == 0) buf[w] = bits;
    __syncthreads();
    return buf[0] | buf[1] | buf[2] | buf[3];
}

}  // namespace

template <int TW, int TH, int KIND, int OWN>
__global__ __launch_bounds__(kSweepThreads) __attribute__((amdgpu_waves_per_eu(4)))
void k_resident_sweep(ResidentArgs a) {
    constexpr int PW = TW + 2, PH = TH + 2, PP = PW * PH, CB = PP + 1;
    constexpr int CPT = TW * TH / kSweepThreads;
    constexpr int kEvery = OWN == kOwnOne ? kChunk : kChunkMany;
    constexpr int kParts = OWN == kOwnOne ? 1 : kManyParts, kSteps = kSweepRound / kParts;
    static_assert(kSteps % TH == 0, "a part takes up where the one before ended");
    __shared__ float sh[sweep_lds_words<TW, TH>()];
    __shared__ uint32_t s_or[3][4];
    __shared__ uint32_t s_cmd[2];
    __shared__ uint32_t s_pub;
    __shared__ uint32_t s_seeded[kResMaxOwned / 32];   // bit k: owned tile k holds a source
    __shared__ uint32_t s_opened[kResMaxOwned / 32];   // bit k: owned tile k has been opened
    __shared__ uint32_t s_best[2][4], s_bk[2][4];      // kOwnWant: each wave's smallest want, and whose it is
    __shared__ uint32_t s_key[OWN == kOwnScan ? kResMaxScan : 1];       // kOwnScan, of owned tile k: its
    __shared__ uint32_t s_tile[OWN == kOwnScan ? kResMaxScan : 1];      // neighbours' smallest new border value,
    __shared__ uint32_t s_from[OWN == kOwnScan ? kResMaxScan : 1][4];   // its id, the borders that face it
    float* const t_s = sh;
    float* const c_s = sh + CB;
    char* const shb = reinterpret_cast<char*>(sh);
    const int tid = threadIdx.x, L = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t b = blockIdx.x, N = gridDim.x, T = a.tiles;
    const float eps = a.eps;

    if (tid == 0) {
        if (last_in(a.ctl, kResArrived, b, N)) decide(a.ctl, 1u);
        s_pub = 0u;
    }
    if (tid < (int)(kResMaxOwned / 32)) s_seeded[tid] = s_opened[tid] = 0u;
    const uint64_t t_start = now_ticks();

    // ---- the tiles of this work-group ----
    const uint32_t m = (T - b + N - 1) / N;            // b < N <= T
    uint32_t* const want = a.want + (size_t)b * a.want_stride;
    if constexpr (OWN == kOwnScan) {
        if (tid < (int)m) {
            const ResTile& d = a.rtile[b + (uint32_t)tid * N];
            s_tile[tid] = d.g;
            for (int q = 0; q < 4; ++q) s_from[tid][q] = d.face[q];
            s_key[tid] = kInfBits;
        }
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
    auto seeded = [&](uint32_t k) {
        atomicOr(&s_seeded[k >> 5], 1u << (k & 31u));
        if constexpr (OWN == kOwnScan) s_key[k] = 0u;
        if constexpr (OWN == kOwnWant) st_agent(&want[k], 0u);
    };
    if (many_sources(a.n_seeds)) {
        if ((uint32_t)tid < m && holds_source<TW * TH>(a, b + (uint32_t)tid * N)) seeded((uint32_t)tid);
    } else {
        for (uint32_t i = tid; i < a.n_seeds; i += kSweepThreads) {
            const uint32_t r = a.seeds[4 * i + 3];
            if (r % N == b) seeded(r / N);
        }
    }
    wait_stores();
    __syncthreads();

    // ---- the open tile: in LDS, wave w keeping its side w ----
    uint32_t cur = kNoTile, cg = 0u, rounds = 0u, reached = 0u;
    int sx = 0, sy = 0, W = 0;
    char* tb = nullptr;
    bool act = false;
    int q_own = PW + 1, q_halo = 0;
    const uint32_t* from = a.edges;
    uint32_t* to = a.edges;
    float pace = 0.0f;                  // of the tile's times in `want`
    uint32_t* call = nullptr;           // the want of the tile across this side
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
    // Read owned tile k, write the open one back meanwhile, and put k in its place.
    auto open = [&](uint32_t k) {
        const ResTile d = uniform_tile(a.rtile + (b + k * N));
        // A tile opened for the first time is +INF but for its sources: nothing is read.
        const bool fresh = ((s_opened[k >> 5] >> (k & 31u)) & 1u) == 0u;
        const int nsx = (int)(d.ext & 0xFFu), nsy = (int)(d.ext >> 8);
        const char* const fb = static_cast<const char*>(d.field);
        char* const nt = reinterpret_cast<char*>(d.time);
        const int c = tid % TW, r0 = tid / TW;
        const int len = (w & 1) ? nsx : nsy;
        const uint32_t face = w == 0 ? d.face[0] : w == 1 ? d.face[1] : w == 2 ? d.face[2] : d.face[3];
        const uint32_t told = w == 0 ? d.call[0] : w == 1 ? d.call[1] : w == 2 ? d.call[2] : d.call[3];
        const bool nact = face != kNoTile && L < len;
        const uint32_t* const nfrom = a.edges + (size_t)(face == kNoTile ? 0u : face) * 64 + L;
        uint32_t* const nto = a.edges + ((size_t)d.g * 4 + w) * 64 + L;
        // Cells past the grid read the tile's first cell and become +INF (no load waits on a branch).
        float tv[CPT], cv[CPT];
#pragma unroll
        for (int j = 0; j < CPT; ++j) {
            const int r = r0 + (kSweepThreads / TW) * j;
            const uint32_t off = c < nsx && r < nsy ? (uint32_t)r * d.w + (uint32_t)c : 0u;
            cv[j] = load_cost_at<KIND>(fb + off * field_bytes<KIND>());
            tv[j] = __builtin_inff();
        }
        if (!fresh) {
#pragma unroll
            for (int j = 0; j < CPT; ++j) {
                const int r = r0 + (kSweepThreads / TW) * j;
                const uint32_t off = c < nsx && r < nsy ? (uint32_t)r * d.w + (uint32_t)c : 0u;
                tv[j] = *gmem(reinterpret_cast<const float*>(nt + off * 4u));
            }
        }
        const float nhalo = nact ? __uint_as_float(ld_agent(nfrom)) : __builtin_inff();
        const float nsent = nact ? __uint_as_float(ld_agent(nto)) : __builtin_inff();
        if (cur != kNoTile) {
            commit();
            if constexpr (OWN == kOwnScan) a.seen[(size_t)cg * 256 + w * 64 + L] = __float_as_uint(halo);
            __syncthreads();
        }
        cur = k;
        cg = d.g;
        sx = nsx;
        sy = nsy;
        W = (int)d.w;
        tb = nt;
        act = nact;
        from = nfrom;
        to = nto;
        if constexpr (OWN == kOwnWant) {
            call = a.want + told;
            pace = d.pace;
        }
        halo = nhalo;
        sent = nsent;
        // box words of lane L's border cell and of the halo cell across this side
        const int Lc = min(L, len - 1);
        q_own = w == 0 ? (Lc + 1) * PW + 1 : w == 2 ? (Lc + 1) * PW + sx : w == 1 ? PW + Lc + 1 : sy * PW + Lc + 1;
        q_halo = w == 0 ? q_own - 1 : w == 2 ? q_own + 1 : w == 1 ? q_own - PW : q_own + PW;
#pragma unroll
        for (int j = 0; j < CPT; ++j) {
            const int r = r0 + (kSweepThreads / TW) * j;
            const bool in_grid = c < sx && r < sy;
            t_s[(r + 1) * PW + c + 1] = in_grid ? tv[j] : __builtin_inff();
            c_s[(r + 1) * PW + c + 1] = in_grid ? cv[j] : __builtin_inff();
        }
        // A partial tile's last column or row has no neighbour; its far halo stays +INF.
        if (act) t_s[q_halo] = halo;
        else if (L < ((w & 1) ? TW : TH))
            t_s[w == 0 ? (L + 1) * PW : w == 2 ? (L + 1) * PW + PW - 1 : w == 1 ? L + 1 : (PH - 1) * PW + L + 1] = __builtin_inff();
        const bool sources = fresh && ((s_seeded[k >> 5] >> (k & 31u)) & 1u);
        __syncthreads();
        if (fresh && tid == 0) s_opened[k >> 5] |= 1u << (k & 31u);
        if (sources && many_sources(a.n_seeds)) {
#pragma unroll 1
            for (int i = tid; i < TW * TH; i += kSweepThreads)
                if (is_source<TW * TH>(a, b + k * N, (uint32_t)i)) t_s[(i / TW + 1) * PW + i % TW + 1] = 0.0f;
        } else if (sources) {
            for (uint32_t i = tid; i < a.n_seeds; i += kSweepThreads) {
                const int x = (int)(a.seeds[4 * i] - d.x0), y = (int)(a.seeds[4 * i + 1] - d.y0);
                if (a.seeds[4 * i + 2] == d.inst && x >= 0 && x < sx && y >= 0 && y < sy) t_s[(y + 1) * PW + x + 1] = 0.0f;
            }
        }
    };
    if (OWN == kOwnOne || m == 1u) open(0u);

    // ---- every work-group is running, or none goes on ----
    if (tid == 0) s_cmd[0] = await_decision(a.ctl, t_start);
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
    bool work = (OWN == kOwnOne || m == 1u) && (s_seeded[0] & 1u);
    while (go) {
        if (work) {
            __builtin_amdgcn_s_setprio(kWorkPriority);
            if (!(st & 1u)) {
                ++st;
                if (tid == 0) st_agent64(&a.state[b], ((unsigned long long)acked << 32) | st);
            }
            bool more, pub = false;
            float ahead = __builtin_inff();        // the neighbour's border cell, being loaded
            if (act) ahead = __uint_as_float(ld_agent(from));
            bool ch = false;
            // With several tiles to a work-group the neighbour's owner is told as well, once the
            // border is visible (at the next exchange): key is the smallest value not yet told.
            uint32_t key = kInfBits;
            auto tell = [&]() {
                if (OWN == kOwnWant && key != kInfBits) {
                    if (L == 0) __hip_atomic_fetch_min(call, key, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    key = kInfBits;
                }
            };
            auto publish = [&]() {
                const float mine = t_s[q_own];
                const bool out = act && __float_as_uint(mine) < __float_as_uint(sent) && __float_as_uint(mine) < __float_as_uint(halo);
                if (out) {
                    st_agent(to, __float_as_uint(mine));
                    sent = mine;
                }
                if (OWN == kOwnWant && __ballot(out))
                    key = min(key, __float_as_uint(fminf(pace * wave_min(out ? mine : __builtin_inff()), kLatest)));
            };
            auto exchange = [&]() {
                const float v = ahead;
                if constexpr (OWN == kOwnWant) {
                    // The load of `ahead` was issued after the last border store: both are done.
                    __asm__ volatile("" ::"v"(v) : "memory");
                    tell();
                }
                if (__float_as_uint(v) < __float_as_uint(halo)) {
                    halo = v;
                    t_s[q_halo] = v;
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
            bool first = true;
            do {
                ch = false;
                // The open tile's neighbours announce what the exchanges see by themselves.
                if (OWN == kOwnWant && tid == 0) st_agent(&want[cur], kInfBits);
                for (int part = first ? 0 : kParts - 1; part < kParts; ++part) {
                    switch (w) {
                        case 0: sweep_round<TW, TH, 1, true, kEvery, kSteps>(shb, L, exchange); break;
                        case 1: sweep_round<TW, TH, -1, true, kEvery, kSteps>(shb, L, exchange); break;
                        case 2: sweep_round<TW, TH, 1, false, kEvery, kSteps>(shb, L, exchange); break;
                        default: sweep_round<TW, TH, -1, false, kEvery, kSteps>(shb, L, exchange); break;
                    }
                }
                first = false;
                ++rounds;
                // The withdrawal is complete before the next look: a wave with a neighbour has waited
                // for loads that it issued later.
                if (OWN == kOwnWant && w == 0 && __ballot(act) == 0ull) wait_stores();
                const bool stop = (rounds & 1023u) == 0u && must_stop(a.ctl, a.cmd, b, N, t_start);
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
            if (OWN == kOwnWant && key != kInfBits) {
                wait_stores();
                tell();
            }
            work = false;
            __builtin_amdgcn_s_setprio(0);
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
            bool asked = false;                 // kOwnWant: the open tile's own want is set
            if (OWN == kOwnScan && m > 1u) {
                // the neighbours' borders of every closed tile, four tiles' loads at a time
                for (uint32_t k0 = 0; k0 < m; k0 += 4) {
                    float nv[4], sv[4];
#pragma unroll
                    for (uint32_t j = 0; j < 4; ++j) {
                        const uint32_t k = min(k0 + j, m - 1u);
                        const uint32_t fo = __builtin_amdgcn_readfirstlane(s_from[k][w]);
                        nv[j] = sv[j] = __builtin_inff();
                        // (cells past a partial tile's extent are never published and stay +INF)
                        if (k0 + j < m && k != cur && fo != kNoTile) {
                            nv[j] = __uint_as_float(ld_agent(a.edges + (size_t)fo * 64 + L));
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
            if (OWN == kOwnWant && m > 1u) {
                uint32_t own = (uint32_t)tid < m ? ld_agent(&want[tid]) : kInfBits;
                asked = (uint32_t)tid == cur && own != kInfBits;
                if (asked) {
                    // The borders it announces are visible and the next look reads them.
                    st_agent(&want[tid], kInfBits);
                    wait_stores();
                    own = kInfBits;
                }
                const float best = wave_min(__uint_as_float(own));
                const unsigned long long who = __ballot(own == __float_as_uint(best));
                if (L == 0) {
                    s_best[poll & 1u][w] = __float_as_uint(best);
                    s_bk[poll & 1u][w] = (uint32_t)(w * 64 + __builtin_ctzll(who));
                }
            }
            const bool ch = __float_as_uint(v) < __float_as_uint(halo);
            if (ch) {
                halo = v;
                t_s[q_halo] = v;
            }
            if (tid == 0) s_cmd[poll & 1u] = c;
            const uint32_t r = any4(bits | (__ballot(ch) ? 2u : 0u) | (__ballot(asked) ? 32u : 0u));
            cmd = s_cmd[poll & 1u];
            if (cmd == kCmdDone || cmd == kCmdAbort) break;
            if (r & 2u) {
                if (any4(__ballot(border_improves()) ? 1u : 0u)) {
                    work = true;
                    break;
                }
                continue;
            }
            if (r & 32u) continue;
            if (OWN != kOwnOne && m > 1u) {
                // the owned tile with the smallest new border value, if any has one
                uint32_t best = kInfBits, bk = 0u;
                if constexpr (OWN == kOwnScan) {
                    for (uint32_t k = 0; k < m; ++k) {
                        const uint32_t v2 = s_key[k];
                        if (v2 < best) { best = v2; bk = k; }
                    }
                    __syncthreads();        // every wave has read the keys
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const uint32_t v2 = s_best[poll & 1u][i];
                        if (v2 < best) { best = v2; bk = s_bk[poll & 1u][i]; }
                    }
                }
                best = __builtin_amdgcn_readfirstlane(best);
                bk = __builtin_amdgcn_readfirstlane(bk);
                if (best != kInfBits) {
                    // Each wave withdraws the want before it reads its side's border: open() waits
                    // for the tile's record first, which it reads after the withdrawal (the barrier
                    // to the compiler keeps it so, and vector memory completes in order).  What is
                    // announced later is seen by the looks at the open tile.
                    if constexpr (OWN == kOwnScan) {
                        if (tid == 0) s_key[bk] = kInfBits;
                    } else {
                        if (L == 0) st_agent(&want[bk], kInfBits);
                        __asm__ volatile("" ::: "memory");
                    }
                    // The visit counter turns odd before anything of the new tile is published.
                    if (!(st & 1u)) {
                        ++st;
                        if (tid == 0) st_agent64(&a.state[b], ((unsigned long long)acked << 32) | st);
                    }
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
            if ((s_opened[k >> 5] >> (k & 31u)) & 1u) continue;
            const ResTile d = uniform_tile(a.rtile + (b + k * N));
            const int ex = (int)(d.ext & 0xFFu), ey = (int)(d.ext >> 8);
            for (int i = tid; i < TW * TH; i += kSweepThreads) {
                const int x = i % TW, y = i / TW;
                if (x < ex && y < ey) gmem(d.time)[(size_t)y * d.w + x] = __builtin_inff();
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
        report_totals(a, sum_rounds, sum_rounds, sum_cells, most, !go || ld_agent(&a.ctl[kResFailed]) != 0u);
    }
}

template <int TW, int TH, int KIND, int OWN>
static hipError_t launch_own(const ResidentArgs& a, uint32_t groups, hipStream_t s, hipEvent_t ev0, hipEvent_t ev1) {
    if (ev0 && ev1)
        hipExtLaunchKernelGGL((k_resident_sweep<TW, TH, KIND, OWN>), dim3(groups), dim3(kSweepThreads), 0, s, ev0, ev1, 0, a);
    else
        hipLaunchKernelGGL((k_resident_sweep<TW, TH, KIND, OWN>), dim3(groups), dim3(kSweepThreads), 0, s, a);
    return hipGetLastError();
}

template <int TW, int TH, int KIND>
static hipError_t launch_resident_t(const ResidentArgs& a, uint32_t groups, hipStream_t s, hipEvent_t ev0, hipEvent_t ev1) {
    if (groups == 0 || groups > a.tiles || groups > kResMaxGroups || (uint64_t)a.tiles > (uint64_t)groups * kResMaxOwned)
        return hipErrorInvalidValue;
    if (a.tiles == groups) return launch_own<TW, TH, KIND, kOwnOne>(a, groups, s, ev0, ev1);
    if (a.seen) {
        if (a.tiles > groups * kResMaxScan) return hipErrorInvalidValue;
        return launch_own<TW, TH, KIND, kOwnScan>(a, groups, s, ev0, ev1);
    }
    if (!a.want || (uint64_t)groups * a.want_stride < a.tiles) return hipErrorInvalidValue;
    return launch_own<TW, TH, KIND, kOwnWant>(a, groups, s, ev0, ev1);
}

template <int TW, int TH, int KIND>
static int occ_resident_t() {
    int least = 0;
    auto with = [&](auto kernel) {
        int nb = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, kernel, kSweepThreads, 0) != hipSuccess) nb = 0;
        least = nb;
    };
    with(k_resident_sweep<TW, TH, KIND, kOwnOne>);
    int n = least;
    with(k_resident_sweep<TW, TH, KIND, kOwnScan>);
    n = least < n ? least : n;
    with(k_resident_sweep<TW, TH, KIND, kOwnWant>);
    return least < n ? least : n;
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

hipError_t launch_resident_init(const ResidentArgs& a, const GhcmInst* h_inst, GhcmInst* d_inst,
                                const uint32_t* h_seeds, uint32_t groups, int kind, hipStream_t s) {
    return launch_init<64, 64>(a, h_inst, d_inst, h_seeds, groups, 256u, kResMaxGroups, kind, s);
}

}  // namespace ghcm
