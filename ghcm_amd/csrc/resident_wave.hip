// resident_wave.hip -- the resident solve for the one-wave tiles (8x8, 16x16, 32x8, 32x32).
//
// In the wave loop these tiles are bound by latency: a launch of 13-80 us per tile crossing, in
// which one wave64 stages a tile in LDS, relaxes it a cell a pass and commits it.  Here a wave64
// keeps its tile in registers for the whole solve (lane L holds column L mod TW of TW TH / 64 rows)
// and waves never wait for one another: no LDS, no barrier, no launch per crossing.  Left and right
// neighbours come by DPP, rows above and below from the lane's own registers or by one
// ds_bpermute; a pass relaxes every cell (systolic and FIM tiles alike: what a FIM pass would skip
// costs nothing in a lane that is there anyway), rows down and up again.
//
//   inbox      each tile has one inbox, the cells across its four borders, each word written only
//              by the neighbour that owns the cell (agent-scope stores, published and read by the
//              rules of resident.hip).  A look at all neighbours is one run of 128 bytes for an
//              8x8 tile; its loads are in flight while kPasses passes run.
//   work       a tile is worked on from a cell that would improve by eps until none falls at all;
//              while it is idle none of its times changes.
//   end        as in resident.hip, the counters per tile and watched by a work-group of its own.
//
// Bound by the round trip of a border through the memory side (about 1 us) per crossing.  Measured
// (MI355X, whole calls, wave loop -> this): 512^2 rings in 8x8 systolic tiles 3,852 -> 1,169 us,
// 640 x 384 smooth in 16x16 FIM tiles 3,130 -> 359, 700 x 500 smooth in 8x8 / 16x16 / 32x8
// systolic and 32x32 FIM tiles 1,505 / 1,480 / 1,888 / 11,058 -> 417 / 434 / 459 / 979.
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

constexpr int kWaveGroup = 512;                      // threads of a work-group: eight tiles
constexpr uint32_t kTilesPerGroup = kWaveGroup / 64;
constexpr uint32_t kStatesPerThread = kResMaxWaveTiles / kWaveGroup;

// Rows of a lane: lane L holds column L mod TW, rows (L / TW) R .. + R - 1.
template <int TW, int TH>
constexpr int lane_rows() { return TW * TH / 64; }

// Words of a tile's inbox (x-, y-, x+, y+: the cells across each border) and where a side starts.
template <int TW, int TH>
constexpr uint32_t inbox_words() { return 2u * (TW + TH); }
template <int TW, int TH>
__host__ __device__ constexpr uint32_t inbox_side(int s) {
    return s == 0 ? 0u : s == 1 ? (uint32_t)TH : s == 2 ? (uint32_t)(TH + TW) : (uint32_t)(2 * TH + TW);
}

}  // namespace

template <int TW, int TH, int KIND>
__device__ __forceinline__ void resident_wave(const ResidentArgs& a) {
    constexpr int R = lane_rows<TW, TH>();
    // Passes between two looks, about one look's latency: for 8x8 tiles 2, 4, 6 and 9 of them 1,346,
    // 1,169, 1,182 and 1,246 us (512^2 rings), for 16x16 1, 2, 3 and 5 443, 358, 369 and 398 us (640 x
    // 384), for 32x32 1,034, 979, 1,112 and 1,360 us (700 x 500), 2,550, 2,700, 3,002 and 3,350 (1300^2).
    constexpr int kPasses = R == 1 ? 4 : 2;
    __shared__ uint32_t s_word;
    const int tid = threadIdx.x, L = tid & 63;
    const uint32_t G = gridDim.x - 1u, T = a.tiles;
    const float eps = a.eps;
    const float inf = __builtin_inff();

    // ---- every work-group is running, or none goes on ----
    const uint64_t t_start = now_ticks();
    if (tid == 0) {
        if (last_in(a.ctl, kResArrived, blockIdx.x, gridDim.x)) decide(a.ctl, 1u);
        s_word = await_decision(a.ctl, t_start);
    }
    __syncthreads();
    const bool go = s_word != 2u;
    __syncthreads();

    if (blockIdx.x == G) {
        // ---- the watcher ----
        if (go) {
            uint32_t phase = 0u, epoch = 0u, ver[kStatesPerThread];
#pragma unroll
            for (uint32_t k = 0; k < kStatesPerThread; ++k) ver[k] = 0u;
            for (;;) {
                bool busy = false, differs = false, unacked = false;
#pragma unroll
                for (uint32_t k = 0; k < kStatesPerThread; ++k) {
                    const uint32_t i = (uint32_t)tid + kWaveGroup * k;
                    if (i < T) {
                        const unsigned long long s = ld_agent64(&a.state[i]);
                        busy |= ((uint32_t)s & 1u) != 0u;
                        differs |= (uint32_t)s != ver[k];
                        unacked |= (uint32_t)(s >> 32) != epoch;
                        if (phase == 0u) ver[k] = (uint32_t)s;
                    }
                }
                const bool any_busy = __syncthreads_or(busy) != 0;
                const bool any_diff = __syncthreads_or(differs) != 0;
                const bool any_unacked = __syncthreads_or(unacked) != 0;
                uint32_t send = 0u;
                if (phase == 0u) {
                    if (!any_busy) {
                        send = ++epoch;
                        phase = 1u;
                    }
                } else if (any_busy || any_diff) {
                    phase = 0u;
                } else if (phase == 1u) {
                    if (!any_unacked) phase = 2u;
                } else {
                    send = kCmdDone;
                }
                if (tid == 0) s_word = send != kCmdDone && now_ticks() - t_start > kLimitTicks ? 1u : 0u;
                __syncthreads();
                if (s_word) {
                    send = kCmdAbort;
                    if (tid == 0) st_agent(&a.ctl[kResFailed], 1u);
                }
                if (send)
                    for (uint32_t i = tid; i < T; i += kWaveGroup) st_agent(&a.cmd[i], send);
                __syncthreads();
                if (send == kCmdDone || send == kCmdAbort) break;
                __builtin_amdgcn_s_sleep(1);
            }
            // every tile has left
            if (tid == 0)
                while (ld_agent(&a.ctl[kResLeft]) != min(T, kResSpread)) __builtin_amdgcn_s_sleep(4);
            __syncthreads();
        }
        __shared__ unsigned long long red[3][kWaveGroup];
        unsigned long long visits = 0, cells = 0, most = 0;
        if (go)
            for (uint32_t i = tid; i < T; i += kWaveGroup) {
                const unsigned long long v = ld_agent64(&a.report[i]);
                visits += (uint32_t)v;
                cells += v >> 32;
                if ((uint32_t)v > most) most = (uint32_t)v;
            }
        red[0][tid] = visits;
        red[1][tid] = cells;
        red[2][tid] = most;
        __syncthreads();
        for (int off = kWaveGroup / 2; off > 0; off >>= 1) {
            if (tid < off) {
                red[0][tid] += red[0][tid + off];
                red[1][tid] += red[1][tid + off];
                if (red[2][tid + off] > red[2][tid]) red[2][tid] = red[2][tid + off];
            }
            __syncthreads();
        }
        if (tid == 0) report_totals(a, red[0][0], red[0][0], red[1][0], (uint32_t)red[2][0], !go || ld_agent(&a.ctl[kResFailed]) != 0u);
        return;
    }
    const uint32_t rank = blockIdx.x + (uint32_t)(tid >> 6) * G;
    if (!go || rank >= T) return;

    // ---- the tile, in registers ----
    const ResTile d = uniform_tile(a.rtile + rank);
    const int x = L % TW, g = L / TW;
    const int sx = (int)(d.ext & 0xFFu), sy = (int)(d.ext >> 8);
    const bool left = x == 0, right = x == TW - 1, top = g == 0, bottom = g == 64 / TW - 1;
    const char* const fb = static_cast<const char*>(d.field);
    char* const tb = reinterpret_cast<char*>(d.time);
    float t[R], c[R], hx[R], ox[R];                // times, costs, x halo, x border as published
    float ht = inf, hb = inf, ot = inf, ob = inf;  // top and bottom halo, top and bottom border as published
#pragma unroll
    for (int k = 0; k < R; ++k) {
        const int r = g * R + k;
        const bool in_grid = x < sx && r < sy;
        const uint32_t off = in_grid ? (uint32_t)r * d.w + (uint32_t)x : 0u;
        const float v = load_cost_at<KIND>(fb + off * field_bytes<KIND>());
        c[k] = in_grid ? v : inf;
        t[k] = hx[k] = ox[k] = inf;
    }
    // This lane's words: the inbox cells it reads, and the neighbours' inbox cells it writes.
    const uint32_t* const in = a.edges + (size_t)d.g * inbox_words<TW, TH>();
    const uint32_t* const in_x = in + inbox_side<TW, TH>(left ? 0 : 2) + g * R;
    const uint32_t* const in_t = in + inbox_side<TW, TH>(1) + x;
    const uint32_t* const in_b = in + inbox_side<TW, TH>(3) + x;
    auto box = [&](int s) -> uint32_t* {
        return a.edges + (size_t)(d.face[s] == kNoTile ? 0u : d.face[s] >> 2) * inbox_words<TW, TH>() + inbox_side<TW, TH>(s ^ 2);
    };
    const bool has_x = (left && d.face[0] != kNoTile) || (right && d.face[2] != kNoTile);
    const bool has_t = top && d.face[1] != kNoTile, has_b = bottom && d.face[3] != kNoTile;
    uint32_t* const out_x = (left ? box(0) : box(2)) + g * R;
    uint32_t* const out_t = box(1) + x;
    uint32_t* const out_b = box(3) + x;

    bool work = many_sources(a.n_seeds) && holds_source<TW * TH>(a, rank) != 0u;
    if (work) {
#pragma unroll
        for (int k = 0; k < R; ++k)
            if (is_source<TW * TH>(a, rank, (uint32_t)((g * R + k) * TW + x))) t[k] = 0.0f;
    }
    for (uint32_t i0 = 0; i0 < (many_sources(a.n_seeds) ? 0u : a.n_seeds); i0 += 64) {
        const uint32_t i = min(i0 + (uint32_t)L, a.n_seeds - 1u);
        unsigned long long mine = __ballot(a.seeds[4 * i + 3] == rank);
        const uint32_t px = a.seeds[4 * i] - d.x0, py = a.seeds[4 * i + 1] - d.y0;
        work |= mine != 0ull;
        while (mine) {
            const int j = __builtin_ctzll(mine);
            mine &= mine - 1;
            const int qx = __builtin_amdgcn_readlane((int)px, j), qy = __builtin_amdgcn_readlane((int)py, j);
#pragma unroll
            for (int k = 0; k < R; ++k)
                if (x == qx && g * R + k == qy) t[k] = 0.0f;
        }
    }

    // The update of cell k from its four neighbours.
    auto update = [&](int k, float above, float below) -> float {
        // lanes 0 and 63 have no source lane and keep hx
        float l = __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(hx[k]), __float_as_int(t[k]), 0x138, 0xF, 0xF, false));
        float r = __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(hx[k]), __float_as_int(t[k]), 0x130, 0xF, 0xF, false));
        l = left ? hx[k] : l;
        r = right ? hx[k] : r;
        const float ax = umin_bits(l, r), ay = umin_bits(above, below);
        return godunov_raw(ax, ay, umin_bits(ax, ay), c[k]);
    };
    // The cells above and below this lane's.
    auto ends = [&](float& first, float& last) {
        const float pu = __int_as_float(__builtin_amdgcn_ds_bpermute(4 * (L - TW), __float_as_int(t[R - 1])));
        const float pd = __int_as_float(__builtin_amdgcn_ds_bpermute(4 * (L + TW), __float_as_int(t[0])));
        first = top ? ht : pu;
        last = bottom ? hb : pd;
    };
    // One pass over the tile, rows down and (with several rows to a lane) up again; whether a cell
    // fell.  Work on a tile goes on until none does, whatever eps: the passes are nearly free, and
    // changes below eps would otherwise add up along a front (640 x 384 1.41e-7 from FP64 at eps,
    // 1.02e-7 so, the wave loop 1.20e-7).
    auto pass = [&]() -> bool {
        float first, last;
        ends(first, last);
        bool fell = false;
        auto relax = [&](int k) {
            const float n = update(k, k ? t[k - 1] : first, k + 1 < R ? t[k + 1] : last);
            fell |= __float_as_uint(n) < __float_as_uint(t[k]);
            t[k] = umin_bits(t[k], n);
        };
#pragma unroll
        for (int k = 0; k < R; ++k) relax(k);
#pragma unroll
        for (int k = R - 2; k >= 0; --k) relax(k);
        return __ballot(fell) != 0ull;
    };
    // Whether a cell would improve by eps, which begins work on the tile.  No time changes: an
    // improvement below eps that was kept here would be published to no one, and the next one
    // would be measured against it, so that many of them left the neighbours behind without limit.
    auto unsettled = [&]() -> bool {
        float first, last;
        ends(first, last);
        bool imp = false;
#pragma unroll
        for (int k = 0; k < R; ++k)
            imp |= improves(update(k, k ? t[k - 1] : first, k + 1 < R ? t[k + 1] : last), t[k], eps);
        return __ballot(imp) != 0ull;
    };
    float nx[R], nt = inf, nb = inf;
#pragma unroll
    for (int k = 0; k < R; ++k) nx[k] = inf;
    auto look = [&]() {
        if (has_x) {
#pragma unroll
            for (int k = 0; k < R; ++k) nx[k] = __uint_as_float(ld_agent(in_x + k));
        }
        if (has_t) nt = __uint_as_float(ld_agent(in_t));
        if (has_b) nb = __uint_as_float(ld_agent(in_b));
    };
    // What the last look found that is new.
    auto take = [&]() -> bool {
        bool ch = __float_as_uint(nt) < __float_as_uint(ht) || __float_as_uint(nb) < __float_as_uint(hb);
        ht = umin_bits(ht, nt);
        hb = umin_bits(hb, nb);
#pragma unroll
        for (int k = 0; k < R; ++k) {
            ch |= __float_as_uint(nx[k]) < __float_as_uint(hx[k]);
            hx[k] = umin_bits(hx[k], nx[k]);
        }
        return __ballot(ch) != 0ull;
    };
    // Border cells that fell since they were last published, and below the cell across.
    auto publish = [&]() {
        if (has_x) {
#pragma unroll
            for (int k = 0; k < R; ++k)
                if (__float_as_uint(t[k]) < __float_as_uint(ox[k]) && __float_as_uint(t[k]) < __float_as_uint(hx[k])) {
                    st_agent(out_x + k, __float_as_uint(t[k]));
                    ox[k] = t[k];
                }
        }
        if (has_t && __float_as_uint(t[0]) < __float_as_uint(ot) && __float_as_uint(t[0]) < __float_as_uint(ht)) {
            st_agent(out_t, __float_as_uint(t[0]));
            ot = t[0];
        }
        if (has_b && __float_as_uint(t[R - 1]) < __float_as_uint(ob) && __float_as_uint(t[R - 1]) < __float_as_uint(hb)) {
            st_agent(out_b, __float_as_uint(t[R - 1]));
            ob = t[R - 1];
        }
    };

    uint32_t st = 1u, acked = 0u, pend = 0u, visits = 0u;
    auto put_state = [&]() {
        if (L == 0) st_agent64(&a.state[rank], ((unsigned long long)acked << 32) | st);
    };
    for (;;) {
        if (work) {
            __builtin_amdgcn_s_setprio(kWorkPriority);
            bool visible = (st & 1u) != 0u;         // (the first counter is odd from the start)
            if (!(st & 1u)) {
                ++st;
                put_state();
            }
            for (;;) {
                ++visits;
                look();
                bool more = false;
#pragma unroll 1
                for (int p = 0; p < kPasses; ++p) {
                    more = pass();
                    if (!more) break;
                }
                if (!visible) {
                    wait_stores();              // busy is visible before any border store
                    visible = true;
                }
                publish();
                more |= take();
                if ((visits & 1023u) == 0u && __ballot(must_stop(a.ctl, a.cmd, rank, T, t_start))) break;
                if (!more) break;
            }
            work = false;
            __builtin_amdgcn_s_setprio(0);
        }
        if (st & 1u) {
            wait_stores();
            ++st;
            put_state();
        }
        uint32_t cmd = 0u;
        for (;;) {
            look();
            cmd = __builtin_amdgcn_readfirstlane(ld_agent(&a.cmd[rank]));
            if (take()) {
                work = unsettled();
                if (work) break;
            } else if (cmd == kCmdDone || cmd == kCmdAbort) {
                break;
            } else if (cmd != acked) {
                if (cmd == pend) {
                    acked = cmd;
                    put_state();
                }
                pend = cmd;
            }
            if (cmd == kCmdAbort) break;
            __builtin_amdgcn_s_sleep(8);
        }
        if (!work) break;
    }
    // ---- write the tile and leave ----
    uint32_t reached = 0u;
#pragma unroll
    for (int k = 0; k < R; ++k) {
        const int r = g * R + k;
        if (x < sx && r < sy) {
            *gmem(reinterpret_cast<float*>(tb + ((uint32_t)r * d.w + (uint32_t)x) * 4u)) = t[k];
            reached += __float_as_uint(t[k]) < kInfBits ? 1u : 0u;
        }
    }
    reached = wave_sum(reached);
    if (L == 0) {
        st_agent64(&a.report[rank], ((unsigned long long)reached << 32) | visits);
        wait_stores();
        (void)last_in(a.ctl, kResLeft, rank, T);
    }
}

template <int TW, int TH, int KIND>
__global__ __launch_bounds__(kWaveGroup) void k_resident_wave(ResidentArgs a) {
    resident_wave<TW, TH, KIND>(a);
}
// 8x8 tiles, in at most 80 scalar registers: a SIMD has 800, handed out by 16, and 16 of each wave's
// are the trap handler's, so 80 let eight waves run on it and the 88 that the compiler takes by
// itself only seven -- three of these work-groups per CU instead of four, which the occupancy query
// does not know: grids of 6,137 to 8,184 tiles joined too few and went to the wave loop (640^2 to
// 744 x 704: 2,770-3,390 us; now 700-850).  Of 16x16 and
// 32x8 tiles the vector registers (79) allow six, of 32x32 (212 to 228) two: 6,136 and 2,040 tiles.
template <int KIND>
__global__ __launch_bounds__(kWaveGroup) __attribute__((amdgpu_num_sgpr(80))) void k_resident_wave8(ResidentArgs a) {
    resident_wave<8, 8, KIND>(a);
}
template <int TW, int TH, int KIND>
constexpr auto wave_kernel() {
    if constexpr (TW == 8 && TH == 8) return &k_resident_wave8<KIND>;
    else return &k_resident_wave<TW, TH, KIND>;
}

template <int TW, int TH, int KIND>
static hipError_t launch_wave_t(const ResidentArgs& a, uint32_t groups, hipStream_t s, hipEvent_t ev0, hipEvent_t ev1) {
    if (a.tiles == 0 || a.tiles > kResMaxWaveTiles || groups != (a.tiles + kTilesPerGroup - 1) / kTilesPerGroup)
        return hipErrorInvalidValue;
    if (ev0 && ev1)
        hipExtLaunchKernelGGL((wave_kernel<TW, TH, KIND>()), dim3(groups + 1), dim3(kWaveGroup), 0, s, ev0, ev1, 0, a);
    else
        hipLaunchKernelGGL((wave_kernel<TW, TH, KIND>()), dim3(groups + 1), dim3(kWaveGroup), 0, s, a);
    return hipGetLastError();
}

template <int TW, int TH, int KIND>
static int occ_wave_t() {
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, wave_kernel<TW, TH, KIND>(), kWaveGroup, 0) != hipSuccess)
        return 0;
    return nb;
}

template <int TW, int TH>
static hipError_t launch_wave_init_t(const ResidentArgs& a, const GhcmInst* h_inst, GhcmInst* d_inst, const uint32_t* h_seeds,
                                     int kind, hipStream_t s) {
    return launch_init<TW, TH>(a, h_inst, d_inst, h_seeds, a.tiles, inbox_words<TW, TH>(), kResMaxWaveTiles, kind, s);
}

template <int TW, int TH>
static ResidentWaveKernel pick_wave(int kind) {
    const uint32_t in = inbox_words<TW, TH>();
    switch (kind) {
        case 0: return {&launch_wave_t<TW, TH, 0>, &launch_wave_init_t<TW, TH>, &occ_wave_t<TW, TH, 0>, in};
        case 1: return {&launch_wave_t<TW, TH, 1>, &launch_wave_init_t<TW, TH>, &occ_wave_t<TW, TH, 1>, in};
        case 2: return {&launch_wave_t<TW, TH, 2>, &launch_wave_init_t<TW, TH>, &occ_wave_t<TW, TH, 2>, in};
        case 3: return {&launch_wave_t<TW, TH, 3>, &launch_wave_init_t<TW, TH>, &occ_wave_t<TW, TH, 3>, in};
    }
    return {nullptr, nullptr, nullptr, 0u};
}

ResidentWaveKernel get_resident_wave_kernel(int tw, int th, int kind, int mode) {
    if (mode != 0 && mode != 1) return {nullptr, nullptr, nullptr, 0u};
    if (tw == 8 && th == 8) return pick_wave<8, 8>(kind);
    if (tw == 16 && th == 16) return pick_wave<16, 16>(kind);
    if (tw == 32 && th == 8) return pick_wave<32, 8>(kind);
    if (tw == 32 && th == 32) return pick_wave<32, 32>(kind);
    return {nullptr, nullptr, nullptr, 0u};
}

}  // namespace ghcm
