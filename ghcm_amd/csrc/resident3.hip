// resident3.hip -- the resident solve for 3-D sweep tiles (64 x 8 x 8), by the rules of resident.hip:
// a work-group of eight wave64s keeps its tile in LDS (two to a CU: the boxes are 55.6 KB), each
// wave sweeps one octant and looks after four or five of the tile's 34 border rows of 64 cells,
// which go out and come in every kChunk3 steps; a round without new halo values is followed by a
// check of every cell.
//
// For volumes of at most one tile per resident work-group (512 on 256 CUs), where a wave is bound
// by the latency of one visit (29 us, of which the round of sweeps is 14).  Measured (MI355X, whole
// calls, wave loop -> this): 150 x 90 x 61 (288 tiles) 888 -> 432 us, 70 x 200 x 60 (400 tiles) 828 ->
// 503 us.  Larger volumes are bound by the sweeps' issue slots (two waves per SIMD to a work-group),
// and starting a round for every new border then costs more than waves of visits do: with several
// tiles to a work-group 256 x 128 x 128 1,700 against 1,675 us, 256^3 6,430 against 3,910.
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "ghcm_dev.h"
#include "resident.h"
#include "resident_dev.h"
#include "tile3_dev.h"
#include "tile_dev.h"

namespace ghcm {

namespace {

// Steps between two exchanges, and of a round: one period of the skew, so that every lane relaxes
// every cell of its row once and the next round takes up where this one ended.  150 x 90 x 61 at
// 80 steps and 20 between exchanges 505 us, 80 / 8 463, 128 / 16 490, 64 / 16 455, 64 / 8 447.
constexpr int kChunk3 = 8;
constexpr int kRound3 = 64;
static_assert(kRound3 % kS3X == 0, "a round covers every cell, or unsettled ones are swept for ever");
constexpr int kBlocks3 = 5;       // border rows a wave looks after (34 over eight waves)

// OR of `bits` over the eight waves; one barrier.  Consecutive calls use different buffers.
__device__ __forceinline__ uint32_t wg_or8(uint32_t bits, uint32_t* buf, int w, int L) {
    if (L == 0) buf[w] = bits;
    __syncthreads();
    return (buf[0] | buf[1]) | (buf[2] | buf[3]) | (buf[4] | buf[5]) | (buf[6] | buf[7]);
}

// Tiles are dealt out plane by plane, each plane rotated against the one before.
__device__ __forceinline__ uint32_t rank3(uint32_t nx, uint32_t ny, uint32_t tx, uint32_t ty, uint32_t tz) {
    const uint32_t P = nx * ny, p = tx + nx * ty;
    const uint32_t rot = (uint32_t)(((uint64_t)tz * shear(P)) % P);
    return tz * P + (p + rot >= P ? p + rot - P : p + rot);
}

}  // namespace

template <int KIND>
__global__ __launch_bounds__(kS3Threads) __attribute__((amdgpu_waves_per_eu(4)))
void k_resident_sweep3(Resident3Args a) {
    constexpr int PX = kS3PX, PL = kS3Plane;
    __shared__ float sh[2 * kS3Box];
    __shared__ uint32_t s_or[3][8];
    __shared__ uint32_t s_cmd[2];
    __shared__ uint32_t s_pub;
    float* const t_s = sh;
    float* const c_s = sh + kS3Box;
    char* const shb = reinterpret_cast<char*>(sh);
    const int tid = threadIdx.x, L = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t b = blockIdx.x, N = gridDim.x;
    const float eps = a.eps;
    const float inf = __builtin_inff();

    if (tid == 0) {
        if (last_in(a.ctl, kResArrived, b, N)) decide(a.ctl, 1u);
        s_pub = 0u;
    }
    const uint64_t t_start = now_ticks();
    // The whole time box at +INF: its edges and corners are never written again.
    for (int i = tid; i < kS3Box; i += kS3Threads) t_s[i] = inf;
    __syncthreads();

    // ---- the tile: in LDS; wave w keeps border rows w, w + 8, ... of the 34 ----
    // Border row bi: 0 x-, 1 x+ (lane = y + 8 z), 2-9 y- and 10-17 y+ (plane by plane, lane = x),
    // 18-25 z- and 26-33 z+ (row by row, lane = x).
    const ResTile3 d = uniform_tile(a.rtile + b);
    const int sx = (int)(d.ext & 0xFFu), sy = (int)((d.ext >> 8) & 0xFFu), sz = (int)(d.ext >> 16);
    int q_own[kBlocks3], q_step[kBlocks3];          // box word of the border cell; from it to the halo cell
    uint32_t from_row[kBlocks3];                    // the facing border row in edges
    bool act[kBlocks3];
    float halo[kBlocks3], sent[kBlocks3], ahead[kBlocks3];
#pragma unroll
    for (int i = 0; i < kBlocks3; ++i) {
        const int bi = w + 8 * i;
        const int y = L & 7, z = L >> 3;
        if (bi < 2) {
            q_own[i] = s3_box(bi == 0 ? 1 : kS3X, y + 1, z + 1);
            q_step[i] = bi == 0 ? -1 : 1;
        } else if (bi < 18) {
            const bool hi = bi >= 10;
            q_own[i] = s3_box(L + 1, hi ? kS3Y : 1, ((bi - 2) & 7) + 1);
            q_step[i] = hi ? PX : -PX;
        } else {
            const bool hi = bi >= 26;
            q_own[i] = s3_box(L + 1, ((bi - 18) & 7) + 1, hi ? kS3Z : 1);
            q_step[i] = hi ? PL : -PL;
        }
        if (bi >= 34) { q_own[i] = s3_box(1, 1, 1); q_step[i] = 0; }
        const int s = bi == 0 ? 0 : bi == 1 ? 2 : bi < 10 ? 1 : bi < 18 ? 3 : bi < 26 ? 4 : 5;
        uint32_t nb = kNoTile;
#pragma unroll
        for (int q = 0; q < 6; ++q) nb = s == q ? d.face[q] : nb;
        // the facing row of the opposite side: same place within the side
        const int facing = bi < 2 ? bi ^ 1 : bi < 10 ? bi + 8 : bi < 18 ? bi - 8 : bi < 26 ? bi + 8 : bi - 8;
        const int part = bi < 2 ? 0 : bi < 18 ? (bi - 2) & 7 : (bi - 18) & 7;
        const bool in = bi < 2 ? y < sy && z < sz : bi < 18 ? L < sx && part < sz : L < sx && part < sy;
        act[i] = bi < 34 && nb != kNoTile && in;
        from_row[i] = act[i] ? nb * 34u + (uint32_t)facing : 0u;
        halo[i] = sent[i] = ahead[i] = inf;
    }

    // Cells past the grid read the tile's first cell and become +INF.
    {
        const char* const fb = static_cast<const char*>(d.field);
        float cv[kS3Z];
#pragma unroll
        for (int z = 0; z < kS3Z; ++z) {
            const size_t off = L < sx && w < sy && z < sz ? (size_t)z * d.plane + (size_t)w * d.w + (size_t)L : 0u;
            cv[z] = load_cost_at<KIND>(fb + off * field_bytes<KIND>());
        }
#pragma unroll
        for (int z = 0; z < kS3Z; ++z)
            c_s[s3_box(L + 1, w + 1, z + 1)] = L < sx && w < sy && z < sz ? cv[z] : inf;
    }
    bool seeded = false;
    if (many_sources(a.n_seeds)) {
        seeded = holds_source<kS3X * kS3Y * kS3Z>(a, b) != 0u;
        if (seeded)
#pragma unroll 1
            for (int z = 0; z < kS3Z; ++z)
                if (is_source<kS3X * kS3Y * kS3Z>(a, b, (uint32_t)((z * kS3Y + w) * kS3X + L)))
                    t_s[s3_box(L + 1, w + 1, z + 1)] = 0.0f;
    }
    for (uint32_t i = tid; i < (many_sources(a.n_seeds) ? 0u : a.n_seeds); i += kS3Threads)
        if (a.seeds[4 * i + 3] == b) {
            t_s[s3_box((int)(a.seeds[4 * i] - d.x0) + 1, (int)(a.seeds[4 * i + 1] - d.y0) + 1,
                       (int)(a.seeds[4 * i + 2] - d.z0) + 1)] = 0.0f;
            seeded = true;
        }
    if (tid == 0) s_cmd[0] = await_decision(a.ctl, t_start);
    __syncthreads();
    const bool go = s_cmd[0] != 2u;
    __syncthreads();

    auto cell_improves = [&](int q) -> bool {
        return improves(godunov3(umin_bits(t_s[q - 1], t_s[q + 1]), umin_bits(t_s[q - PX], t_s[q + PX]),
                                 umin_bits(t_s[q - PL], t_s[q + PL]), c_s[q]), t_s[q], eps);
    };
    // Whether one of this wave's border cells would improve, given the whole box.
    auto border_improves = [&]() -> bool {
        bool r = false;
#pragma unroll
        for (int i = 0; i < kBlocks3; ++i)
            if (act[i] && cell_improves(q_own[i])) r = true;
        return r;
    };

    uint32_t st = 1u, acked = 0u, pend = 0u, cmd = 0u, rounds = 0u;
    int ob = 0;
    auto any8 = [&](uint32_t bits) -> uint32_t {
        const uint32_t r = wg_or8(bits, s_or[ob], w, L);
        ob = ob == 2 ? 0 : ob + 1;
        return r;
    };
    auto put_state = [&]() {
        if (tid == 0) st_agent64(&a.state[b], ((unsigned long long)acked << 32) | st);
    };
    auto look = [&]() {
#pragma unroll
        for (int i = 0; i < kBlocks3; ++i)
            if (act[i]) ahead[i] = __uint_as_float(ld_agent(a.edges + (size_t)from_row[i] * 64 + L));
    };
    // Puts what the last look found that is new into the halo.
    auto take = [&]() -> bool {
        bool ch = false;
#pragma unroll
        for (int i = 0; i < kBlocks3; ++i)
            if (__float_as_uint(ahead[i]) < __float_as_uint(halo[i])) {
                halo[i] = ahead[i];
                t_s[q_own[i] + q_step[i]] = ahead[i];
                ch = true;
            }
        return ch;
    };
    uint32_t phase = 0u, epoch = 0u, ver = 0u;      // watcher (work-group 0)
    uint32_t poll = 0;
    bool work = any8(__ballot(seeded) ? 1u : 0u) != 0u;
    while (go) {
        if (work) {
            __builtin_amdgcn_s_setprio(kWorkPriority);
            if (!(st & 1u)) {
                ++st;
                put_state();
            }
            bool more, pub = false, ch = false;
            look();
            auto publish = [&]() {
#pragma unroll
                for (int i = 0; i < kBlocks3; ++i) {
                    const float mine = t_s[q_own[i]];
                    const bool out = act[i] && __float_as_uint(mine) < __float_as_uint(sent[i]) &&
                                     __float_as_uint(mine) < __float_as_uint(halo[i]);
                    if (out) {
                        st_agent(a.edges + ((size_t)d.g * 34u + (uint32_t)(w + 8 * i)) * 64 + L, __float_as_uint(mine));
                        sent[i] = mine;
                    }
                }
            };
            auto exchange = [&]() {
                ch |= take();
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
                look();
            };
            do {
                ch = false;
                switch (w) {
                    case 0: sweep3_round<1, 1, 1, kChunk3, kRound3>(shb, L, exchange); break;
                    case 1: sweep3_round<-1, 1, 1, kChunk3, kRound3>(shb, L, exchange); break;
                    case 2: sweep3_round<1, -1, 1, kChunk3, kRound3>(shb, L, exchange); break;
                    case 3: sweep3_round<-1, -1, 1, kChunk3, kRound3>(shb, L, exchange); break;
                    case 4: sweep3_round<1, 1, -1, kChunk3, kRound3>(shb, L, exchange); break;
                    case 5: sweep3_round<-1, 1, -1, kChunk3, kRound3>(shb, L, exchange); break;
                    case 6: sweep3_round<1, -1, -1, kChunk3, kRound3>(shb, L, exchange); break;
                    default: sweep3_round<-1, -1, -1, kChunk3, kRound3>(shb, L, exchange); break;
                }
                ++rounds;
                const bool stop = (rounds & 1023u) == 0u && must_stop(a.ctl, a.cmd, b, N, t_start);
                uint32_t r = any8((__ballot(ch) ? 1u : 0u) | (__ballot(stop) ? 4u : 0u));
                if (!(r & 1u)) {
                    pub = true;
                    publish();
                    const bool fresh = take();
                    look();
                    bool res = false;
#pragma unroll
                    for (int z = 0; z < kS3Z; ++z) res |= cell_improves(s3_box(L + 1, w + 1, z + 1));
                    r |= any8((__ballot(res) ? 1u : 0u) | (__ballot(fresh) ? 2u : 0u));
                    if ((r & 3u) == 2u) r |= any8(__ballot(border_improves()) ? 1u : 0u);
                    more = (r & 5u) == 1u;
                } else {
                    more = (r & 4u) == 0u;
                }
            } while (more);
            work = false;
            __builtin_amdgcn_s_setprio(0);
        }
        bool idle = false;
        for (;;) {
            ++poll;
            look();
            uint32_t c = 0u;
            if (w == 0) c = ld_agent(&a.cmd[b]);
            uint32_t bits = 0u;
            if (b == 0 && idle) {
                bool busy = false, differs = false, unacked = false;
                if ((uint32_t)tid < N) {
                    const unsigned long long s = ld_agent64(&a.state[tid]);
                    busy = ((uint32_t)s & 1u) != 0u;
                    differs = (uint32_t)s != ver;
                    unacked = (uint32_t)(s >> 32) != epoch;
                    if (phase == 0u) ver = (uint32_t)s;
                }
                bits = (__ballot(busy) ? 4u : 0u) | (__ballot(differs) ? 8u : 0u) | (__ballot(unacked) ? 16u : 0u);
            }
            const bool ch = take();
            if (tid == 0) s_cmd[poll & 1u] = c;
            const uint32_t r = any8(bits | (__ballot(ch) ? 2u : 0u));
            cmd = s_cmd[poll & 1u];
            if (cmd == kCmdDone || cmd == kCmdAbort) break;
            if (r & 2u) {
                if (any8(__ballot(border_improves()) ? 1u : 0u)) {
                    work = true;
                    break;
                }
                continue;
            }
            if (!idle) {
                idle = true;
                if (st & 1u) {
                    wait_stores();
                    __syncthreads();
                    if (tid == 0) s_pub = 0u;
                    ++st;
                    put_state();
                }
                phase = 0u;
                continue;
            }
            if (cmd != acked) {
                if (cmd == pend) {
                    acked = cmd;
                    put_state();
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
                if (send && (uint32_t)tid < N) st_agent(&a.cmd[tid], send);
            }
            __builtin_amdgcn_s_sleep(2);
        }
        if (!work) break;
    }
    uint32_t reached = 0u;
    if (go) {
#pragma unroll
        for (int z = 0; z < kS3Z; ++z) {
            if (L < sx && w < sy && z < sz) {
                const float t = t_s[s3_box(L + 1, w + 1, z + 1)];
                gmem(d.time)[(size_t)z * d.plane + (size_t)w * d.w + (size_t)L] = t;
                reached += __float_as_uint(t) < kInfBits ? 1u : 0u;
            }
        }
    }
    // ---- leave: the last work-group out reports the solve ----
    reached = wave_sum(reached);
    __syncthreads();
    if (L == 0) s_or[0][w] = reached;
    __syncthreads();
    if (tid == 0) {
        uint32_t n = 0;
        for (int i = 0; i < 8; ++i) n += s_or[0][i];
        st_agent64(&a.report[b], ((unsigned long long)n << 32) | rounds);
        wait_stores();
        s_cmd[0] = last_in(a.ctl, kResLeft, b, N) ? 1u : 0u;
    }
    __syncthreads();
    if (s_cmd[0] == 0u) return;
    unsigned long long* const red = reinterpret_cast<unsigned long long*>(sh);
    const unsigned long long v = (uint32_t)tid < N ? ld_agent64(&a.report[tid]) : 0ull;
    red[tid] = v;
    __syncthreads();
    if (tid == 0) {
        unsigned long long sum = 0, cells = 0;
        uint32_t most = 0;
        for (uint32_t i = 0; i < N; ++i) {
            sum += (uint32_t)red[i];
            cells += red[i] >> 32;
            most = max(most, (uint32_t)red[i]);
        }
        report_totals(a, sum, sum, cells, most, !go || ld_agent(&a.ctl[kResFailed]) != 0u);
    }
}

// The state of a 3-D resident solve in one launch (see k_resident_init).
template <int FB>
__global__ void k_resident3_init(Resident3Args a, const GhcmInst* h_inst, const uint32_t* h_seeds) {
    const size_t i0 = (size_t)blockIdx.x * blockDim.x + threadIdx.x, stride = (size_t)gridDim.x * blockDim.x;
    const uint4 inf4 = make_uint4(kInfBits, kInfBits, kInfBits, kInfBits);
    uint4* const e4 = reinterpret_cast<uint4*>(a.edges);
    for (size_t i = i0; i < (size_t)a.tiles * (kRes3Words / 4); i += stride) e4[i] = inf4;
    for (size_t i = i0; i < kRes3MaxGroups; i += stride) {
        a.state[i] = 1ull;
        a.cmd[i] = 0u;
    }
    for (size_t i = i0; i < kResCtlWords; i += stride) a.ctl[i] = 0u;
    const GhcmInst in = h_inst[0];
    const uint32_t nx = in.tiles_x, ny = in.tiles_y, nz = in.tiles_z;
    if (many_sources(a.n_seeds)) clear_sources<kS3X * kS3Y * kS3Z>(a, i0, stride);
    for (size_t i = i0; i < (many_sources(a.n_seeds) ? 0u : a.n_seeds); i += stride) {
        const uint32_t x = h_seeds[4 * i], y = h_seeds[4 * i + 1], z = h_seeds[4 * i + 2];
        a.seeds[4 * i] = x;
        a.seeds[4 * i + 1] = y;
        a.seeds[4 * i + 2] = z;
        a.seeds[4 * i + 3] = rank3(nx, ny, x / kS3X, y / kS3Y, z / kS3Z);
    }
    for (size_t t = i0; t < a.tiles; t += stride) {
        const uint32_t tx = (uint32_t)t % nx, ty = (uint32_t)t / nx % ny, tz = (uint32_t)t / (nx * ny);
        ResTile3 d;
        d.g = (uint32_t)t;
        d.w = in.w;
        d.plane = (uint64_t)in.w * in.h;
        d.x0 = tx * kS3X;
        d.y0 = ty * kS3Y;
        d.z0 = tz * kS3Z;
        const size_t org = (size_t)d.z0 * d.plane + (size_t)d.y0 * in.w + d.x0;
        d.field = static_cast<const char*>(in.field) + org * FB;
        d.time = in.time + org;
        d.ext = min(in.w - d.x0, (uint32_t)kS3X) | min(in.h - d.y0, (uint32_t)kS3Y) << 8 | min(in.d - d.z0, (uint32_t)kS3Z) << 16;
        for (int s = 0; s < 6; ++s) {
            const int qx = (int)tx + (s == 0 ? -1 : s == 2 ? 1 : 0), qy = (int)ty + (s == 1 ? -1 : s == 3 ? 1 : 0);
            const int qz = (int)tz + (s == 4 ? -1 : s == 5 ? 1 : 0);
            const bool ok = qx >= 0 && qy >= 0 && qz >= 0 && qx < (int)nx && qy < (int)ny && qz < (int)nz;
            d.face[s] = ok ? (uint32_t)qx + nx * ((uint32_t)qy + ny * (uint32_t)qz) : kNoTile;
        }
        a.rtile[rank3(nx, ny, tx, ty, tz)] = d;
    }
}

// With many sources: each one's cell marked in its tile's bits (see k_resident_sources).
__global__ void k_resident3_sources(Resident3Args a, const GhcmInst* h_inst, const uint32_t* h_seeds) {
    const uint32_t nx = h_inst->tiles_x, ny = h_inst->tiles_y;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < a.n_seeds; i += (size_t)gridDim.x * blockDim.x) {
        const uint32_t x = h_seeds[4 * i], y = h_seeds[4 * i + 1], z = h_seeds[4 * i + 2];
        mark_source<kS3X * kS3Y * kS3Z>(a, rank3(nx, ny, x / kS3X, y / kS3Y, z / kS3Z),
                                        (z % kS3Z * kS3Y + y % kS3Y) * kS3X + x % kS3X);
    }
}

template <int KIND>
static hipError_t launch_resident3_t(const Resident3Args& a, hipStream_t s, hipEvent_t ev0, hipEvent_t ev1) {
    if (a.tiles == 0 || a.tiles > kRes3MaxGroups) return hipErrorInvalidValue;
    if (ev0 && ev1)
        hipExtLaunchKernelGGL((k_resident_sweep3<KIND>), dim3(a.tiles), dim3(kS3Threads), 0, s, ev0, ev1, 0, a);
    else
        hipLaunchKernelGGL((k_resident_sweep3<KIND>), dim3(a.tiles), dim3(kS3Threads), 0, s, a);
    return hipGetLastError();
}

template <int KIND>
static hipError_t launch_resident3_init_t(const Resident3Args& a, const GhcmInst* h_inst, const uint32_t* h_seeds, hipStream_t s) {
    hipLaunchKernelGGL((k_resident3_init<(int)field_bytes<KIND>()>), dim3(a.tiles), dim3(256), 0, s, a, h_inst, h_seeds);
    if (many_sources(a.n_seeds))
        hipLaunchKernelGGL(k_resident3_sources, sources_grid(a.n_seeds), dim3(256), 0, s, a, h_inst, h_seeds);
    return hipGetLastError();
}

template <int KIND>
static int occ_resident3_t() {
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k_resident_sweep3<KIND>, kS3Threads, 0) != hipSuccess) return 0;
    return nb;
}

Resident3Kernel get_resident3_kernel(int kind) {
    switch (kind) {
        case 0: return {&launch_resident3_t<0>, &launch_resident3_init_t<0>, &occ_resident3_t<0>};
        case 1: return {&launch_resident3_t<1>, &launch_resident3_init_t<1>, &occ_resident3_t<1>};
        case 2: return {&launch_resident3_t<2>, &launch_resident3_init_t<2>, &occ_resident3_t<2>};
        case 3: return {&launch_resident3_t<3>, &launch_resident3_init_t<3>, &occ_resident3_t<3>};
    }
    return {nullptr, nullptr, nullptr};
}

}  // namespace ghcm
