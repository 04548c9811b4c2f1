// resident.h -- host-side entry points of resident.hip: the 2-D solve with every tile resident
// in the LDS of its own work-group for the whole solve.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "ghcm_dev.h"

namespace ghcm {

// Words of ResidentArgs::ctl.
constexpr uint32_t kResSpread = 32;          // arrival counters beside the top one
enum : uint32_t {
    kResDecision = 0,    // 0: undecided, 1: every work-group is running, 2: not all came in time
    kResFailed = 1,      // 1: given up for want of time; the wave loop takes over
    kResArrived = kCounterStride,                                   // work-groups running
    kResLeft = kResArrived + (1 + kResSpread) * kCounterStride,     // work-groups done
    kResCtlWords = kResLeft + (1 + kResSpread) * kCounterStride
};

constexpr uint32_t kResMaxGroups = 1024;     // work-groups whose states one of them watches
constexpr uint32_t kResMaxScan = 16;         // tiles of one work-group that scans their borders,
constexpr uint32_t kResAlwaysScan = 6;       // with this many sources or more, tiles up to which it does
constexpr uint32_t kResScanSources = 64;
constexpr uint32_t kResMaxOwned = 256;       // tiles of one work-group (one want a thread)
// Up to this many sources every tile reads their list; with more it reads the marks of its own cells.
constexpr uint32_t kResFewSources = 1024;
__host__ __device__ constexpr bool many_sources(uint64_t n) { return n > kResFewSources; }
// Bytes of the sources' part of the workspace, `cells` to a tile.
constexpr size_t source_bytes(uint64_t n, uint64_t tiles, uint32_t cells) {
    return many_sources(n) ? (size_t)(tiles * (cells / 8u + 4u)) : (size_t)(16u * n);
}

// What a work-group needs to open a tile: one read.
struct alignas(16) ResTile {
    const void* field;       // its first cell in the field and in the times
    float*      time;
    uint32_t    w;           // cells per row of the grid
    uint32_t    ext;         // its columns | rows << 8
    uint32_t    g;           // its id
    uint32_t    inst;
    uint32_t    face[4];     // across side s: id * 4 + side of the border facing it, or kNoTile
    uint32_t    call[4];     // and where in `want` its owner is told
    uint32_t    x0, y0;      // its origin
    float       pace;        // 1 / (tiles across and down its grid): times by it are compared in `want`
    uint32_t    pad;
};

struct ResidentArgs {
    uint32_t        n_inst;
    ResTile*        rtile;   // [tiles] by rank (the order in which tiles are dealt out)
    uint32_t*       seeds;   // few sources: [n_seeds] (x, y, instance, rank of its tile)
                             // many: [tiles] by rank, a bit a cell, row by row, set where it is a source;
                             // then [tiles] by rank, 1: holds a source
    uint32_t        n_seeds;
    uint32_t        tiles;
    float           eps;
    uint32_t*       edges;   // [tiles][4][64] published border cells (float bits), side-major
    // With several tiles to a work-group, one of (the other null):
    uint32_t*       seen;    // [tiles][4][64] the neighbours' facing borders a closed tile was left with
    uint32_t*       want;    // [groups][want_stride] smallest new border value of an owned tile's neighbours, by pace
    uint32_t        want_stride;
    unsigned long long* state;  // [groups] (acknowledged epoch << 32) | visit counter, odd while busy
    uint32_t*       cmd;     // [groups] epoch to acknowledge, or kCmdDone / kCmdAbort
    uint32_t*       ctl;     // kResCtlWords
    unsigned long long* report; // [groups] (cells written << 32) | rounds
    HostRec*        rec;     // totals, busy_waves (most rounds of a work-group), wave (1: given up), tag
    uint32_t        tag;
};

struct ResidentKernel {
    hipError_t (*launch)(const ResidentArgs&, uint32_t groups, hipStream_t, hipEvent_t ev0, hipEvent_t ev1);
    int (*blocks_per_cu)();
};
// Null launch where no resident form is built (64 x 64 sweep tiles only).
ResidentKernel get_resident_kernel(int tile_w, int tile_h, int kind, int mode);
// h_inst, h_seeds: device views of the mapped host instance table and source list; d_inst: n_inst
// records of device memory (written with many sources only).
hipError_t launch_resident_init(const ResidentArgs& a, const GhcmInst* h_inst, GhcmInst* d_inst,
                                const uint32_t* h_seeds, uint32_t groups, int kind, hipStream_t s);

// The one-wave tiles (8x8, 16x16, 32x8, 32x32): one wave64 per tile, the tile in its registers.
// Here `edges` holds the tiles' inboxes (`inbox_words` each: the cells across each border, written
// by the neighbours), and state, cmd and report are per tile.
constexpr uint32_t kResMaxWaveTiles = 8192;
struct ResidentWaveKernel {
    hipError_t (*launch)(const ResidentArgs&, uint32_t groups, hipStream_t, hipEvent_t ev0, hipEvent_t ev1);
    hipError_t (*init)(const ResidentArgs&, const GhcmInst* h_inst, GhcmInst* d_inst, const uint32_t* h_seeds, int kind,
                       hipStream_t);
    int (*blocks_per_cu)();
    uint32_t inbox_words;
};
// mode: 0 systolic, 1 FIM.
ResidentWaveKernel get_resident_wave_kernel(int tile_w, int tile_h, int kind, int mode);

// 3-D sweep tiles (64 x 8 x 8), one work-group per tile.  `edges` holds kRes3Words a tile (34 rows of
// 64 border cells), `seeds` (x, y, z, rank of its tile).
constexpr uint32_t kRes3Words = 34 * 64;
struct alignas(16) ResTile3 {
    const void* field;       // its first cell in the field and in the times
    float*      time;
    uint64_t    plane;       // cells per plane of the grid
    uint32_t    w;           // cells per row
    uint32_t    ext;         // its columns | rows << 8 | planes << 16
    uint32_t    g;           // its id
    uint32_t    x0, y0, z0;
    uint32_t    face[6];     // the tile across side s (0 x-, 1 y-, 2 x+, 3 y+, 4 z-, 5 z+), or kNoTile
    uint32_t    pad[2];
};
struct Resident3Args {
    ResTile3*       rtile;   // [tiles] by rank
    uint32_t*       seeds;   // as in ResidentArgs, the cells plane by plane
    uint32_t        n_seeds, tiles;
    float           eps;
    uint32_t*       edges;
    unsigned long long* state;
    uint32_t*       cmd;
    uint32_t*       ctl;
    unsigned long long* report;
    HostRec*        rec;
    uint32_t        tag;
};
constexpr uint32_t kRes3MaxGroups = 512;
struct Resident3Kernel {
    hipError_t (*launch)(const Resident3Args&, hipStream_t, hipEvent_t ev0, hipEvent_t ev1);
    hipError_t (*init)(const Resident3Args&, const GhcmInst* h_inst, const uint32_t* h_seeds, hipStream_t);
    int (*blocks_per_cu)();
};
Resident3Kernel get_resident3_kernel(int kind);

}  // namespace ghcm
