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
    kResFailed = 1,      // 1: given up (declined, or out of time); the wave loop takes over
    kResArrived = kCounterStride,                                   // work-groups running
    kResLeft = kResArrived + (1 + kResSpread) * kCounterStride,     // work-groups done
    kResCtlWords = kResLeft + (1 + kResSpread) * kCounterStride
};

constexpr uint32_t kResMaxGroups = 1024;     // work-groups whose states one of them watches
constexpr uint32_t kResMaxOwned = 32;        // tiles of one work-group

struct ResidentArgs {
    const GhcmInst* inst;
    uint32_t        n_inst;
    const uint32_t* tinst;   // instance of each tile (null with one instance)
    const uint32_t* seeds;   // [n_seeds] (x, y, instance)
    uint32_t        n_seeds;
    uint32_t        tiles;
    float           eps;
    uint32_t*       edges;   // [tiles][4][64] published border cells (float bits), side-major
    uint32_t*       seen;    // [tiles][4][64] the neighbours' facing borders a closed tile was left with
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
// h_inst, h_seeds: device views of the mapped host instance table and source list.
hipError_t launch_resident_init(const ResidentArgs& a, const GhcmInst* h_inst, const uint32_t* h_seeds,
                                hipStream_t s);

}  // namespace ghcm
