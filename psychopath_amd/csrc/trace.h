// Launch interface of the traversal kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/psy_rt.h"
#include "layout.h"

namespace psy {

constexpr int TRACE_BLOCK = 128;           // lanes per workgroup (two wave64s)
constexpr int TRACE_LDS_DEPTH = 24;        // stack entries per lane held in LDS
// Total stack entries per lane: the bound 3 * (instance-BVH depth + mesh-BVH
// depth) + 2 for two BVH4s of the deepest the builder makes (depth 22, from
// a binary depth of at most 42: src/accel/bvh_base.rs:7, bvh4.rs:87).
constexpr int TRACE_STACK_CAPACITY = 3 * (22 + 22) + 2;

// The persistent kernels take their rays from TRACE_RANGES counters, one per
// XCD's worth of waves and TRACE_RANGE_WORDS words apart (a cache line each).
constexpr uint32_t TRACE_RANGES = 8;
constexpr uint32_t TRACE_RANGE_WORDS = 32;
constexpr uint32_t TRACE_WORK_WORDS = TRACE_RANGES * TRACE_RANGE_WORDS;

struct TraceArgs {
    // scene
    const GpuNode* nodes;
    const GpuBox4* motion;
    const uint8_t* tris;
    const GpuMesh* meshes;
    const GpuInstance* instances;
    const GpuXform* xforms;
    const GpuXform* inv_static;
    const GpuRectLight* rect_lights;
    const GpuSphereLight* sphere_lights;
    const float* light_samples;  // time samples of the lights (layout.h)
    const uint8_t* order_table;  // visit order of node slots per [octant][code], 8 x 48 bytes
    const GpuGroup* groups;      // nested scenes: instance paths (layout.h), else NULL
    uint32_t top_root;
    uint32_t wide;               // node addresses need 64-bit offsets
    uint32_t odd_boxes;          // some node's box needs the full test (PackedScene)
    // rays (device)
    const float *ox, *oy, *oz, *dx, *dy, *dz, *time, *max_t;
    const uint8_t* flags;
    uint32_t all_occlusion;    // every ray is an occlusion ray (flags ignored)
    uint64_t n;                // ray count, or the capacity when n_dev is set
    const uint32_t* n_dev;     // device-resident ray count (persistent kernel), or NULL
    // Persistent kernels: occlusion rays traced in the same launch after the
    // n rays above (counted by n2_dev; NULL: none), at index n2_at of the
    // same ray arrays.  Ray i's result is the kind byte n2_kind[n2_out[i]].
    const uint32_t* n2_dev;
    uint32_t n2_at;
    const uint32_t* n2_out;
    uint8_t* n2_kind;
    // Persistent kernels, for a caller that launches one after another: the
    // first block zeroes clear0[0], clear1[0] and clear_run[0, clear_run_n)
    // where not NULL, adds the rays to *tally, and when `work_next` is set
    // zeroes those counters, which the next launch then takes without a
    // reset of its own (so must this launch's `work` be clear).
    uint32_t *clear0, *clear1, *clear_run;
    uint32_t clear_run_n;
    unsigned long long* tally;
    unsigned int* work_next;
    // hits (device): 32-byte records when `rec` is set, else structure of
    // arrays
    uint4* rec;
    uint8_t* kind;
    float *t, *b0, *b1, *b2;
    uint32_t *prim_id, *inst_id;
    // counters (device, 5 x u64) for the instrumented kernel
    unsigned long long* counters;
};

// Launch shape of the persistent kernel (chosen per scene by the autotuner).
struct TraceTuning {
    uint32_t cus;          // compute units of the device
    uint32_t waves_per_cu; // wave64 workgroups launched per CU, at most as many as it holds
    uint32_t refill_min;  // idle lanes that trigger a refill (1..64)
    uint32_t lds_depth;   // stack entries per lane kept in LDS (8, 16, or 24 for 32)
    uint32_t occupancy;   // register budget: 4 at most 128 VGPRs, 8 the compiler's choice
    uint32_t leaf_min;    // waiting lanes that end a descent round (1..64), 0: per-lane descents
    uint32_t coop;        // 1: wave-cooperative node fetch (static scenes)
};

// One lane per ray, one launch-wide grid (trace.hip).
hipError_t launch_trace(const TraceArgs& args, bool counted, hipStream_t stream);

// Persistent waves with lane refill (trace_persistent.hip).  `work`:
// TRACE_WORK_WORDS device words, the ray counters, which the launch resets.
hipError_t launch_trace_persistent(const TraceArgs& args, bool counted, bool has_xf, bool has_motion,
                                   unsigned int* work, const TraceTuning& tune, hipStream_t stream);

}  // namespace psy
