// kernels.h -- host-side launchers of the render, query and post-process kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "rtx.h"
#include "rtx_internal.h"

namespace rtx {

constexpr int kRenderBlock = 256;
constexpr int kTraceBlock = 256;

constexpr uint32_t kShadeBatch = 40;   // default shading batch

// per-context scratch for the persistent kernels
struct LaunchScratch {
    uint32_t* counter = nullptr;   // work counter and the ordered frames' narrow waves (device, 4 words)
    uint32_t* gstack = nullptr;    // traversal stack overflow (device)
    uint32_t gstride = 0;          // lanes covered by gstack (grid * block)
    uint32_t grid = 0;             // persistent grid size in blocks
    uint32_t shade_batch = kShadeBatch;   // render: finished lanes that trigger a wave's shading step
    uint32_t shade_auto = 1;       // 1: nobody chose shade_batch, and whole frames and batches take a larger one
    uint32_t inner_frac = 36;      // traversal: node phase ends below inner_frac/64 of the going lanes
    uint32_t tile_w = 8;           // render: work tile of tile_w x (64 / tile_w) pixels
    uint32_t stack_lds = kStackLDS;   // render: traversal stack entries per lane in LDS (16 or 32)
    uint32_t grid_max = 0;         // blocks the overflow stack area was sized for
    uint32_t gstack_entries = 0;   // overflow entries per lane (beyond the smallest LDS part)
    uint16_t* pix_cost = nullptr;    // render: cost of each work slot's pixel in the one-sample probe (device)
    uint32_t* tile_cost = nullptr;   // render: cost of each tile from them (device)
    uint32_t* tile_order = nullptr;  // render: the tiles in descending probe cost (device)
    uint32_t tile_cap = 0;           // tiles the three arrays hold
    uint32_t iterative = 0;          // render: 1 = the iterative programs' semantics, 0 = the recursive ones
};

// Plain frames of at least kOrderMinSpp samples per pixel and at least
// kOrderMinPixelsPerLane pixels per lane of the persistent grid render their
// tiles longest first: a one-sample probe launch counts the node visits and
// rays of each pixel, a tile's cost is the largest sum of a neighbourhood in
// it, and the frame takes its tiles in descending order of that (stable, so
// equal costs keep their order).  A lane renders whole pixels, so at the end
// of a frame a wave waits for its most expensive last pixel; longest first
// makes the last pixels cheap ones, and the most expensive pixels get waves
// of fewer lanes.  A smaller frame is spread instead (from 1.4 to 2 pixels per
// lane, ordered against spread: level 4 1.00 to 1.17x, level 6 0.86x, mixed
// levels 0.79 to 0.90x).  The adjoint, of whose blocks three of four are
// resident at once, orders frames from 2 pixels per 5 lanes on (640x360:
// 1.06x, 480x270: 1.07x, 900x500: 1.07x; 320x180: 0.96x, 200x120: 0.90x).
// No pixel depends on the order.
// The probe is one sample more: ordered against not, 1080p and 720p frames of
// levels 4 and 6 and of mixed levels, 5 samples 0.89 to 1.01x, 8 samples 0.97
// to 1.08x, 11 samples 1.02 to 1.13x, 14 samples 1.04 to 1.17x.  The adjoint's
// frames are smaller and stay at 16.
constexpr uint32_t kOrderMinSpp = 10;
constexpr uint32_t kOrderMinSppAdjoint = 16;
constexpr uint32_t kOrderMinPixelsPerLane = 2;
inline bool frame_ordered(const rtx_lp_general& lp, const LaunchScratch& ls, bool adjoint = false) {
    const uint64_t px = (uint64_t)lp.image_w * lp.image_h;
    return adjoint ? lp.spp >= kOrderMinSppAdjoint && 5 * px >= 2 * (uint64_t)ls.gstride
                   : lp.spp >= kOrderMinSpp && px >= (uint64_t)kOrderMinPixelsPerLane * ls.gstride;
}
// tiles of a frame (64 work slots each) for a tile width
inline uint32_t frame_tiles(const rtx_lp_general& lp, uint32_t tile_w) {
    const uint32_t th = 64u / tile_w;
    return ((lp.image_w + tile_w - 1u) / tile_w) * ((lp.image_h + th - 1u) / th);
}

// One frame of a launch: scene, launch parameters and its slice of the
// global work index space (64 slots per tile).
struct Job {
    DevScene sc;
    rtx_lp_general lp;
    float3 ambient;
    uint32_t tiles_x, tiles_y;
    uint32_t work_begin, work_end;
};

Job make_job(const DevScene& sc, const rtx_lp_general& lp, float3 ambient, uint32_t tile_w, uint32_t work_begin);

// Optional per-pixel traversal statistics (node visits, triangle tests).
struct TraceCounters {
    uint64_t* nodes = nullptr;
    uint64_t* tris = nullptr;
    uint64_t* wave_cycles = nullptr;   // [0] cycles in traversal, [1] cycles in the whole loop (sum over waves)
};

hipError_t launch_render(const DevScene& sc, const rtx_lp_general& lp, float3 ambient, const LaunchScratch& ls,
                         hipStream_t s);
hipError_t launch_render_counted(const DevScene& sc, const rtx_lp_general& lp, float3 ambient,
                                 const LaunchScratch& ls, const TraceCounters& tc, hipStream_t s);
// all jobs of a batch in one persistent launch (d_jobs sorted by work_begin)
hipError_t launch_render_batch(const Job* d_jobs, const Job& first, uint32_t njobs, uint32_t nwork,
                               const LaunchScratch& ls, uint32_t tile_w, hipStream_t s);
// adjoint of a frame: dparams (float4 per instance: d albedo rgb, d fuzz) =
// dL/d params given dL/d rawRGB (lp.rawRGB holds the forward image); tape:
// depth x kAdjointTapeWords words per lane (one record per shaded hit: at
// most depth - 1 recursive, depth iterative), lane stride tape_stride
constexpr uint32_t kAdjointTapeWords = 14;
constexpr uint32_t kAdjointLdsInsts = 2048;   // instances whose gradients a block sums in LDS first
hipError_t launch_adjoint(const DevScene& sc, const rtx_lp_general& lp, float3 ambient, const LaunchScratch& ls,
                          const rtx_float3* dldi, float* dparams, uint32_t* tape, uint32_t tape_stride, hipStream_t s);
hipError_t launch_set_materials(const DevScene& sc, const float* params, hipStream_t s);
hipError_t launch_get_materials(const DevScene& sc, float* params, hipStream_t s);
hipError_t launch_pick(const DevScene& sc, const rtx_lp_general& lp, const LaunchScratch& ls, hipStream_t s);
hipError_t launch_trace(const DevScene& sc, const rtx_ray* rays, uint32_t n, rtx_hit* hits,
                        const LaunchScratch& ls, hipStream_t s);
hipError_t launch_rng(const uint32_t* seeds, uint32_t n, uint32_t k, float* out, hipStream_t s);
hipError_t launch_pp(const rtx_float3* src, rtx_uchar4* dst, int w, int h, bool srgb, hipStream_t s);

// occupancy-derived persistent grid (blocks) for the render / trace kernels
uint32_t render_blocks_per_cu();
uint32_t trace_blocks_per_cu();

}  // namespace rtx
