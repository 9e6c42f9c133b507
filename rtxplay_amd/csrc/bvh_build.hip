// bvh_build.hip -- on-device acceleration structure build.
//
// Replaces the OptiX GAS/IAS builds of optx/scene.cxx:38-273 (optixAccelBuild)
// with: instance flattening to world space, a top-down binned SAH BVH built
// level by level on the device (Wald 2007, "On fast construction of SAH-based
// bounding volume hierarchies"), triangle reordering into leaf order, and a
// collapse into the 128-byte 4-wide node layout the traversal reads.  The
// same builder makes the levels of a two-level scene: one tree per mesh over
// its object-space triangles and one over the instances' world boxes (one
// instance per leaf); tlas.hip assembles and refits them.
//
// Determinism: every level is processed in task order, child nodes and tasks
// are placed by an exclusive scan (no atomics decide positions) and the
// partition is stable, so the same input always gives the same BVH.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <mutex>
#include <string>
#include <vector>

#include "bvh_build.h"
#include "node.h"

namespace rtx {

namespace {

#ifndef RTX_SAH_BINS
#define RTX_SAH_BINS 64
#endif
constexpr int kBins = RTX_SAH_BINS;
constexpr int kBuildBlock = 256;
constexpr uint32_t kSmallTask = 256;   // primitives per task below which a level runs a wave per task
constexpr uint32_t kWideTasks = 512;      // levels of at most this many tasks, averaging ...
constexpr uint32_t kWideMinPrims = 8192;  // ... at least this many primitives, spread each task
constexpr uint32_t kWideBlocks = 1024;    // over kWideBlocks / tasks chunks, ...
constexpr uint32_t kWideMinChunk = 2048;  // ... of this many primitives at least (on average)
constexpr uint32_t kRootBlocks = 2048;                   // blocks of the root bounds reduction at most
constexpr int kScanBlock = 1024;
// SAH constants (cost of one node visit vs one triangle test)
// 1: the 4-wide tree is the SAH-optimal grouping of the binary one; 0: each
// wide node opens its largest-area inner child until it has 4 children
#ifndef RTX_DP_COLLAPSE
#define RTX_DP_COLLAPSE 1
#endif
#ifndef RTX_SAH_TRAV
#define RTX_SAH_TRAV 1.0f
#endif
constexpr float kCostTrav = RTX_SAH_TRAV;
constexpr float kCostIsect = 1.0f;
constexpr float kFarAway = 1e38f;   // coordinate of the degenerate triangle

struct BuildTask {
    uint32_t node, begin, end, depth;
    float4 clo, chi;   // centroid bounds of the task's primitives
};

struct SplitOut {
    uint32_t kind;     // 0 leaf, 1 split
    uint32_t nleft;
    uint32_t pad0, pad1;
    float4 clo_l, chi_l, clo_r, chi_r;
};

// binary node during the build: lo.w/hi.w carry the links as uint bits
//   inner: lo.w = left child (right = left + 1), hi.w = 0
//   leaf : lo.w = first leaf-ordered primitive, hi.w = count (>= 1)
struct BNode {
    float4 lo, hi;
};

struct BuildStats {
    uint32_t max_leaf, pad;
    double sah;
};

// One level of the binary tree (tasks) or of the 4-wide tree (nodes): how many
// and the index of the first.  The counts stay on the device: the kernels of a
// level read theirs, and a level's scan writes the next one's (and its count
// to the host, which runs a level ahead with grids for the most there can be).
struct Level {
    uint32_t n, first;
};
constexpr uint32_t kMaxLevels = 128;   // levels held at once (a deeper tree wraps round)

__device__ __forceinline__ uint32_t f2o(float f) {
    uint32_t u = __float_as_uint(f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float o2f(uint32_t u) {
    return __uint_as_float((u & 0x80000000u) ? (u & 0x7FFFFFFFu) : ~u);
}

__device__ __forceinline__ float area3(float lx, float ly, float lz, float hx, float hy, float hz) {
    const float dx = hx - lx, dy = hy - ly, dz = hz - lz;
    if (!(dx >= 0.f) || !(dy >= 0.f) || !(dz >= 0.f)) return 0.f;
    return 2.f * (dx * dy + dy * dz + dz * dx);
}

__device__ __forceinline__ float comp4(const float4& v, int k) { return k == 0 ? v.x : (k == 1 ? v.y : v.z); }

__device__ __forceinline__ int bin_of(float c, float lo, float scale) {
    int b = (int)((c - lo) * scale);
    return b < 0 ? 0 : (b >= kBins ? kBins - 1 : b);
}

// ---------------------------------------------------------------------------
// flatten: one thread per world-space triangle (instance-major order)
// world = R v + t evaluated as ((v.x*t0 + v.y*t1) + v.z*t2) + t3, one
// rounding per operation (optx/optics_r.cu:61-75 with contraction ruled out)
// ---------------------------------------------------------------------------
__global__ void k_flatten(const InstBuild* __restrict__ insts, uint32_t ninst,
                          const MeshRef* __restrict__ meshes, uint32_t N,
                          float4* __restrict__ tri_world, float4* __restrict__ plo,
                          float4* __restrict__ phi) {
    const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= N) return;
    uint32_t lo = 0, hi = ninst - 1;
    while (lo < hi) {
        const uint32_t mid = (lo + hi + 1) >> 1;
        if (insts[mid].tri_base <= p) lo = mid; else hi = mid - 1;
    }
    const InstBuild& in = insts[lo];
    const uint32_t j = p - in.tri_base;
    const MeshRef m = meshes[in.mesh];
    float3 w[3];
    for (int c = 0; c < 3; c++) {
        const uint32_t vi = m.ices[3 * j + c];
        const float vx = m.vces[3 * vi + 0], vy = m.vces[3 * vi + 1], vz = m.vces[3 * vi + 2];
        float r[3];
        for (int k = 0; k < 3; k++) {
            float acc = __fmul_rn(vx, in.xf[4 * k + 0]);
            acc = __fadd_rn(acc, __fmul_rn(vy, in.xf[4 * k + 1]));
            acc = __fadd_rn(acc, __fmul_rn(vz, in.xf[4 * k + 2]));
            r[k] = __fadd_rn(acc, in.xf[4 * k + 3]);
        }
        w[c] = make_float3(r[0], r[1], r[2]);
    }
    tri_world[3 * (size_t)p + 0] = make_float4(w[0].x, w[0].y, w[0].z, __uint_as_float(p));
    tri_world[3 * (size_t)p + 1] = make_float4(w[1].x, w[1].y, w[1].z, __uint_as_float(lo));
    tri_world[3 * (size_t)p + 2] = make_float4(w[2].x, w[2].y, w[2].z, __uint_as_float(j));
    plo[p] = make_float4(fminf(fminf(w[0].x, w[1].x), w[2].x), fminf(fminf(w[0].y, w[1].y), w[2].y),
                         fminf(fminf(w[0].z, w[1].z), w[2].z), 0.f);
    phi[p] = make_float4(fmaxf(fmaxf(w[0].x, w[1].x), w[2].x), fmaxf(fmaxf(w[0].y, w[1].y), w[2].y),
                         fmaxf(fmaxf(w[0].z, w[1].z), w[2].z), 0.f);
}

// root task: centroid bounds of all primitives as ordered ints (minima of x,
// y, z, then maxima), reduced per block and merged across blocks by atomics;
// min and max are exact, so the result does not depend on their order
__global__ void k_root_init(uint32_t* __restrict__ rb, BuildStats* __restrict__ st, Level* __restrict__ lev,
                            Level* __restrict__ wlev) {
    if (threadIdx.x < 6) rb[threadIdx.x] = threadIdx.x < 3 ? 0xFFFFFFFFu : 0u;
    if (threadIdx.x == 0) {
        st->max_leaf = 0u;
        st->sah = 0.0;
        lev->n = wlev->n = 1u;
        lev->first = wlev->first = 0u;
    }
}
__global__ __launch_bounds__(256) void k_root_bounds(const float4* __restrict__ plo, const float4* __restrict__ phi,
                                                     uint32_t N, uint32_t* __restrict__ rb) {
    __shared__ uint32_t s_b[6];
    if (threadIdx.x < 6) s_b[threadIdx.x] = threadIdx.x < 3 ? 0xFFFFFFFFu : 0u;
    __syncthreads();
    uint32_t lo[3] = {0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu}, hi[3] = {0u, 0u, 0u};
    for (uint32_t p = blockIdx.x * blockDim.x + threadIdx.x; p < N; p += gridDim.x * blockDim.x) {
        const float4 a = plo[p], b = phi[p];
        const float c[3] = {.5f * (a.x + b.x), .5f * (a.y + b.y), .5f * (a.z + b.z)};
        for (int k = 0; k < 3; k++) {
            lo[k] = min(lo[k], f2o(c[k]));
            hi[k] = max(hi[k], f2o(c[k]));
        }
    }
    for (int k = 0; k < 3; k++) { atomicMin(&s_b[k], lo[k]); atomicMax(&s_b[3 + k], hi[k]); }
    __syncthreads();
    if (threadIdx.x < 3) atomicMin(&rb[threadIdx.x], s_b[threadIdx.x]);
    else if (threadIdx.x < 6) atomicMax(&rb[threadIdx.x], s_b[threadIdx.x]);
}
__global__ void k_root_task(const uint32_t* __restrict__ rb, uint32_t N, BuildTask* __restrict__ task) {
    if (threadIdx.x != 0) return;
    BuildTask t;
    t.node = 0; t.begin = 0; t.end = N; t.depth = 0;
    t.clo = make_float4(o2f(rb[0]), o2f(rb[1]), o2f(rb[2]), 0.f);
    t.chi = make_float4(o2f(rb[3]), o2f(rb[4]), o2f(rb[5]), 0.f);
    *task = t;
}

// lev[0] takes lev[kMaxLevels]'s place: levels kMaxLevels and up use the array again
__global__ void k_level_wrap(Level* lev) { lev[0] = lev[kMaxLevels]; }

__global__ void k_zero_word(uint32_t* p) { *p = 0u; }

__global__ void k_iota(uint32_t* __restrict__ idx, uint32_t N) {
    const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p < N) idx[p] = p;
}

// inclusive scans over the 64 lanes of a wave (all of them active) in six DPP
// steps: shifts by 1, 2, 4 and 8 within the 16-lane rows, then the rows' last
// lanes broadcast to the rows above.  Lanes without a source keep their value.
// (Shuffles go through LDS: the SAH decision of a 64-bin task took 290 of them.)
template <class Op>
__device__ __forceinline__ uint32_t wave_scan(uint32_t v, uint32_t none, Op op) {
#define RTX_SCAN_STEP(ctrl, rows) \
    v = op(v, (uint32_t)__builtin_amdgcn_update_dpp((int)none, (int)v, ctrl, rows, 0xf, false))
    RTX_SCAN_STEP(0x111, 0xf);   // row_shr:1
    RTX_SCAN_STEP(0x112, 0xf);   // row_shr:2
    RTX_SCAN_STEP(0x114, 0xf);   // row_shr:4
    RTX_SCAN_STEP(0x118, 0xf);   // row_shr:8
    RTX_SCAN_STEP(0x142, 0xa);   // row_bcast:15 into rows 1 and 3
    RTX_SCAN_STEP(0x143, 0xc);   // row_bcast:31 into rows 2 and 3
#undef RTX_SCAN_STEP
    return v;
}
__device__ __forceinline__ uint32_t scan_add(uint32_t v) {
    return wave_scan(v, 0u, [](uint32_t a, uint32_t b) { return a + b; });
}
__device__ __forceinline__ float scan_min(float v) {
    return __uint_as_float(wave_scan(__float_as_uint(v), __float_as_uint(FLT_MAX), [](uint32_t a, uint32_t b) {
        return __float_as_uint(fminf(__uint_as_float(a), __uint_as_float(b)));
    }));
}
__device__ __forceinline__ float scan_max(float v) {
    return __uint_as_float(wave_scan(__float_as_uint(v), __float_as_uint(-FLT_MAX), [](uint32_t a, uint32_t b) {
        return __float_as_uint(fmaxf(__uint_as_float(a), __uint_as_float(b)));
    }));
}

// block-wide exclusive scan of one value per thread; returns the prefix and
// the block total.  `ws` holds one slot per wave plus one.
template <int BLOCK>
__device__ __forceinline__ uint32_t block_scan(uint32_t v, uint32_t* ws, uint32_t& total) {
    const uint32_t lane = threadIdx.x & 63u, wid = threadIdx.x >> 6;
    const uint32_t x = scan_add(v);
    if (lane == 63u) ws[wid] = x;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t run = 0;
        for (int i = 0; i < BLOCK / 64; i++) { const uint32_t t = ws[i]; ws[i] = run; run += t; }
        ws[BLOCK / 64] = run;
    }
    __syncthreads();
    const uint32_t excl = ws[wid] + x - v;
    total = ws[BLOCK / 64];
    __syncthreads();
    return excl;
}

// ---------------------------------------------------------------------------
// one BVH level.  Per task: bin the primitives (3 axes x 64 bins; per-thread
// runs of equal bins are merged before the LDS atomics), evaluate SAH, choose
// leaf / SAH split / median split, partition stably.  Levels of a few big
// tasks (the top of the tree) spread each task over many blocks: partial bins
// per chunk, one block per task merges them and decides, and the partition
// runs chunk by chunk at offsets from the chunks' left counts.  Binning is a
// set of min / max / sum and the partition is stable, so both paths give the
// same tree.
// ---------------------------------------------------------------------------
// LDS state of one task's decision
struct LevelLds {
    uint32_t cnt[3][kBins];
    uint32_t b[3][kBins][12];   // lo.xyz, hi.xyz, clo.xyz, chi.xyz (ordered ints)
    uint32_t pcnt[3][kBins];    // primitives in bins 0..b
    float best_cost[3];
    int best_bin[3];
    float nb[6];                // node bounds
    int axis, bin, kind;
    uint32_t nleft;
};
static_assert(kBins == 64, "the SAH evaluation takes one bin per lane of a wave");
constexpr uint32_t kPartialWords = 3 * kBins * 13;   // counts, then bounds, of one chunk's bins

// a task's binning frame: centroid bounds low corner and bins per unit
struct TaskGeom {
    float cl[3], scale[3];
};
__device__ __forceinline__ TaskGeom task_geom(const BuildTask& task) {
    TaskGeom g;
    const float cl[3] = {task.clo.x, task.clo.y, task.clo.z};
    const float ch[3] = {task.chi.x, task.chi.y, task.chi.z};
    for (int k = 0; k < 3; k++) {
        const float ext = ch[k] - cl[k];
        g.cl[k] = cl[k];
        g.scale[k] = ext > 0.f ? (float)kBins * (1.f - 1e-6f) / ext : 0.f;
    }
    return g;
}

__device__ __forceinline__ bool bound_is_min(int k) { return k < 3 || (k >= 6 && k < 9); }

template <int BLOCK>
__device__ __forceinline__ void bins_clear(LevelLds& L) {
    for (int i = threadIdx.x; i < 3 * kBins; i += BLOCK) {
        const int ax = i / kBins, b = i % kBins;
        L.cnt[ax][b] = 0;
        for (int k = 0; k < 12; k++) L.b[ax][b][k] = bound_is_min(k) ? 0xFFFFFFFFu : 0u;
    }
}

// bins idx[r0, r1): each thread walks a contiguous run of the range
template <int BLOCK>
__device__ __forceinline__ void bins_add(LevelLds& L, const TaskGeom& g, const uint32_t* __restrict__ idx,
                                         const float4* __restrict__ plo, const float4* __restrict__ phi,
                                         uint32_t r0, uint32_t r1) {
    const uint32_t n = r1 - r0;
    const uint32_t chunk = (n + BLOCK - 1) / BLOCK;
    const uint32_t b0 = r0 + min(n, threadIdx.x * chunk);
    const uint32_t b1 = r0 + min(n, (threadIdx.x + 1) * chunk);
    int cur[3] = {-1, -1, -1};
    uint32_t cnt[3] = {0, 0, 0};
    uint32_t acc[3][12];
    auto flush = [&](int ax) {
        if (cur[ax] < 0 || cnt[ax] == 0) return;
        const int b = cur[ax];
        atomicAdd(&L.cnt[ax][b], cnt[ax]);
        for (int k = 0; k < 3; k++) {
            atomicMin(&L.b[ax][b][k], acc[ax][k]);
            atomicMax(&L.b[ax][b][3 + k], acc[ax][3 + k]);
            atomicMin(&L.b[ax][b][6 + k], acc[ax][6 + k]);
            atomicMax(&L.b[ax][b][9 + k], acc[ax][9 + k]);
        }
    };
    // (the next primitive's box and the index after it are in flight while one
    // is binned: 8 M-triangle levels over 1024 blocks 260 -> 226 us each; runs
    // of 1, 2, 4, 8 and 16 primitives a thread instead, which read whole lines,
    // flush their bins more often: 0.83, 0.97, 1.04, 1.01 and 0.93x of that
    // scene's build, against 1.03x, and 0.76 to 0.96x of a 0.5 M-triangle one)
    float4 a_next = make_float4(0.f, 0.f, 0.f, 0.f), h_next = a_next;
    uint32_t p_next = 0;
    if (b0 < b1) {
        const uint32_t p = idx[b0];
        p_next = idx[min(b0 + 1u, b1 - 1u)];
        a_next = plo[p];
        h_next = phi[p];
    }
    for (uint32_t i = b0; i < b1; i++) {
        const float4 a = a_next, h = h_next;
        a_next = plo[p_next];
        h_next = phi[p_next];
        p_next = idx[min(i + 2u, b1 - 1u)];
        const float c[3] = {.5f * (a.x + h.x), .5f * (a.y + h.y), .5f * (a.z + h.z)};
        const uint32_t v[12] = {f2o(a.x), f2o(a.y), f2o(a.z), f2o(h.x), f2o(h.y), f2o(h.z),
                                f2o(c[0]), f2o(c[1]), f2o(c[2]), f2o(c[0]), f2o(c[1]), f2o(c[2])};
#pragma unroll
        for (int ax = 0; ax < 3; ax++) {
            const int b = bin_of(c[ax], g.cl[ax], g.scale[ax]);
            if (b != cur[ax]) {
                flush(ax);
                cur[ax] = b;
                cnt[ax] = 0;
#pragma unroll
                for (int k = 0; k < 12; k++) acc[ax][k] = v[k];
            }
            cnt[ax]++;
#pragma unroll
            for (int k = 0; k < 3; k++) {
                acc[ax][k] = min(acc[ax][k], v[k]);
                acc[ax][3 + k] = max(acc[ax][3 + k], v[3 + k]);
                acc[ax][6 + k] = min(acc[ax][6 + k], v[6 + k]);
                acc[ax][9 + k] = max(acc[ax][9 + k], v[9 + k]);
            }
        }
    }
    flush(0); flush(1); flush(2);
}

// SAH decision from the task's bins (every thread of the block calls it):
// the first wave evaluates the splits, one lane per bin -- inclusive prefix
// (bins 0..b) and suffix (bins b..63) bounds and counts by wave scans; min and
// max are exact, so they equal a bin-by-bin sweep.  The split after bin b
// costs area(prefix b) * count + area(suffix b+1) * count; the cheapest wins,
// the lowest bin on ties (the order of a sweep with a strict <).  Thread 0
// then writes the node's bounds and chooses leaf / SAH split / median split.
__device__ __forceinline__ void sah_decide(LevelLds& L, const BuildTask& task, uint32_t n,
                                           BNode* __restrict__ bnodes, uint32_t max_leaf) {
    if (threadIdx.x < 64) {
        const int b = (int)threadIdx.x, m = kBins - 1 - b;
        for (int ax = 0; ax < 3; ax++) {
            const uint32_t cb = L.cnt[ax][b], cm = L.cnt[ax][m];
            // bins 0..b, and in lane b the bins 63-b..63 (a prefix of the mirrored bins)
            float pl[3], ph[3], ml[3], mh[3];
            for (int k = 0; k < 3; k++) {
                pl[k] = scan_min(cb ? o2f(L.b[ax][b][k]) : FLT_MAX);
                ph[k] = scan_max(cb ? o2f(L.b[ax][b][3 + k]) : -FLT_MAX);
                ml[k] = scan_min(cm ? o2f(L.b[ax][m][k]) : FLT_MAX);
                mh[k] = scan_max(cm ? o2f(L.b[ax][m][3 + k]) : -FLT_MAX);
            }
            const uint32_t pc = scan_add(cb), mc = scan_add(cm);
            // the suffix from bin b + 1 on is lane 62 - b's
            const float mt = area3(ml[0], ml[1], ml[2], mh[0], mh[1], mh[2]) * (float)mc;
            const int from = (kBins - 2 - b) & 63;
            const float rt = __shfl(mt, from, 64);
            const uint32_t rc0 = __shfl(mc, from, 64);
            const uint32_t rc = b < kBins - 1 ? rc0 : 0u;
            const float cost = area3(pl[0], pl[1], pl[2], ph[0], ph[1], ph[2]) * (float)pc + rt;
            const bool valid = b < kBins - 1 && pc != 0 && rc != 0 && cost < FLT_MAX;
            // the least cost, its lowest bin
            const float least = __uint_as_float(
                (uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(scan_min(valid ? cost : FLT_MAX)), 63));
            const uint64_t at = __ballot(valid && cost == least);
            L.pcnt[ax][b] = pc;
            if (b == 0) {
                L.best_cost[ax] = least;
                L.best_bin[ax] = __ffsll((unsigned long long)at) - 1;
            }
            if (ax == 0 && b == kBins - 1) {
                // node bounds: the union of the axis-0 bins
                for (int k = 0; k < 3; k++) { L.nb[k] = pl[k]; L.nb[3 + k] = ph[k]; }
            }
        }
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        const float lx = L.nb[0], ly = L.nb[1], lz = L.nb[2], hx = L.nb[3], hy = L.nb[4], hz = L.nb[5];
        BNode nd;
        nd.lo = make_float4(lx, ly, lz, 0.f);
        nd.hi = make_float4(hx, hy, hz, 0.f);
        bnodes[task.node] = nd;
        int axis = -1;
        float best = FLT_MAX;
        for (int ax = 0; ax < 3; ax++)
            if (L.best_bin[ax] >= 0 && L.best_cost[ax] < best) { best = L.best_cost[ax]; axis = ax; }
        const float A = area3(lx, ly, lz, hx, hy, hz);
        const float leaf_cost = kCostIsect * (float)n * A;
        const float split_cost = kCostTrav * A + kCostIsect * best;
        int kind;   // 0 leaf, 1 SAH split, 2 median split
        if (n <= 1) kind = 0;
        else if (n <= max_leaf && (axis < 0 || leaf_cost <= split_cost)) kind = 0;
        else if (axis < 0 || task.depth >= (uint32_t)(kMaxTreeDepth - 28)) kind = 2;
        else kind = 1;
        L.kind = kind;
        L.axis = axis;
        L.bin = axis >= 0 ? L.best_bin[axis] : -1;
        L.nleft = kind == 1 ? L.pcnt[axis][L.bin] : n / 2;
    }
    __syncthreads();
}

// the task's split record: for a SAH split the centroid bounds of the two
// children (bins 0..bin and bin+1..63, reduced by the first wave); for a
// leaf or a median split by index the task's own bounds
__device__ __forceinline__ void split_out(const LevelLds& L, const BuildTask& task, SplitOut* __restrict__ out,
                                          uint32_t slot) {
    SplitOut so;
    so.kind = L.kind == 0 ? 0u : 1u;
    so.nleft = L.nleft;
    so.pad0 = so.pad1 = 0;
    if (L.kind == 1) {
        if (threadIdx.x < 64) {
            const int ax = L.axis, sb = L.bin, b = (int)threadIdx.x;
            const bool has = L.cnt[ax][b] != 0, left = b <= sb;
            float v[12];
#pragma unroll
            for (int k = 0; k < 3; k++) {
                const float lo = o2f(L.b[ax][b][6 + k]), hi = o2f(L.b[ax][b][9 + k]);
                v[k] = has && left ? lo : FLT_MAX;
                v[3 + k] = has && left ? hi : -FLT_MAX;
                v[6 + k] = has && !left ? lo : FLT_MAX;
                v[9 + k] = has && !left ? hi : -FLT_MAX;
            }
#pragma unroll
            for (int k = 0; k < 3; k++) {
                v[k] = scan_min(v[k]);
                v[3 + k] = scan_max(v[3 + k]);
                v[6 + k] = scan_min(v[6 + k]);
                v[9 + k] = scan_max(v[9 + k]);
            }
            if (b == kBins - 1) {   // the last lane's scans hold all bins
                so.clo_l = make_float4(v[0], v[1], v[2], 0.f);
                so.chi_l = make_float4(v[3], v[4], v[5], 0.f);
                so.clo_r = make_float4(v[6], v[7], v[8], 0.f);
                so.chi_r = make_float4(v[9], v[10], v[11], 0.f);
                out[slot] = so;
            }
        }
    } else if (threadIdx.x == 0) {
        so.clo_l = so.clo_r = task.clo;
        so.chi_l = so.chi_r = task.chi;
        out[slot] = so;
    }
}

// stable partition of idx[r0, r1) into tmp: the range's primitives left of
// the split go to tmp[lbase ...], the others to tmp[rbase ...], each in order
template <int BLOCK>
__device__ __forceinline__ void partition_range(const TaskGeom& g, int ax, int sb, const uint32_t* __restrict__ idx,
                                                uint32_t* __restrict__ tmp, const float4* __restrict__ plo,
                                                const float4* __restrict__ phi, uint32_t r0, uint32_t r1,
                                                uint32_t lbase, uint32_t rbase, uint32_t* ws) {
    const int PER = 4;
    const uint32_t n = r1 - r0;
    for (uint32_t t0 = 0; t0 < n; t0 += BLOCK * PER) {
        uint32_t vals[PER];
        uint32_t flags = 0, nl = 0;
#pragma unroll
        for (int e = 0; e < PER; e++) {
            const uint32_t i = t0 + threadIdx.x * PER + e;
            vals[e] = 0;
            if (i < n) {
                const uint32_t p = idx[r0 + i];
                vals[e] = p;
                const float4 a = plo[p], h = phi[p];
                const float c = .5f * (comp4(a, ax) + comp4(h, ax));
                if (bin_of(c, g.cl[ax], g.scale[ax]) <= sb) { flags |= 1u << e; nl++; }
            }
        }
        uint32_t tot_l;
        const uint32_t pre_l = block_scan<BLOCK>(nl, ws, tot_l);
        const uint32_t cnt_here = (uint32_t)max(0, min(PER, (int)n - (int)(t0 + threadIdx.x * PER)));
        const uint32_t pre_all = min(n - t0, threadIdx.x * (uint32_t)PER);
        uint32_t l = lbase + pre_l, r = rbase + (pre_all - pre_l);
#pragma unroll
        for (int e = 0; e < PER; e++) {
            if ((uint32_t)e >= cnt_here) break;
            if (flags & (1u << e)) tmp[l++] = vals[e]; else tmp[r++] = vals[e];
        }
        const uint32_t tile_n = min((uint32_t)(BLOCK * PER), n - t0);
        lbase += tot_l;
        rbase += tile_n - tot_l;
    }
}

// one task on the whole block: bins, decision, stable partition, split record
template <int BLOCK>
__device__ __forceinline__ void level_task(LevelLds& L, uint32_t* s_ws, const BuildTask& task, uint32_t slot,
                                           const float4* __restrict__ plo, const float4* __restrict__ phi,
                                           uint32_t* __restrict__ idx, uint32_t* __restrict__ tmp,
                                           BNode* __restrict__ bnodes, SplitOut* __restrict__ out, uint32_t max_leaf) {
    const uint32_t n = task.end - task.begin;
    const TaskGeom g = task_geom(task);
    bins_clear<BLOCK>(L);
    __syncthreads();
    bins_add<BLOCK>(L, g, idx, plo, phi, task.begin, task.end);
    __syncthreads();
    sah_decide(L, task, n, bnodes, max_leaf);
    if (L.kind == 1) {
        partition_range<BLOCK>(g, L.axis, L.bin, idx, tmp, plo, phi, task.begin, task.end, task.begin,
                               task.begin + L.nleft, s_ws);
        __syncthreads();
        for (uint32_t i = threadIdx.x; i < n; i += BLOCK) idx[task.begin + i] = tmp[task.begin + i];
    }
    split_out(L, task, out, slot);
}

// one block per task
template <int BLOCK>
__global__ __launch_bounds__(BLOCK) void k_level(
        const Level* __restrict__ lev, const BuildTask* __restrict__ tasks, const float4* __restrict__ plo,
        const float4* __restrict__ phi, uint32_t* __restrict__ idx, uint32_t* __restrict__ tmp,
        BNode* __restrict__ bnodes, SplitOut* __restrict__ out, uint32_t max_leaf) {
    __shared__ LevelLds L;
    __shared__ uint32_t s_ws[BLOCK / 64 + 1];
    if (blockIdx.x >= lev->n) return;
    level_task<BLOCK>(L, s_ws, tasks[blockIdx.x], blockIdx.x, plo, phi, idx, tmp, bnodes, out, max_leaf);
}

// ---------------------------------------------------------------------------
// Levels of small tasks: a thread per task of at most kTinyTask primitives,
// a wave per listed bigger task.  The thread makes the wave's decision: the
// same bins, prefix and suffix bounds as minima and maxima over the same
// primitives, the same cost expression and the same tie rule (the lowest
// bin).  It evaluates only the splits after an occupied bin: a split after
// an empty bin partitions like the split after the occupied bin below it and
// has the same cost at a higher bin, so it never wins.  (A minimum over
// zeros of both signs may keep the other sign than the wave's; the boxes and
// SAH costs are equal as numbers either way.)
#ifndef RTX_TINY_BITS
#define RTX_TINY_BITS 4
#endif
constexpr uint32_t kTinyBits = RTX_TINY_BITS;     // position bits of a sort key
constexpr uint32_t kTinyTask = 1u << kTinyBits;   // a power of two (the bitonic sort)
constexpr uint32_t kTinyLevel = 8192;  // tasks of a level below which a wave per task runs them all (fewer launches)
constexpr uint32_t kListGrid = 4096;   // waves of the listed-task kernel at most

__device__ __forceinline__ float centroid(const float4& a, const float4& h, int ax) {
    return .5f * (comp4(a, ax) + comp4(h, ax));
}

__device__ void tiny_task(const BuildTask& task, uint32_t slot, const float4* __restrict__ plo,
                          const float4* __restrict__ phi, uint32_t* __restrict__ idx, uint32_t* __restrict__ tmp,
                          BNode* __restrict__ bnodes, SplitOut* __restrict__ out, uint32_t max_leaf) {
    const uint32_t n = task.end - task.begin;
    const TaskGeom g = task_geom(task);
    const uint32_t* ix = idx + task.begin;
    float nlx = FLT_MAX, nly = FLT_MAX, nlz = FLT_MAX, nhx = -FLT_MAX, nhy = -FLT_MAX, nhz = -FLT_MAX;
    for (uint32_t i = 0; i < n; i++) {
        const uint32_t p = ix[i];
        const float4 a = plo[p], h = phi[p];
        nlx = fminf(nlx, a.x); nly = fminf(nly, a.y); nlz = fminf(nlz, a.z);
        nhx = fmaxf(nhx, h.x); nhy = fmaxf(nhy, h.y); nhz = fmaxf(nhz, h.z);
    }
    float best_cost[3];
    int best_bin[3];
    for (int ax = 0; ax < 3; ax++) {
        // the primitives in order of their bin (bin << kTinyBits | position, a bitonic
        // sort over kTinyTask register slots; absent slots sort last)
        uint32_t key[kTinyTask];
#pragma unroll
        for (uint32_t i = 0; i < kTinyTask; i++) {
            key[i] = 0xFFFFFFFFu;
            if (i < n) {
                const uint32_t p = ix[i];
                key[i] = ((uint32_t)bin_of(centroid(plo[p], phi[p], ax), g.cl[ax], g.scale[ax]) << kTinyBits) | i;
            }
        }
#pragma unroll
        for (uint32_t k = 2; k <= kTinyTask; k <<= 1) {
#pragma unroll
            for (uint32_t j = k >> 1; j > 0; j >>= 1) {
#pragma unroll
                for (uint32_t i = 0; i < kTinyTask; i++) {
                    const uint32_t l = i ^ j;
                    if (l > i) {
                        const uint32_t a = key[i], b = key[l];
                        const bool lo_first = (i & k) == 0;
                        key[i] = lo_first ? min(a, b) : max(a, b);
                        key[l] = lo_first ? max(a, b) : min(a, b);
                    }
                }
            }
        }
        // prefix terms area(bins <= bin of position k) * count and suffix terms
        // area(bins of positions >= k) * count, as the wave's scans form them
        float tl[kTinyTask], tr[kTinyTask];
        float lx0 = FLT_MAX, ly0 = FLT_MAX, lz0 = FLT_MAX, lx1 = -FLT_MAX, ly1 = -FLT_MAX, lz1 = -FLT_MAX;
#pragma unroll
        for (uint32_t k = 0; k < kTinyTask; k++) {
            tl[k] = 0.f;
            if (k < n) {
                const uint32_t p = ix[key[k] & (kTinyTask - 1u)];
                const float4 a = plo[p], h = phi[p];
                lx0 = fminf(lx0, a.x); ly0 = fminf(ly0, a.y); lz0 = fminf(lz0, a.z);
                lx1 = fmaxf(lx1, h.x); ly1 = fmaxf(ly1, h.y); lz1 = fmaxf(lz1, h.z);
                tl[k] = area3(lx0, ly0, lz0, lx1, ly1, lz1) * (float)(k + 1);
            }
        }
        float rx0 = FLT_MAX, ry0 = FLT_MAX, rz0 = FLT_MAX, rx1 = -FLT_MAX, ry1 = -FLT_MAX, rz1 = -FLT_MAX;
#pragma unroll
        for (int k = (int)kTinyTask - 1; k >= 0; k--) {
            tr[k] = 0.f;
            if ((uint32_t)k < n) {
                const uint32_t p = ix[key[k] & (kTinyTask - 1u)];
                const float4 a = plo[p], h = phi[p];
                rx0 = fminf(rx0, a.x); ry0 = fminf(ry0, a.y); rz0 = fminf(rz0, a.z);
                rx1 = fmaxf(rx1, h.x); ry1 = fmaxf(ry1, h.y); rz1 = fmaxf(rz1, h.z);
                tr[k] = area3(rx0, ry0, rz0, rx1, ry1, rz1) * (float)(n - (uint32_t)k);
            }
        }
        // a split after bin b of position k: position k + 1 holds a higher bin
        uint64_t best = ~0ull;
#pragma unroll
        for (uint32_t k = 0; k + 1 < kTinyTask; k++) {
            if (k + 1 < n && (key[k] >> kTinyBits) != (key[k + 1] >> kTinyBits)) {
                const float cost = tl[k] + tr[k + 1];
                if (cost < FLT_MAX) {
                    const uint64_t c = ((uint64_t)__float_as_uint(cost) << 32) | (key[k] >> kTinyBits);
                    best = c < best ? c : best;
                }
            }
        }
        best_cost[ax] = best == ~0ull ? FLT_MAX : __uint_as_float((uint32_t)(best >> 32));
        best_bin[ax] = best == ~0ull ? -1 : (int)(uint32_t)best;
    }
    BNode nd;
    nd.lo = make_float4(nlx, nly, nlz, 0.f);
    nd.hi = make_float4(nhx, nhy, nhz, 0.f);
    bnodes[task.node] = nd;
    int axis = -1;
    float best = FLT_MAX;
    for (int ax = 0; ax < 3; ax++)
        if (best_bin[ax] >= 0 && best_cost[ax] < best) { best = best_cost[ax]; axis = ax; }
    const float A = area3(nlx, nly, nlz, nhx, nhy, nhz);
    const float leaf_cost = kCostIsect * (float)n * A;
    const float split_cost = kCostTrav * A + kCostIsect * best;
    int kind;   // 0 leaf, 1 SAH split, 2 median split (as in sah_decide)
    if (n <= 1) kind = 0;
    else if (n <= max_leaf && (axis < 0 || leaf_cost <= split_cost)) kind = 0;
    else if (axis < 0 || task.depth >= (uint32_t)(kMaxTreeDepth - 28)) kind = 2;
    else kind = 1;
    SplitOut so;
    so.kind = kind == 0 ? 0u : 1u;
    so.pad0 = so.pad1 = 0;
    if (kind == 1) {
        // stable partition into tmp and back, with the centroid bounds of both sides
        const int sb = best_bin[axis];
        float llx = FLT_MAX, lly = FLT_MAX, llz = FLT_MAX, lhx = -FLT_MAX, lhy = -FLT_MAX, lhz = -FLT_MAX;
        float rlx = FLT_MAX, rly = FLT_MAX, rlz = FLT_MAX, rhx = -FLT_MAX, rhy = -FLT_MAX, rhz = -FLT_MAX;
        uint32_t nl = 0;
        for (uint32_t i = 0; i < n; i++) {
            const uint32_t p = ix[i];
            const float4 a = plo[p], h = phi[p];
            const float cx = centroid(a, h, 0), cy = centroid(a, h, 1), cz = centroid(a, h, 2);
            const float ca = axis == 0 ? cx : (axis == 1 ? cy : cz);
            if (bin_of(ca, g.cl[axis], g.scale[axis]) <= sb) {
                llx = fminf(llx, cx); lly = fminf(lly, cy); llz = fminf(llz, cz);
                lhx = fmaxf(lhx, cx); lhy = fmaxf(lhy, cy); lhz = fmaxf(lhz, cz);
                tmp[task.begin + nl++] = p;
            } else {
                rlx = fminf(rlx, cx); rly = fminf(rly, cy); rlz = fminf(rlz, cz);
                rhx = fmaxf(rhx, cx); rhy = fmaxf(rhy, cy); rhz = fmaxf(rhz, cz);
            }
        }
        uint32_t r = nl;
        for (uint32_t i = 0; i < n; i++) {
            const uint32_t p = ix[i];
            if (bin_of(centroid(plo[p], phi[p], axis), g.cl[axis], g.scale[axis]) > sb) tmp[task.begin + r++] = p;
        }
        for (uint32_t i = 0; i < n; i++) idx[task.begin + i] = tmp[task.begin + i];
        so.nleft = nl;
        so.clo_l = make_float4(llx, lly, llz, 0.f);
        so.chi_l = make_float4(lhx, lhy, lhz, 0.f);
        so.clo_r = make_float4(rlx, rly, rlz, 0.f);
        so.chi_r = make_float4(rhx, rhy, rhz, 0.f);
    } else {
        so.nleft = n / 2;
        so.clo_l = so.clo_r = task.clo;
        so.chi_l = so.chi_r = task.chi;
    }
    out[slot] = so;
}

// a thread per task; tasks above kTinyTask primitives are appended to `big`
// (one atomic per wave: their order in the list does not matter, each task
// writes only its own slot and primitive range)
__global__ __launch_bounds__(256) void k_level_tiny(const Level* __restrict__ lev, const BuildTask* __restrict__ tasks,
                                                    const float4* __restrict__ plo, const float4* __restrict__ phi,
                                                    uint32_t* __restrict__ idx, uint32_t* __restrict__ tmp,
                                                    BNode* __restrict__ bnodes, SplitOut* __restrict__ out,
                                                    uint32_t max_leaf, uint32_t* __restrict__ big,
                                                    uint32_t* __restrict__ nbig) {
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    bool is_big = false;
    if (t < lev->n) {
        const BuildTask task = tasks[t];
        if (task.end - task.begin > kTinyTask) is_big = true;
        else tiny_task(task, t, plo, phi, idx, tmp, bnodes, out, max_leaf);
    }
    const uint64_t m = __ballot(is_big);
    if (m) {
        const uint32_t lane = threadIdx.x & 63u;
        const int first = __ffsll((unsigned long long)m) - 1;
        uint32_t base = 0;
        if (lane == (uint32_t)first) base = atomicAdd(nbig, (uint32_t)__popcll(m));
        base = __shfl(base, first, 64);
        if (is_big) big[base + (uint32_t)__popcll(m & ((1ull << lane) - 1ull))] = t;
    }
}

// a wave per listed task, grid-strided over the list
__global__ __launch_bounds__(64) void k_level_list(const BuildTask* __restrict__ tasks,
                                                   const uint32_t* __restrict__ big, const uint32_t* __restrict__ nbig,
                                                   const float4* __restrict__ plo, const float4* __restrict__ phi,
                                                   uint32_t* __restrict__ idx, uint32_t* __restrict__ tmp,
                                                   BNode* __restrict__ bnodes, SplitOut* __restrict__ out,
                                                   uint32_t max_leaf) {
    __shared__ LevelLds L;
    __shared__ uint32_t s_ws[2];
    const uint32_t nb = *nbig;
    for (uint32_t k = blockIdx.x; k < nb; k += gridDim.x) {
        const uint32_t t = big[k];
        level_task<64>(L, s_ws, tasks[t], t, plo, phi, idx, tmp, bnodes, out, max_leaf);
        __syncthreads();
    }
}

// big tasks, step 1: block (chunk c, task t) bins chunk c of the task into
// partial[t * G + c]
__device__ __forceinline__ void chunk_range(const BuildTask& task, uint32_t G, uint32_t c, uint32_t& r0,
                                            uint32_t& r1) {
    const uint32_t n = task.end - task.begin, chunk = (n + G - 1) / G;
    r0 = task.begin + min(n, c * chunk);
    r1 = task.begin + min(n, (c + 1) * chunk);
}

template <int BLOCK>
__global__ __launch_bounds__(BLOCK) void k_bin_wide(const Level* __restrict__ lev,
                                                    const BuildTask* __restrict__ tasks, const float4* __restrict__ plo,
                                                    const float4* __restrict__ phi, const uint32_t* __restrict__ idx,
                                                    uint32_t G, uint32_t* __restrict__ partial) {
    __shared__ LevelLds L;
    if (blockIdx.y >= lev->n) return;
    const BuildTask task = tasks[blockIdx.y];
    uint32_t r0, r1;
    chunk_range(task, G, blockIdx.x, r0, r1);
    bins_clear<BLOCK>(L);
    __syncthreads();
    bins_add<BLOCK>(L, task_geom(task), idx, plo, phi, r0, r1);
    __syncthreads();
    uint32_t* P = partial + (size_t)(blockIdx.y * G + blockIdx.x) * kPartialWords;
    const uint32_t* c = &L.cnt[0][0];
    const uint32_t* bb = &L.b[0][0][0];
    for (uint32_t i = threadIdx.x; i < 3 * kBins; i += BLOCK) P[i] = c[i];
    for (uint32_t i = threadIdx.x; i < 3 * kBins * 12; i += BLOCK) P[3 * kBins + i] = bb[i];
}

// big tasks, step 2a: the chunks' bins of each task merged into one set
// (sums of counts, minima and maxima of bounds: exact, in any order).
// Block (x, t) merges words 16x .. 16x+15 of task t: 16 groups of 16
// threads each reduce every 16th chunk, then the first group the groups.
constexpr uint32_t kMergeWords = 16;
static_assert(kPartialWords % kMergeWords == 0, "whole blocks of merged words");
__global__ __launch_bounds__(256) void k_merge_wide(const Level* __restrict__ lev,
                                                    uint32_t G, const uint32_t* __restrict__ partial,
                                                    uint32_t* __restrict__ merged) {
    __shared__ uint32_t s_v[256 / kMergeWords][kMergeWords + 1];
    if (blockIdx.y >= lev->n) return;
    const uint32_t w = threadIdx.x % kMergeWords, grp = threadIdx.x / kMergeWords;
    const uint32_t i = blockIdx.x * kMergeWords + w;
    // word kind: 0 count (sum), 1 lower bound (min), 2 upper bound (max)
    const int kind = i < 3 * kBins ? 0 : (bound_is_min((int)((i - 3 * kBins) % 12)) ? 1 : 2);
    const uint32_t* P = partial + (size_t)blockIdx.y * G * kPartialWords + i;
    uint32_t v = kind == 1 ? 0xFFFFFFFFu : 0u;
    for (uint32_t k = grp; k < G; k += 256 / kMergeWords) {
        const uint32_t x = P[(size_t)k * kPartialWords];
        v = kind == 0 ? v + x : (kind == 1 ? min(v, x) : max(v, x));
    }
    s_v[grp][w] = v;
    __syncthreads();
    if (grp == 0) {
        for (uint32_t g = 1; g < 256 / kMergeWords; g++) {
            const uint32_t x = s_v[g][w];
            v = kind == 0 ? v + x : (kind == 1 ? min(v, x) : max(v, x));
        }
        merged[(size_t)blockIdx.y * kPartialWords + i] = v;
    }
}

// big tasks, step 2b: one block per task reads its G sets of bins (one, after
// k_merge_wide), merges them and decides as k_level does; wsplit[t] = (kind,
// axis, bin, nleft) for the partition
template <int BLOCK>
__global__ __launch_bounds__(BLOCK) void k_decide_wide(const Level* __restrict__ lev,
                                                       const BuildTask* __restrict__ tasks, uint32_t G,
                                                       const uint32_t* __restrict__ partial,
                                                       BNode* __restrict__ bnodes, SplitOut* __restrict__ out,
                                                       uint4* __restrict__ wsplit, uint32_t max_leaf) {
    __shared__ LevelLds L;
    if (blockIdx.x >= lev->n) return;
    const BuildTask task = tasks[blockIdx.x];
    const uint32_t* P = partial + (size_t)blockIdx.x * G * kPartialWords;
    uint32_t* c = &L.cnt[0][0];
    uint32_t* bb = &L.b[0][0][0];
    for (uint32_t i = threadIdx.x; i < 3 * kBins; i += BLOCK) {
        uint32_t s = 0;
        for (uint32_t k = 0; k < G; k++) s += P[(size_t)k * kPartialWords + i];
        c[i] = s;
    }
    for (uint32_t i = threadIdx.x; i < 3 * kBins * 12; i += BLOCK) {
        const bool mn = bound_is_min((int)(i % 12));
        uint32_t v = mn ? 0xFFFFFFFFu : 0u;
        for (uint32_t k = 0; k < G; k++) {
            const uint32_t x = P[(size_t)k * kPartialWords + 3 * kBins + i];
            v = mn ? min(v, x) : max(v, x);
        }
        bb[i] = v;
    }
    __syncthreads();
    sah_decide(L, task, task.end - task.begin, bnodes, max_leaf);
    split_out(L, task, out, blockIdx.x);
    if (threadIdx.x == 0) wsplit[blockIdx.x] = make_uint4((uint32_t)L.kind, (uint32_t)L.axis, (uint32_t)L.bin, L.nleft);
}

// big tasks, step 3: primitives left of the split in each chunk, from the
// chunk's own bins (a wave per chunk, a lane per bin; a pass over the
// primitives took 0.12 ms per level of 8 M)
__global__ __launch_bounds__(256) void k_count_wide(const Level* __restrict__ lev,
                                                    uint32_t G, const uint32_t* __restrict__ partial,
                                                    const uint4* __restrict__ wsplit, uint32_t* __restrict__ lcount) {
    const uint32_t c = blockIdx.x * 4u + (threadIdx.x >> 6), b = threadIdx.x & 63u;
    if (blockIdx.y >= lev->n) return;
    const uint4 w = wsplit[blockIdx.y];
    if (w.x != 1u || c >= G) return;   // the whole wave: no SAH split, or past the last chunk
    const size_t chunk = (size_t)blockIdx.y * G + c;
    uint32_t n = b <= w.z ? partial[chunk * kPartialWords + w.y * kBins + b] : 0u;
    for (int off = 32; off > 0; off >>= 1) n += __shfl_xor(n, off, 64);
    if (b == 0) lcount[chunk] = n;
}

// big tasks, step 4: each chunk partitions stably into tmp after the left
// and right primitives of the chunks before it
template <int BLOCK>
__global__ __launch_bounds__(BLOCK) void k_scatter_wide(const Level* __restrict__ lev,
                                                        const BuildTask* __restrict__ tasks,
                                                        const float4* __restrict__ plo,
                                                        const float4* __restrict__ phi, const uint32_t* __restrict__ idx,
                                                        uint32_t* __restrict__ tmp, uint32_t G,
                                                        const uint4* __restrict__ wsplit,
                                                        const uint32_t* __restrict__ lcount) {
    __shared__ uint32_t s_ws[BLOCK / 64 + 1];
    __shared__ uint32_t s_lb;
    if (blockIdx.y >= lev->n) return;
    const uint4 w = wsplit[blockIdx.y];
    if (w.x != 1u) return;
    const BuildTask task = tasks[blockIdx.y];
    uint32_t r0, r1;
    chunk_range(task, G, blockIdx.x, r0, r1);
    if (threadIdx.x == 0) s_lb = 0;
    __syncthreads();
    uint32_t before_me = 0;
    for (uint32_t k = threadIdx.x; k < blockIdx.x; k += BLOCK) before_me += lcount[blockIdx.y * G + k];
    if (before_me) atomicAdd(&s_lb, before_me);
    __syncthreads();
    const uint32_t lb = s_lb, before = r0 - task.begin;
    partition_range<BLOCK>(task_geom(task), (int)w.y, (int)w.z, idx, tmp, plo, phi, r0, r1, task.begin + lb,
                           task.begin + w.w + (before - lb), s_ws);
}

// big tasks, step 5: the partitioned ranges back into idx
__global__ void k_copy_wide(const Level* __restrict__ lev,
                            const BuildTask* __restrict__ tasks, uint32_t G, const uint4* __restrict__ wsplit,
                            const uint32_t* __restrict__ tmp, uint32_t* __restrict__ idx) {
    if (blockIdx.y >= lev->n || wsplit[blockIdx.y].x != 1u) return;
    uint32_t r0, r1;
    chunk_range(tasks[blockIdx.y], G, blockIdx.x, r0, r1);
    for (uint32_t i = r0 + threadIdx.x; i < r1; i += blockDim.x) idx[i] = tmp[i];
}

// The values of a level to scan: its tasks' split flags (each split makes two
// tasks) or its wide nodes' counts of inner children.
struct KindOf {
    const SplitOut* so;
    static constexpr uint32_t kMakes = 2;
    __device__ __forceinline__ uint32_t operator()(uint32_t i) const { return so[i].kind; }
};
struct CountOf {
    const uint32_t* p;
    static constexpr uint32_t kMakes = 1;
    __device__ __forceinline__ uint32_t operator()(uint32_t i) const { return p[i]; }
};
// the next level, after lev[0], from the sum of a level's values
__device__ __forceinline__ void level_next(Level* lev, uint32_t n, uint32_t* host) {
    lev[1].n = n;
    lev[1].first = lev[0].first + lev[0].n;
    __hip_atomic_store(host, n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// exclusive scan of a level's values by one block -> out; the next level
template <class Get>
__global__ __launch_bounds__(kScanBlock) void k_scan(Level* __restrict__ lev, Get get, uint32_t* __restrict__ out,
                                                    uint32_t* __restrict__ host) {
    __shared__ uint32_t s_ws[kScanBlock / 64 + 1];
    const uint32_t n = lev->n;
    uint32_t carry = 0;
    for (uint32_t base = 0; base < n; base += kScanBlock) {
        const uint32_t i = base + threadIdx.x;
        const uint32_t v = i < n ? get(i) : 0u;
        uint32_t tot;
        const uint32_t ex = block_scan<kScanBlock>(v, s_ws, tot);
        if (i < n) out[i] = carry + ex;
        carry += tot;
    }
    if (threadIdx.x == 0) level_next(lev, Get::kMakes * carry, host);
}

// the same scan over many blocks, for long levels: tile sums, a scan of
// them by one block, then each tile rescanned from its offset
constexpr uint32_t kScanTile = 4 * kScanBlock;
template <class Get>
__global__ __launch_bounds__(kScanBlock) void k_scan_tiles(const Level* __restrict__ lev, Get get,
                                                          uint32_t* __restrict__ tsum) {
    __shared__ uint32_t s_n;
    const uint32_t n = lev->n;
    if (threadIdx.x == 0) s_n = 0;
    __syncthreads();
    uint32_t c = 0;
    const uint32_t b0 = blockIdx.x * kScanTile;
    for (uint32_t i = b0 + threadIdx.x; i < n && i < b0 + kScanTile; i += kScanBlock) c += get(i);
    if (c) atomicAdd(&s_n, c);
    __syncthreads();
    if (threadIdx.x == 0) tsum[blockIdx.x] = s_n;
}
__global__ __launch_bounds__(kScanBlock) void k_scan_sums(Level* __restrict__ lev, uint32_t makes,
                                                         const uint32_t* __restrict__ tsum,
                                                         uint32_t* __restrict__ toff, uint32_t* __restrict__ host) {
    __shared__ uint32_t s_ws[kScanBlock / 64 + 1];
    const uint32_t nt = (lev->n + kScanTile - 1) / kScanTile;
    uint32_t carry = 0;
    for (uint32_t base = 0; base < nt; base += kScanBlock) {
        const uint32_t i = base + threadIdx.x;
        const uint32_t v = i < nt ? tsum[i] : 0u;
        uint32_t tot;
        const uint32_t ex = block_scan<kScanBlock>(v, s_ws, tot);
        if (i < nt) toff[i] = carry + ex;
        carry += tot;
    }
    if (threadIdx.x == 0) level_next(lev, makes * carry, host);
}
template <class Get>
__global__ __launch_bounds__(kScanBlock) void k_scan_apply(const Level* __restrict__ lev, Get get,
                                                          const uint32_t* __restrict__ toff,
                                                          uint32_t* __restrict__ out) {
    __shared__ uint32_t s_ws[kScanBlock / 64 + 1];
    const uint32_t n = lev->n, b0 = blockIdx.x * kScanTile;
    if (b0 >= n) return;
    uint32_t carry = toff[blockIdx.x];
    for (uint32_t base = b0; base < b0 + kScanTile && base < n; base += kScanBlock) {
        const uint32_t i = base + threadIdx.x;
        const uint32_t v = i < n ? get(i) : 0u;
        uint32_t tot;
        const uint32_t ex = block_scan<kScanBlock>(v, s_ws, tot);
        if (i < n) out[i] = carry + ex;
        carry += tot;
    }
}

// (lev[1], the next level, is written by the scan before)
__global__ void k_emit(const Level* __restrict__ lev, const BuildTask* __restrict__ tasks,
                       const SplitOut* __restrict__ so, const uint32_t* __restrict__ rank, BNode* __restrict__ bnodes,
                       BuildTask* __restrict__ next) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= lev[0].n) return;
    const uint32_t node_base = lev[1].first;
    const BuildTask t = tasks[i];
    const SplitOut s = so[i];
    if (s.kind == 0) {
        bnodes[t.node].lo.w = __uint_as_float(t.begin);
        bnodes[t.node].hi.w = __uint_as_float(t.end - t.begin);
        return;
    }
    const uint32_t L = node_base + 2 * rank[i];
    bnodes[t.node].lo.w = __uint_as_float(L);
    bnodes[t.node].hi.w = __uint_as_float(0u);
    BuildTask a, b;
    a.node = L; a.begin = t.begin; a.end = t.begin + s.nleft; a.depth = t.depth + 1;
    a.clo = s.clo_l; a.chi = s.chi_l;
    b.node = L + 1; b.begin = t.begin + s.nleft; b.end = t.end; b.depth = t.depth + 1;
    b.clo = s.clo_r; b.chi = s.chi_r;
    next[2 * rank[i]] = a;
    next[2 * rank[i] + 1] = b;
}

// SAH cost (relative to the root area) and largest leaf of the finished binary
// tree (statistics): grid-strided partial sums, a wave reduction, then one
// atomic per block (the order of the double sums varies from run to run in the
// last bits).  The counts of leaves and inner nodes and the depth follow from
// the counts of nodes and levels: every inner node has two children, and the
// last level holds only leaves.
constexpr uint32_t kSahBlocks = 1024;
__global__ __launch_bounds__(256) void k_sah(const BNode* __restrict__ bnodes, uint32_t nnodes,
                                             BuildStats* __restrict__ st) {
    __shared__ double s_v[256 / 64];
    __shared__ uint32_t s_m[256 / 64];
    double v = 0.0;
    uint32_t most = 0;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < nnodes; i += gridDim.x * blockDim.x) {
        const BNode nd = bnodes[i];
        const float a = area3(nd.lo.x, nd.lo.y, nd.lo.z, nd.hi.x, nd.hi.y, nd.hi.z);
        const uint32_t cnt = __float_as_uint(nd.hi.w);
        v += cnt ? (double)kCostIsect * cnt * a : (double)kCostTrav * a;
        most = max(most, cnt);
    }
    for (int off = 32; off > 0; off >>= 1) {
        v += __shfl_down(v, off, 64);
        most = max(most, (uint32_t)__shfl_down(most, off, 64));
    }
    if ((threadIdx.x & 63) == 0) {
        s_v[threadIdx.x >> 6] = v;
        s_m[threadIdx.x >> 6] = most;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0.0;
        for (int w = 0; w < 256 / 64; w++) {
            t += s_v[w];
            most = max(most, s_m[w]);
        }
        if (t != 0.0) atomicAdd(&st->sah, t);
        if (most) atomicMax(&st->max_leaf, most);
    }
}

// ---------------------------------------------------------------------------
// collapse of the binary tree into 4-wide nodes, level by level from the root
// (the grouping of builds with RTX_DP_COLLAPSE=0; the default is the
// SAH-optimal one below).  A wide node starts from a binary node's two
// children and repeatedly opens the inner child of largest surface area until
// it has 4 children or only leaves; its inner children become the wide nodes
// of the next level.
__global__ void k_collapse4(const Level* __restrict__ lev, const BNode* __restrict__ bn,
                            const uint32_t* __restrict__ front, uint4* __restrict__ cid, uint32_t* __restrict__ ninner) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= lev->n) return;
    const uint32_t L = __float_as_uint(bn[front ? front[i] : 0u].lo.w);
    uint32_t c0 = L, c1 = L + 1, c2 = kNoChild, c3 = kNoChild;
    uint32_t cnt = 2;
    for (int it = 0; it < 2; it++) {
        // inner child of largest area among c0..c(cnt-1)
        float best = -1.f;
        int bk = -1;
        for (int k = 0; k < 4; k++) {
            const uint32_t c = k == 0 ? c0 : k == 1 ? c1 : k == 2 ? c2 : c3;
            if ((uint32_t)k >= cnt) break;
            const BNode b = bn[c];
            if (__float_as_uint(b.hi.w) != 0u) continue;    // leaf
            const float a = area3(b.lo.x, b.lo.y, b.lo.z, b.hi.x, b.hi.y, b.hi.z);
            if (a > best) { best = a; bk = k; }
        }
        if (bk < 0) break;
        const uint32_t opened = bk == 0 ? c0 : bk == 1 ? c1 : bk == 2 ? c2 : c3;
        const uint32_t Lb = __float_as_uint(bn[opened].lo.w);
        if (bk == 0) c0 = Lb; else if (bk == 1) c1 = Lb; else if (bk == 2) c2 = Lb; else c3 = Lb;
        if (cnt == 2) c2 = Lb + 1; else c3 = Lb + 1;
        cnt++;
    }
    uint32_t m = 0;
    for (int k = 0; k < 4; k++) {
        const uint32_t c = k == 0 ? c0 : k == 1 ? c1 : k == 2 ? c2 : c3;
        if (c != kNoChild && __float_as_uint(bn[c].hi.w) == 0u) m++;
    }
    cid[i] = make_uint4(c0, c1, c2, c3);
    ninner[i] = m;
}

// ---------------------------------------------------------------------------
// SAH-optimal collapse (after Ylitie, Karras and Laine 2017, "Efficient
// incoherent ray traversal on GPUs through compressed wide BVHs", for 4-wide
// nodes).  D(n, k) is the least SAH cost of the binary subtree at n as a
// forest of at most k roots, each root a leaf (all the subtree's primitives,
// at most max_leaf, contiguous in the leaf order) or a 4-wide node whose
// children are a forest of at most 4 roots under it:
//   D(n, 1) = min(A(n) * n_prims * C_isect  [n_prims <= max_leaf],
//                 A(n) * C_trav + min_i D(L, i) + D(R, 4 - i))
//   D(n, k) = min(D(n, 1), min_{0<i<k} D(L, i) + D(R, k - i))
// bottom-up, one binary level at a time (the build allocates the nodes level
// by level, so a level's children are all in the next one).  A binary leaf
// stays a leaf; the root stays a 4-wide node.  The collapse then takes each
// wide node's children from the choices (split of the 4 roots between L and
// R, then each subtree's own split).  The binary tree and its statistics are
// unchanged; only the grouping into 4-wide nodes and leaves is.
//
// meta bits: 0 the subtree is one leaf; 1-2 the split of 4 roots between L
// and R (1..3 to L); 3-4, 5-6, 7-8 the split for k = 2, 3, 4 (0: the subtree
// itself is the one root, else the roots given to L)
__global__ void k_dp_level(const BNode* __restrict__ bn, uint32_t begin, uint32_t n, float4* __restrict__ dc,
                           uint32_t* __restrict__ ntri, uint32_t* __restrict__ first, uint32_t* __restrict__ meta,
                           uint32_t max_leaf) {
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    const uint32_t i = begin + t;
    const BNode b = bn[i];
    const float A = area3(b.lo.x, b.lo.y, b.lo.z, b.hi.x, b.hi.y, b.hi.z);
    const uint32_t cnt = __float_as_uint(b.hi.w);
    if (cnt) {
        const float c = A * (float)cnt * kCostIsect;
        dc[i] = make_float4(c, c, c, c);
        ntri[i] = cnt;
        first[i] = __float_as_uint(b.lo.w);
        meta[i] = 1u;
        return;
    }
    const uint32_t L = __float_as_uint(b.lo.w), R = L + 1u;
    const float4 dl = dc[L], dr = dc[R];
    const float l[5] = {0.f, dl.x, dl.y, dl.z, dl.w}, r[5] = {0.f, dr.x, dr.y, dr.z, dr.w};
    float d2[5];
    uint32_t b2[5];
    for (int k = 2; k <= 4; k++) {
        float best = l[1] + r[k - 1];
        uint32_t bi = 1;
        for (int s = 2; s < k; s++) {
            const float c = l[s] + r[k - s];
            if (c < best) { best = c; bi = (uint32_t)s; }
        }
        d2[k] = best;
        b2[k] = bi;
    }
    const uint32_t nt = ntri[L] + ntri[R];
    const float cnode = A * kCostTrav + d2[4];
    const bool leaf = i != 0u && nt <= max_leaf && A * (float)nt * kCostIsect <= cnode;
    const float d1 = leaf ? A * (float)nt * kCostIsect : cnode;
    uint32_t m = (leaf ? 1u : 0u) | (b2[4] << 1);
    float d[5];
    d[1] = d1;
    for (int k = 2; k <= 4; k++) {
        const bool self = d1 <= d2[k];
        d[k] = self ? d1 : d2[k];
        m |= (self ? 0u : b2[k]) << (3 + 2 * (k - 2));
    }
    dc[i] = make_float4(d[1], d[2], d[3], d[4]);
    ntri[i] = nt;
    first[i] = first[L];
    meta[i] = m;
}

// the children of the wide node at binary node front[i]: the forest of 4
// roots that the choices give under it (left subtree first)
__global__ void k_collapse4_dp(const Level* __restrict__ lev, const BNode* __restrict__ bn,
                               const uint32_t* __restrict__ front, const uint32_t* __restrict__ meta,
                               uint4* __restrict__ cid, uint32_t* __restrict__ ninner) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= lev->n) return;
    const uint32_t b = front ? front[i] : 0u;   // the first level is the root alone
    const uint32_t L = __float_as_uint(bn[b].lo.w);
    const uint32_t kl = (meta[b] >> 1) & 3u;
    // (subtree, roots) pairs still to expand; their roots add up to 4, so
    // neither the stack nor the output holds more than 4
    uint32_t sn[4], sk[4], out[4] = {kNoChild, kNoChild, kNoChild, kNoChild};
    int sp = 0, no = 0;
    sn[sp] = L + 1u; sk[sp++] = 4u - kl;
    sn[sp] = L; sk[sp++] = kl;
    while (sp > 0) {
        --sp;
        const uint32_t x = sn[sp], k = sk[sp];
        const uint32_t mx = meta[x];
        const uint32_t s = k == 1u ? 0u : (mx >> (3u + 2u * (k - 2u))) & 3u;
        if (s == 0u) {
            out[no++] = x;
        } else {
            const uint32_t XL = __float_as_uint(bn[x].lo.w);
            sn[sp] = XL + 1u; sk[sp++] = k - s;
            sn[sp] = XL; sk[sp++] = s;
        }
    }
    uint32_t m = 0;
    for (int k = 0; k < no; k++) m += (meta[out[k]] & 1u) ? 0u : 1u;
    cid[i] = make_uint4(out[0], out[1], out[2], out[3]);
    ninner[i] = m;
}

// Writes the wide nodes of one level.  With meta (the SAH-optimal collapse)
// a child is a leaf when its subtree is one (primitives first[c] ..
// first[c] + ntri[c] - 1 of the leaf order); without, when it is a binary leaf.
__global__ void k_write4(const Level* __restrict__ lev, const BNode* __restrict__ bn, const uint4* __restrict__ cid,
                         const uint32_t* __restrict__ off, uint32_t empty_ref, float4* __restrict__ nodes4,
                         uint32_t* __restrict__ next_front, const uint32_t* __restrict__ meta,
                         const uint32_t* __restrict__ ntri, const uint32_t* __restrict__ first) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= lev[0].n) return;
    const uint32_t base_this = lev[0].first, base_next = lev[1].first;
    const uint4 c4 = cid[i];
    float lo[4][3], hi[4][3];
    bool used[4];
    uint32_t ref[4];
    uint32_t j = off[i];
    for (int k = 0; k < 4; k++) {
        const uint32_t c = k == 0 ? c4.x : k == 1 ? c4.y : k == 2 ? c4.z : c4.w;
        used[k] = c != kNoChild;
        if (!used[k]) {
            // an empty slot: an inverted box, which no slab test accepts; its
            // ref is a one-triangle leaf holding a degenerate triangle (no
            // ray hits it), so even then the traversal would stay in bounds
            for (int a = 0; a < 3; a++) lo[k][a] = hi[k][a] = 0.f;
            ref[k] = empty_ref;
            continue;
        }
        const BNode b = bn[c];
        lo[k][0] = b.lo.x; hi[k][0] = b.hi.x;
        lo[k][1] = b.lo.y; hi[k][1] = b.hi.y;
        lo[k][2] = b.lo.z; hi[k][2] = b.hi.z;
        const uint32_t cntp = __float_as_uint(b.hi.w);
        if (meta && (meta[c] & 1u)) {
            ref[k] = leaf_ref(first[c], ntri[c]);
        } else if (!meta && cntp) {
            ref[k] = leaf_ref(__float_as_uint(b.lo.w), cntp);
        } else {
            ref[k] = base_next + j;
            next_front[j] = c;
            j++;
        }
    }
    encode_node(nodes4 + kWideNodeF4 * (size_t)(base_this + i), lo, hi, used, ref);
}

__global__ void k_gather_tris(const float4* __restrict__ tri_world, const uint32_t* __restrict__ idx, uint32_t N,
                              float4* __restrict__ tris) {
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k == N) {
        // the degenerate triangle behind the empty slots of 4-wide nodes
        const float4 p = make_float4(kFarAway, kFarAway, kFarAway, __uint_as_float(kNoHit));
        tris[3 * (size_t)N + 0] = p;
        tris[3 * (size_t)N + 1] = make_float4(kFarAway, kFarAway, kFarAway, 0.f);
        tris[3 * (size_t)N + 2] = make_float4(kFarAway, kFarAway, kFarAway, __uint_as_float(kNoHit));
        return;
    }
    if (k > N) return;
    const size_t p = idx[k];
    tris[3 * (size_t)k + 0] = tri_world[3 * p + 0];
    tris[3 * (size_t)k + 1] = tri_world[3 * p + 1];
    tris[3 * (size_t)k + 2] = tri_world[3 * p + 2];
}

template <typename T>
struct DevBuf {
    T* p = nullptr;
    hipError_t alloc(size_t n) { return hipMalloc((void**)&p, sizeof(T) * (n ? n : 1)); }
    ~DevBuf() { if (p) (void)hipFree(p); }
    T* release() { T* q = p; p = nullptr; return q; }
};

#define RTX_TRY(expr)                                                              \
    do {                                                                           \
        hipError_t e_ = (expr);                                                    \
        if (e_ != hipSuccess) { if (err) *err = std::string(#expr) + ": " + hipGetErrorString(e_); return e_; } \
    } while (0)

inline uint32_t blocks_for(uint64_t n, uint32_t b) { return (uint32_t)((n + b - 1) / b); }

}  // namespace

hipError_t flatten_scene(const InstBuild* d_insts, uint32_t ninst, const MeshRef* d_meshes, uint32_t N,
                         float4* d_tri_world, float4* d_plo, float4* d_phi, hipStream_t s) {
    if (N == 0) return hipSuccess;
    hipLaunchKernelGGL(k_flatten, dim3(blocks_for(N, 256)), dim3(256), 0, s, d_insts, ninst, d_meshes, N,
                       d_tri_world, d_plo, d_phi);
    return hipGetLastError();
}

// ---- workspace of a build ---------------------------------------------------
namespace {
struct KeptBlock {
    std::mutex taken;          // held by the build that uses the block
    uint8_t* base = nullptr;
    size_t cap = 0;
    uint32_t small = 0;        // builds in a row that took a small part of it
    uint32_t* host = nullptr;
};
constexpr int kMaxDevices = 64;
KeptBlock g_kept[kMaxDevices];
size_t round256(size_t n) { return (n + 255) / 256 * 256; }
}  // namespace

BuildWorkspace::BuildWorkspace(int device, size_t bytes) : device_(device) {
    if (device < 0 || device >= kMaxDevices || !g_kept[device].taken.try_lock()) return;
    KeptBlock& k = g_kept[device];
    shared_ = true;
    k.small = k.cap > kShrinkBytes && bytes < k.cap / 8 ? k.small + 1 : 0;
    if (bytes <= kKeepBytes && (k.cap < bytes || k.small == kShrinkAfter)) {
        k.small = 0;
        if (k.base) (void)hipFree(k.base);
        k.base = nullptr;
        k.cap = 0;
        if (hipMalloc((void**)&k.base, bytes) == hipSuccess) k.cap = bytes;
        else (void)hipGetLastError();   // take() allocates piece by piece then
    }
    if (!k.host && hipHostMalloc((void**)&k.host, kHostWords * sizeof(uint32_t), 0) != hipSuccess) k.host = nullptr;
    base_ = k.base;
    cap_ = k.cap;
    host_ = k.host;
}

BuildWorkspace::~BuildWorkspace() {
    if (!done_) (void)hipDeviceSynchronize();   // a build that failed may still be running
    for (void* p : more_) (void)hipFree(p);
    if (shared_) g_kept[device_].taken.unlock();
    else if (host_) (void)hipHostFree(host_);
}

hipError_t BuildWorkspace::take(void** p, size_t bytes) {
    const size_t n = round256(bytes);
    if (used_ + n <= cap_) {
        *p = base_ + used_;
        used_ += n;
        return hipSuccess;
    }
    const hipError_t e = hipMalloc(p, bytes);
    if (e == hipSuccess) more_.push_back(*p);
    return e;
}

hipError_t BuildWorkspace::host_words(uint32_t** h) {
    if (!host_) {
        const hipError_t e = hipHostMalloc((void**)&host_, kHostWords * sizeof(uint32_t), 0);
        if (e != hipSuccess) {
            host_ = nullptr;
            return e;
        }
        if (shared_) g_kept[device_].host = host_;
    }
    *h = host_;
    return hipSuccess;
}

bool build_workspace_drop(int device) {
    if (device < 0 || device >= kMaxDevices) return false;
    KeptBlock& k = g_kept[device];
    if (!k.taken.try_lock()) return false;   // a build is running
    const bool had = k.base != nullptr;
    if (k.base) (void)hipFree(k.base);
    if (k.host) (void)hipHostFree(k.host);
    k.base = nullptr;
    k.host = nullptr;
    k.cap = 0;
    k.small = 0;
    k.taken.unlock();
    return had;
}

size_t bvh_workspace_bytes(uint32_t N) {
    const size_t n = N ? N : 1;
    size_t b = 2 * round256(4 * n) + round256(sizeof(BNode) * 2 * n);                             // idx, tmp, bnodes
    b += round256(4 * n) + 2 * round256(sizeof(BuildTask) * n) + round256(sizeof(SplitOut) * n);  // rank, tasks, so
    b += round256(4 * (n / (kTinyTask + 1) + 1)) + 2 * round256(4 * (n / kScanTile + 2));
    if (N >= kWideMinPrims) b += sizeof(uint32_t) * kPartialWords * (size_t)(kWideBlocks + kWideTasks) + 65536;
    return b + 65536;
}

size_t bvh_result_bytes(uint32_t N) {
    const size_t n = N ? N : 1;
    return round256(sizeof(float4) * 3 * (n + 1)) + round256(sizeof(float4) * kWideNodeF4 * n) + round256(4 * n) + 1024;
}

namespace {
// events of the levels in flight, destroyed at scope exit
struct LevelEvents {
    hipEvent_t e[2] = {nullptr, nullptr};
    hipError_t init() {
        for (auto& x : e) {
            const hipError_t r = hipEventCreateWithFlags(&x, hipEventDisableTiming);
            if (r != hipSuccess) return r;
        }
        return hipSuccess;
    }
    ~LevelEvents() { for (auto& x : e) if (x) (void)hipEventDestroy(x); }
};
}  // namespace

hipError_t build_bvh(const float4* d_tri_world, const float4* d_plo, const float4* d_phi, uint32_t N,
                     hipStream_t s, BuildWorkspace& ws, BuiltBVH* outp, std::string* err, const BvhOptions& opt) {
    BuiltBVH out;
    const uint32_t max_leaf = opt.max_leaf < 1 ? 1u : (opt.max_leaf > kMaxLeaf ? kMaxLeaf : opt.max_leaf);
    if (N == 0) {
        out.root = kEmptyRoot;
        *outp = out;
        return hipSuccess;
    }
    uint32_t* host = nullptr;
    RTX_TRY(ws.host_words(&host));
    LevelEvents ev;
    RTX_TRY(ev.init());
    // results that stay in the workspace come first
    float4 *tris_ws = nullptr, *wide = nullptr;
    uint32_t* idx = nullptr;
    if (!opt.owned) {
        RTX_TRY(ws.get(&wide, kWideNodeF4 * (size_t)N));
        if (opt.gather) RTX_TRY(ws.get(&tris_ws, 3 * ((size_t)N + 1)));
        else RTX_TRY(ws.get(&idx, N));
    }
    const size_t m_all = ws.mark();
    uint32_t *tmp = nullptr, *rank = nullptr, *rb = nullptr, *big = nullptr, *nbig = nullptr, *tsum = nullptr,
             *toff = nullptr, *partial = nullptr, *merged = nullptr, *lcount = nullptr;
    BuildTask *tasks_a = nullptr, *tasks_b = nullptr;
    SplitOut* so = nullptr;
    BNode* bnodes = nullptr;
    BuildStats* st = nullptr;
    Level *lev = nullptr, *wlev = nullptr;
    uint4* wsplit = nullptr;
    if (!idx) RTX_TRY(ws.get(&idx, N));
    RTX_TRY(ws.get(&bnodes, 2 * (size_t)N));
    RTX_TRY(ws.get(&st, 1));
    RTX_TRY(ws.get(&lev, kMaxLevels + 1));
    RTX_TRY(ws.get(&wlev, kMaxLevels + 1));
    RTX_TRY(ws.get(&tsum, (size_t)N / kScanTile + 2));
    RTX_TRY(ws.get(&toff, (size_t)N / kScanTile + 2));
    const size_t m_levels = ws.mark();   // from here on: the binary tree's levels, then the collapse's arrays
    RTX_TRY(ws.get(&tmp, N));
    RTX_TRY(ws.get(&rank, N));
    RTX_TRY(ws.get(&tasks_a, N));
    RTX_TRY(ws.get(&tasks_b, N));
    RTX_TRY(ws.get(&so, N));
    RTX_TRY(ws.get(&rb, 6));
    if (N >= kWideMinPrims) {
        // chunks of a wide level: G * tasks <= N / kWideMinChunk; tasks <= N / kWideMinPrims
        const uint32_t nchunks = std::min(kWideBlocks, N / kWideMinChunk);
        const uint32_t nwide = std::min(kWideTasks, N / kWideMinPrims);
        RTX_TRY(ws.get(&partial, (size_t)nchunks * kPartialWords));
        RTX_TRY(ws.get(&merged, (size_t)nwide * kPartialWords));
        RTX_TRY(ws.get(&lcount, nchunks));
        RTX_TRY(ws.get(&wsplit, nwide));
    }
    // tasks of a small-task level above kTinyTask primitives (at most N / (kTinyTask + 1))
    RTX_TRY(ws.get(&big, N / (kTinyTask + 1) + 1));
    RTX_TRY(ws.get(&nbig, 1));

    hipLaunchKernelGGL(k_iota, dim3(blocks_for(N, 256)), dim3(256), 0, s, idx, N);
    hipLaunchKernelGGL(k_root_init, dim3(1), dim3(64), 0, s, rb, st, lev, wlev);
    hipLaunchKernelGGL(k_root_bounds, dim3(std::min<uint32_t>(blocks_for(N, 256), kRootBlocks)), dim3(256), 0, s,
                       d_plo, d_phi, N, rb);
    hipLaunchKernelGGL(k_root_task, dim3(1), dim3(64), 0, s, rb, N, tasks_a);
    RTX_TRY(hipGetLastError());

    // exclusive scan of a level's values (`most` of them at most) into out, the
    // next level into l[1] and its count to h
    auto scan = [&](Level* l, auto get, uint32_t most, uint32_t* o, uint32_t* h) {
        using Get = decltype(get);
        if (most <= 16 * kScanTile) {
            hipLaunchKernelGGL(k_scan<Get>, dim3(1), dim3(kScanBlock), 0, s, l, get, o, h);
            return;
        }
        const uint32_t nt = (most + kScanTile - 1) / kScanTile;
        hipLaunchKernelGGL(k_scan_tiles<Get>, dim3(nt), dim3(kScanBlock), 0, s, l, get, tsum);
        hipLaunchKernelGGL(k_scan_sums, dim3(1), dim3(kScanBlock), 0, s, l, Get::kMakes, tsum, toff, h);
        hipLaunchKernelGGL(k_scan_apply<Get>, dim3(nt), dim3(kScanBlock), 0, s, l, get, toff, o);
    };

    // The levels, one ahead of the device: level d is launched for the most
    // tasks it can have (two per task of level d - 1) once level d - 2 is done,
    // which gave level d - 1's count, while level d - 1 runs.  (A wait per level
    // left the device idle for 30 to 40 us each: with the shared workspace a
    // level-4 scene builds in 3.8 ms host to host, 8.9 before, and the level-6
    // one in 21.5, 27.6 before.)  The last level launched is an empty one.
    BuildTask* cur = tasks_a;
    BuildTask* nxt = tasks_b;
    std::vector<uint32_t> level_first;   // binary level d: nodes level_first[d] .. level_first[d+1]-1
    uint32_t nnodes = 0;
    for (uint32_t d = 0, known = 1;; d++) {
        // known: tasks of level d - 1 (of the root level for d = 0)
        if (d >= 2) {
            RTX_TRY(hipEventSynchronize(ev.e[d & 1u]));
            known = ((volatile uint32_t*)host)[(d - 1) % kMaxLevels];
            if (known == 0) break;
        }
        if (d != 1) {
            level_first.push_back(nnodes);
            nnodes += known;
        }
        if (d && d % kMaxLevels == 0) hipLaunchKernelGGL(k_level_wrap, dim3(1), dim3(1), 0, s, lev);
        const uint32_t most = (uint32_t)std::min<uint64_t>(N, d == 0 ? 1u : 2ull * known);
        Level* l = lev + d % kMaxLevels;
        // a few big tasks: each spread over G chunks (kWideBlocks in all, of
        // kWideMinChunk primitives at least on average), their bins merged by
        // k_merge_wide; a wave per task once tasks average fewer than
        // kSmallTask primitives, and on levels of kTinyLevel tasks or more a
        // thread per task of at most kTinyTask primitives (the same tree every
        // way: binning, SAH and partition do not depend on the split)
        if (most <= kWideTasks && (uint64_t)N >= (uint64_t)kWideMinPrims * most) {
            const uint32_t G = std::min(kWideBlocks / most, N / (most * kWideMinChunk));
            const dim3 gw(G, most);
            hipLaunchKernelGGL(k_bin_wide<kBuildBlock>, gw, dim3(kBuildBlock), 0, s, l, cur, d_plo, d_phi, idx, G,
                               partial);
            hipLaunchKernelGGL(k_merge_wide, dim3(kPartialWords / kMergeWords, most), dim3(256), 0, s, l, G, partial,
                               merged);
            hipLaunchKernelGGL(k_decide_wide<kBuildBlock>, dim3(most), dim3(kBuildBlock), 0, s, l, cur, 1u, merged,
                               bnodes, so, wsplit, max_leaf);
            hipLaunchKernelGGL(k_count_wide, dim3((G + 3) / 4, most), dim3(256), 0, s, l, G, partial, wsplit, lcount);
            hipLaunchKernelGGL(k_scatter_wide<kBuildBlock>, gw, dim3(kBuildBlock), 0, s, l, cur, d_plo, d_phi, idx,
                               tmp, G, wsplit, lcount);
            hipLaunchKernelGGL(k_copy_wide, gw, dim3(256), 0, s, l, cur, G, wsplit, tmp, idx);
        } else if ((uint64_t)N < (uint64_t)kSmallTask * most && most < kTinyLevel) {
            hipLaunchKernelGGL(k_level<64>, dim3(most), dim3(64), 0, s, l, cur, d_plo, d_phi, idx, tmp, bnodes, so,
                               max_leaf);
        } else if ((uint64_t)N < (uint64_t)kSmallTask * most) {
            hipLaunchKernelGGL(k_zero_word, dim3(1), dim3(1), 0, s, nbig);
            hipLaunchKernelGGL(k_level_tiny, dim3(blocks_for(most, 256)), dim3(256), 0, s, l, cur, d_plo, d_phi, idx,
                               tmp, bnodes, so, max_leaf, big, nbig);
            hipLaunchKernelGGL(k_level_list, dim3(std::min(most, kListGrid)), dim3(64), 0, s, cur, big, nbig, d_plo,
                               d_phi, idx, tmp, bnodes, so, max_leaf);
        } else
            hipLaunchKernelGGL(k_level<kBuildBlock>, dim3(most), dim3(kBuildBlock), 0, s, l, cur, d_plo, d_phi, idx,
                               tmp, bnodes, so, max_leaf);
        scan(l, KindOf{so}, most, rank, host + (d + 1) % kMaxLevels);
        hipLaunchKernelGGL(k_emit, dim3(blocks_for(most, 256)), dim3(256), 0, s, l, cur, so, rank, bnodes, nxt);
        RTX_TRY(hipGetLastError());
        RTX_TRY(hipEventRecord(ev.e[d & 1u], s));
        std::swap(cur, nxt);
    }
    level_first.push_back(nnodes);

    hipLaunchKernelGGL(k_sah, dim3(std::min(blocks_for(nnodes, 256), kSahBlocks)), dim3(256), 0, s, bnodes, nnodes,
                       st);
    RTX_TRY(hipGetLastError());
    const uint32_t ninner = (nnodes - 1) / 2;

    DevBuf<float4> nodes, tris;
    float4* tris_out = tris_ws;
    if (opt.gather) {
        if (opt.owned) {
            RTX_TRY(tris.alloc(3 * ((size_t)N + 1)));
            tris_out = tris.p;
        }
        hipLaunchKernelGGL(k_gather_tris, dim3(blocks_for((uint64_t)N + 1, 256)), dim3(256), 0, s, d_tri_world, idx, N,
                           tris_out);
        RTX_TRY(hipGetLastError());
    }

    // 4-wide nodes: at most one per binary inner node
    ws.reset(m_levels);
    uint32_t nwide = 0, wide_depth = 0;
    if (ninner) {
        const uint32_t *wmeta = nullptr, *wntri = nullptr, *wfirst = nullptr;
#if RTX_DP_COLLAPSE
        // the collapse's choices, bottom-up by binary level
        float4* dpc = nullptr;
        uint32_t *dp_ntri = nullptr, *dp_first = nullptr, *dp_meta = nullptr;
        RTX_TRY(ws.get(&dpc, nnodes));
        RTX_TRY(ws.get(&dp_ntri, nnodes));
        RTX_TRY(ws.get(&dp_first, nnodes));
        RTX_TRY(ws.get(&dp_meta, nnodes));
        for (size_t d = level_first.size() - 1; d-- > 0;) {
            const uint32_t b = level_first[d], n = level_first[d + 1] - b;
            hipLaunchKernelGGL(k_dp_level, dim3(blocks_for(n, 256)), dim3(256), 0, s, bnodes, b, n, dpc, dp_ntri,
                               dp_first, dp_meta, max_leaf);
        }
        RTX_TRY(hipGetLastError());
        wmeta = dp_meta;
        wntri = dp_ntri;
        wfirst = dp_first;
#endif
        uint32_t *fa = nullptr, *fb = nullptr, *cnt = nullptr, *off = nullptr;
        uint4* cid = nullptr;
        if (!wide) RTX_TRY(ws.get(&wide, kWideNodeF4 * (size_t)ninner));
        RTX_TRY(ws.get(&fa, ninner));
        RTX_TRY(ws.get(&fb, ninner));
        RTX_TRY(ws.get(&cnt, ninner));
        RTX_TRY(ws.get(&off, ninner));
        RTX_TRY(ws.get(&cid, ninner));
        // the levels of the 4-wide tree, one ahead of the device like the
        // binary ones (a node has at most four inner children)
        uint32_t* whost = host + kMaxLevels;
        uint32_t* wcur = nullptr;   // the first level is the root alone
        uint32_t* wnxt = fa;
        for (uint32_t d = 0, known = 1;; d++) {
            if (d >= 2) {
                RTX_TRY(hipEventSynchronize(ev.e[d & 1u]));
                known = ((volatile uint32_t*)whost)[(d - 1) % kMaxLevels];
                if (known == 0) break;
            }
            if (d != 1) {
                out.level_begin.push_back(nwide);
                nwide += known;
                wide_depth++;
            }
            if (d && d % kMaxLevels == 0) hipLaunchKernelGGL(k_level_wrap, dim3(1), dim3(1), 0, s, wlev);
            const uint32_t most = (uint32_t)std::min<uint64_t>(ninner, d == 0 ? 1u : 4ull * known);
            Level* l = wlev + d % kMaxLevels;
            const dim3 g(blocks_for(most, 256)), b(256);
#if RTX_DP_COLLAPSE
            hipLaunchKernelGGL(k_collapse4_dp, g, b, 0, s, l, bnodes, wcur, wmeta, cid, cnt);
#else
            hipLaunchKernelGGL(k_collapse4, g, b, 0, s, l, bnodes, wcur, cid, cnt);
#endif
            scan(l, CountOf{cnt}, most, off, whost + (d + 1) % kMaxLevels);
            hipLaunchKernelGGL(k_write4, g, b, 0, s, l, bnodes, cid, off, leaf_ref(N, 1), wide, wnxt, wmeta, wntri,
                               wfirst);
            RTX_TRY(hipGetLastError());
            RTX_TRY(hipEventRecord(ev.e[d & 1u], s));
            wcur = wnxt;
            wnxt = wnxt == fa ? fb : fa;
        }
    }
    BuildStats* hst = (BuildStats*)(host + 2 * kMaxLevels);
    BNode* hroot = (BNode*)(hst + 1);
    static_assert(kMaxLevels % 4 == 0 && sizeof(BuildStats) % 16 == 0, "aligned records");
    static_assert(8 * kMaxLevels + sizeof(BuildStats) + sizeof(BNode) <= 4 * BuildWorkspace::kHostWords, "host words");
    RTX_TRY(hipMemcpyAsync(hst, st, sizeof(BuildStats), hipMemcpyDeviceToHost, s));
    RTX_TRY(hipMemcpyAsync(hroot, bnodes, sizeof(BNode), hipMemcpyDeviceToHost, s));
    if (opt.owned) {
        RTX_TRY(nodes.alloc(kWideNodeF4 * (size_t)(nwide ? nwide : 1)));
        if (nwide)
            RTX_TRY(hipMemcpyAsync(nodes.p, wide, sizeof(float4) * kWideNodeF4 * (size_t)nwide,
                                   hipMemcpyDeviceToDevice, s));
    }
    RTX_TRY(hipStreamSynchronize(s));
    const BNode root = *hroot;
    out.level_begin.push_back(nwide);

    const uint32_t root_cnt = __builtin_bit_cast(uint32_t, root.hi.w);
    const float rx = root.hi.x - root.lo.x, ry = root.hi.y - root.lo.y, rz = root.hi.z - root.lo.z;
    const double root_area = 2.0 * ((double)rx * ry + (double)ry * rz + (double)rz * rx);
    out.nodes = opt.owned ? nodes.release() : wide;
    out.tris = opt.owned ? tris.release() : tris_ws;
    if (!opt.gather) out.order = idx;
    out.root_lo[0] = root.lo.x; out.root_lo[1] = root.lo.y; out.root_lo[2] = root.lo.z;
    out.root_hi[0] = root.hi.x; out.root_hi[1] = root.hi.y; out.root_hi[2] = root.hi.z;
    out.root = root_cnt ? leaf_ref(__builtin_bit_cast(uint32_t, root.lo.w), root_cnt) : 0u;
    out.num_nodes = ninner;
    out.num_wide = nwide;
    out.wide_depth = wide_depth;
    out.num_leaves = nnodes - ninner;
    out.max_depth = (uint32_t)level_first.size() - 1;
    out.max_leaf = hst->max_leaf;
    out.sah = root_area > 0.0 ? hst->sah / root_area : 0.0;
    ws.reset(m_all);
    *outp = out;
    return hipSuccess;
}

}  // namespace rtx
