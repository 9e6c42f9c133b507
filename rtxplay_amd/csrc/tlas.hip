// tlas.hip -- assembly and refit of a two-level scene: the instance
// acceleration structure (IAS) over per-mesh geometry structures (GAS) of
// optx/scene.cxx:38-294, here one 4-wide BVH per mesh over its object-space
// triangles (bottom level) and one over the instances' world boxes (top
// level), all in one node array and one triangle array.
//
// The trees come from build_bvh (bvh_build.hip).  Assembly copies each
// bottom-level tree into the scene arrays and adds the array offsets to its
// refs; the top level's leaves (one instance each) become instance refs.
// Scene::update (optx/scene.cxx:275-294, an OptiX refit) becomes a refit of
// the top level's boxes, level by level from the deepest, with the topology
// kept.
#include <hip/hip_runtime.h>

#include "bvh_build.h"
#include "node.h"

namespace rtx {

namespace {

__device__ __forceinline__ float comp(const float4& v, int j) {
    return j == 0 ? v.x : (j == 1 ? v.y : (j == 2 ? v.z : v.w));
}
__device__ __forceinline__ void set_comp(float4& v, int j, float x) {
    if (j == 0) v.x = x; else if (j == 1) v.y = x; else if (j == 2) v.z = x; else v.w = x;
}

// bottom-level tree copied to node index node_base / triangle index tri_base
__global__ void k_relocate(float4* __restrict__ nodes, uint32_t n, uint32_t node_base, uint32_t tri_base) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float4* o = nodes + (size_t)kWideNodeF4 * (node_base + i);
    float4 rf = o[kNodeRefs];
    for (int j = 0; j < 4; j++) {
        uint32_t r = __float_as_uint(comp(rf, j));
        if (r & kLeafFlag) r += tri_base;           // first triangle (bits 0..26; the host checks the range)
        else if (r != kNoChild) r += node_base;
        set_comp(rf, j, __uint_as_float(r));
    }
    o[kNodeRefs] = rf;
}

// top-level tree: leaf k (one primitive, order[k]) holds instance
// inst_of[order[k]]; the empty slots' leaf (first == nprim) the null instance
__global__ void k_tlas_leaves(float4* __restrict__ nodes, uint32_t n, const uint32_t* __restrict__ order,
                              uint32_t nprim, const uint32_t* __restrict__ inst_of, uint32_t null_inst) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float4* o = nodes + (size_t)kWideNodeF4 * i;
    float4 rf = o[kNodeRefs];
    for (int j = 0; j < 4; j++) {
        const uint32_t r = __float_as_uint(comp(rf, j));
        if (!(r & kLeafFlag)) continue;
        const uint32_t first = r & kLeafFirstMask;
        const uint32_t id = first < nprim ? inst_of[order[first]] : null_inst;
        set_comp(rf, j, __uint_as_float(kInstLeaf | id));
    }
    o[kNodeRefs] = rf;
}

// one level of the top-level refit: each child slot gets the instance's world
// box (ibox: lo, hi per instance) or the inner child's own box (tbox: lo, hi
// per top-level node, written here one level deeper before); slots of the null
// instance stay empty
__global__ void k_refit4(float4* __restrict__ nodes, uint32_t begin, uint32_t n, const float4* __restrict__ ibox,
                         float4* __restrict__ tbox, uint32_t null_ref) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float4* o = nodes + (size_t)kWideNodeF4 * (begin + i);
    const float4 rf = o[kNodeRefs];
    float lo[4][3], hi[4][3], bl[3], bh[3];
    bool used[4];
    uint32_t ref[4];
    for (int k = 0; k < 3; k++) { bl[k] = __builtin_huge_valf(); bh[k] = -__builtin_huge_valf(); }
    for (int j = 0; j < 4; j++) {
        const uint32_t r = __float_as_uint(comp(rf, j));
        ref[j] = r;
        used[j] = r != null_ref;
        const float4* b = (r & kInstLeaf) == kInstLeaf ? ibox + 2 * (size_t)(r & kLeafFirstMask) : tbox + 2 * (size_t)r;
        const float4 a = b[0], c = b[1];
        lo[j][0] = a.x; lo[j][1] = a.y; lo[j][2] = a.z;
        hi[j][0] = c.x; hi[j][1] = c.y; hi[j][2] = c.z;
        if (!used[j]) continue;
        for (int k = 0; k < 3; k++) {
            bl[k] = fminf(bl[k], lo[j][k]);
            bh[k] = fmaxf(bh[k], hi[j][k]);
        }
    }
    encode_node(o, lo, hi, used, ref);
    tbox[2 * (size_t)(begin + i)] = make_float4(bl[0], bl[1], bl[2], 0.f);
    tbox[2 * (size_t)(begin + i) + 1] = make_float4(bh[0], bh[1], bh[2], 0.f);
}

inline uint32_t blocks256(uint32_t n) { return (n + 255u) / 256u; }

}  // namespace

hipError_t relocate_blas(float4* nodes, uint32_t n, uint32_t node_base, uint32_t tri_base, hipStream_t s) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_relocate, dim3(blocks256(n)), dim3(256), 0, s, nodes, n, node_base, tri_base);
    return hipGetLastError();
}

hipError_t tlas_leaves(float4* nodes, uint32_t n, const uint32_t* order, uint32_t nprim, const uint32_t* inst_of,
                       uint32_t null_inst, hipStream_t s) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_tlas_leaves, dim3(blocks256(n)), dim3(256), 0, s, nodes, n, order, nprim, inst_of,
                       null_inst);
    return hipGetLastError();
}

hipError_t refit_tlas(float4* nodes, const std::vector<uint32_t>& level_begin, const float4* ibox, float4* tbox,
                      uint32_t null_ref, hipStream_t s) {
    // level_begin: first node of each level, then the node count
    for (size_t l = level_begin.size(); l-- > 1;) {
        const uint32_t b = level_begin[l - 1], n = level_begin[l] - b;
        if (n == 0) continue;
        hipLaunchKernelGGL(k_refit4, dim3(blocks256(n)), dim3(256), 0, s, nodes, b, n, ibox, tbox, null_ref);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace rtx
