// bvh_build.h -- host interface of the device acceleration-structure build.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <string>
#include <vector>

#include "rtx_internal.h"

namespace rtx {

// one mesh as uploaded by rtx_mesh_add (device pointers)
struct MeshRef {
    const float* vces;     // 3 floats per vertex
    const uint32_t* ices;  // 3 indices per triangle
    uint32_t nv, ni;
};

// one instance for the flatten kernel: 3x4 row-major transform, mesh, first
// world-space triangle of the instance
struct InstBuild {
    float xf[12];
    uint32_t mesh;
    uint32_t tri_base;
    uint32_t pad[2];
};

struct BuiltBVH {
    float4* nodes = nullptr;    // kWideNodeF4 float4 per 4-wide node (owned)
    float4* tris = nullptr;     // 3 float4 per triangle, leaf order, + 1 degenerate triangle at N (owned; gather only)
    uint32_t* order = nullptr;  // leaf order -> primitive (owned; without gather only)
    uint32_t root = kEmptyRoot;
    uint32_t num_nodes = 0, num_leaves = 0, max_depth = 0, max_leaf = 0;   // of the binary SAH tree
    uint32_t num_wide = 0, wide_depth = 0;                                    // of the 4-wide tree
    float root_lo[3] = {0.f, 0.f, 0.f}, root_hi[3] = {0.f, 0.f, 0.f};      // bounds of all primitives
    std::vector<uint32_t> level_begin;   // first wide node of each level (+ the total at the end)
    double sah = 0.0;
};

struct BvhOptions {
    uint32_t max_leaf = kMaxLeaf;   // primitives per leaf at most (1..kMaxLeaf)
    bool gather = true;             // write the leaf-ordered triangles (else return the leaf order; not with owned)
    bool owned = true;              // the result's arrays are allocations of their own (else parts of the workspace)
};

// Device memory of one build: a block that the builds of a device share (one
// at a time; a build that finds it taken by another thread has its own) and
// what does not fit it as allocations of their own, freed with the lease.
// Allocating and freeing the temporaries took 7.5 ms of the 28 ms of the
// 8M-triangle level-6 scene and 9 of 18 ms of the mixed two-level one (now,
// with the levels launched ahead, 21.5 and 8.0 ms, host to host).  The
// block is kept between builds up to kKeepBytes; it shrinks once kShrinkAfter
// builds in a row took less than an eighth of it, and is freed with the
// device's last context, by rtx_ctx_trim, and where an allocation of the
// library finds no memory (build_workspace_drop).  A build ends with its stream
// synchronized, so the next one may use the block on any stream.
class BuildWorkspace {
public:
    static constexpr size_t kKeepBytes = (size_t)4 << 30;
    static constexpr size_t kShrinkBytes = (size_t)64 << 20;   // smaller blocks do not shrink
    static constexpr uint32_t kShrinkAfter = 8;
    // for a build that takes `bytes` at once at most (with that device current)
    BuildWorkspace(int device, size_t bytes);
    ~BuildWorkspace();
    BuildWorkspace(const BuildWorkspace&) = delete;
    BuildWorkspace& operator=(const BuildWorkspace&) = delete;
    template <class T>
    hipError_t get(T** p, size_t n) { return take((void**)p, sizeof(T) * (n ? n : 1)); }
    size_t mark() const { return used_; }
    void reset(size_t m) { used_ = m; }       // gives back what was taken since mark()
    // kHostWords words of pinned host memory that kernels write counts to
    static constexpr uint32_t kHostWords = 1024;
    hipError_t host_words(uint32_t** h);
    // the build's stream has been synchronized after its last use of the memory
    void done() { done_ = true; }

private:
    hipError_t take(void** p, size_t bytes);
    int device_;
    bool shared_ = false, done_ = false;
    uint8_t* base_ = nullptr;
    uint32_t* host_ = nullptr;
    size_t cap_ = 0, used_ = 0;
    std::vector<void*> more_;
};
// frees the block of a device unless a build uses it; false: nothing to free.
// Not for the thread of a running build.
bool build_workspace_drop(int device);
// the workspace bytes that build_bvh over N primitives usually takes (what
// goes beyond is allocated then) and that its result takes when not owned
size_t bvh_workspace_bytes(uint32_t N);
size_t bvh_result_bytes(uint32_t N);

// world-space triangles (3 float4 each: xyz | prim id, inst id, mesh prim) and
// per-primitive bounds, in instance-major order
hipError_t flatten_scene(const InstBuild* d_insts, uint32_t ninst, const MeshRef* d_meshes, uint32_t N,
                         float4* d_tri_world, float4* d_plo, float4* d_phi, hipStream_t s);

// binned SAH BVH over N flattened triangles; synchronous on s
// (without gather, d_tri_world is not read and may be null)
hipError_t build_bvh(const float4* d_tri_world, const float4* d_plo, const float4* d_phi, uint32_t N,
                     hipStream_t s, BuildWorkspace& ws, BuiltBVH* out, std::string* err,
                     const BvhOptions& opt = BvhOptions());

// ---- two-level scenes (tlas.hip) ----
// adds node_base / tri_base to the refs of a bottom-level tree of n wide
// nodes that was copied to nodes[node_base ...] and its triangles to tri_base
hipError_t relocate_blas(float4* nodes, uint32_t n, uint32_t node_base, uint32_t tri_base, hipStream_t s);
// turns the leaf refs of a top-level tree (n wide nodes at nodes[0], one
// primitive per leaf, order = its leaf order over nprim primitives) into
// instance refs kInstLeaf | inst_of[primitive]; empty slots get null_inst
hipError_t tlas_leaves(float4* nodes, uint32_t n, const uint32_t* order, uint32_t nprim, const uint32_t* inst_of,
                       uint32_t null_inst, hipStream_t s);
// refits the top-level boxes from ibox (world lo, hi float4 per instance),
// deepest level first; null_ref = kInstLeaf | null instance; tbox: scratch of
// 2 float4 per top-level node (the nodes' own boxes)
hipError_t refit_tlas(float4* nodes, const std::vector<uint32_t>& level_begin, const float4* ibox, float4* tbox,
                      uint32_t null_ref, hipStream_t s);

}  // namespace rtx
