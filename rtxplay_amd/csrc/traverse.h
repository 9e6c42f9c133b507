// traverse.h -- closest-hit query on the device: the work optixTrace does on
// RT cores in the reference (optx/camera_r.cu:82-99, optx/optics_r.cu:115-132).
//
// Software traversal of the 4-wide BVH (layout in rtx_internal.h) with a
// per-lane stack whose first SLDS entries live in LDS (one column per lane,
// bank-conflict free) and the rest in a global overflow area (LaneStack).  A step pushes
// at most 3 entries per level, so the stack holds at most 3 x (wide-tree
// depth) entries; the launch sizes the overflow area for that.
//
// Triangles use the watertight test of Woop, Benthin and Wald (JCGT 2(1),
// 2013): shared edges and vertices of a closed mesh let no ray through.  The
// edge functions are evaluated without contraction (so the two triangles of
// an edge compute exactly negated values) with an FP64 fallback when one is 0.
// Closest hit: smallest t; an exact tie goes to the lower global primitive id,
// so the result does not depend on traversal order.
//
// Two-level scenes (TL): the top level's leaves are instances.  Entering one
// pushes the world ray (6 words) and a marker on the lane's stack,
// transforms the ray into the instance's object space (the 3x4
// world-to-object rows; the direction is not normalised, so t keeps its
// meaning) and continues at the instance's bottom-level root; popping the
// marker pops the world ray back.  A lane leaves an instance only with no
// leaf parked, and parks no leaf at the top level, so a parked leaf is
// always tested with the ray of its own instance.  Hits keep the instance
// and the primitive index within its mesh; exact ties go to the lower
// (instance, primitive), the order of the global primitive ids.
#pragma once

#include "rtx_internal.h"

namespace rtx {

// The slab test's distances are in units of the ray's t, clamped by a maximum
// with tmin and a minimum with the best hit, so any tmin and tmax will do.
// kBoxPad: the far distance is moved out by 2^-18 of itself, where the
// roundings of an entry and an exit distance are together within 2^-20 of the
// distance (the planes' own margin covers what is relative to their distance
// from the node's origin, node.h).  Distances relative to the best hit, whose
// FMAs the clamp to [0, 1] limits for nothing, save eight instructions a visit
// but gave 0 to 1 % (3 % on a 400x225 frame of 10 samples), and hold neither
// for a negative tmin nor, with tmin within them, where tmin is close to the hit.
constexpr float kBoxPad = 0x1p-18f;

struct TRay {
    float3 o, d;
    float3 idir;    // 1 / d, limited (tray_init)
    float tmin;
    // the watertight test's axis order (kx, ky, kz) as a rotation that puts
    // the dominant axis kz last (rz0: kz = x, rz1: kz = y, else kz = z).
    // Woop et al. (2013) also swap kx and ky when d[kz] < 0 to keep the
    // winding; that negates U, V, W, det and T alike and leaves t, u, v bit
    // for bit the same, and nothing here depends on the winding
    bool rz0, rz1;
    float Sx, Sy, Sz;
    // byte offsets, inside a 4-wide node, of each axis's planes in the order
    // the ray meets them: entry planes, then exit planes
    uint32_t nx, ny, nz;
};


// (a[kx], a[ky], a[kz]) with selects only (no per-lane branches)
__device__ __forceinline__ float3 permute(const TRay& r, float3 a) {
    const float p = r.rz0 ? a.y : (r.rz1 ? a.z : a.x);
    const float q = r.rz0 ? a.z : (r.rz1 ? a.x : a.y);
    const float w = r.rz0 ? a.x : (r.rz1 ? a.y : a.z);
    return f3(p, q, w);
}

__device__ __forceinline__ void tray_init(TRay& r, float3 o, float3 d, float tmin) {
    r.o = o;
    r.d = d;
    r.tmin = tmin;
    const float ax = fabsf(d.x), ay = fabsf(d.y), az = fabsf(d.z);
    const int kz = (ax >= ay && ax >= az) ? 0 : (ay >= az ? 1 : 2);
    const float dz = kz == 0 ? d.x : (kz == 1 ? d.y : d.z);
    r.rz0 = kz == 0;
    r.rz1 = kz == 1;
    const float3 dp = permute(r, d);       // (d[kx], d[ky], d[kz])
    const float3 q = f3(1.f / d.x, 1.f / d.y, 1.f / d.z);
    r.Sz = r.rz0 ? q.x : (r.rz1 ? q.y : q.z);
    // A component 2^72 times smaller than the largest is taken as that much
    // smaller, so that a zero or subnormal one gives finite distances: boxes
    // hold the ray's points to within 2^-42 of their size (node.h).  (Between
    // 2^40 and 2^72 for short directions, so that distances along it stay in range.)
    const float aS = fabsf(r.Sz);
    const float lim = __builtin_amdgcn_fmed3f(aS * 0x1p40f, aS * 0x1p72f, 1e30f);
    r.idir = f3(__builtin_amdgcn_fmed3f(q.x, -lim, lim), __builtin_amdgcn_fmed3f(q.y, -lim, lim),
                __builtin_amdgcn_fmed3f(q.z, -lim, lim));
    r.Sx = dp.x * r.Sz;                     // shear by the reciprocal: no division of its own
    r.Sy = dp.y * r.Sz;
    r.nx = kNodePlanes[0] + (r.idir.x >= 0.f ? 0u : 8u);
    r.ny = kNodePlanes[1] + (r.idir.y >= 0.f ? 0u : 8u);
    r.nz = kNodePlanes[2] + (r.idir.z >= 0.f ? 0u : 8u);
}

// true with t > tmin and barycentrics (u,v) of v1 and v2 on a hit
__device__ __forceinline__ bool watertight(const TRay& r, float3 v0, float3 v1, float3 v2, float& t, float& u,
                                           float& v) {
#pragma clang fp contract(off)
    const float Ax0 = v0.x - r.o.x, Ay0 = v0.y - r.o.y, Az0 = v0.z - r.o.z;
    const float Bx0 = v1.x - r.o.x, By0 = v1.y - r.o.y, Bz0 = v1.z - r.o.z;
    const float Cx0 = v2.x - r.o.x, Cy0 = v2.y - r.o.y, Cz0 = v2.z - r.o.z;
    const float3 A = permute(r, f3(Ax0, Ay0, Az0)), B = permute(r, f3(Bx0, By0, Bz0)),
                 C = permute(r, f3(Cx0, Cy0, Cz0));
    const float Akz = A.z, Bkz = B.z, Ckz = C.z;
    const float Ax = A.x - r.Sx * Akz, Ay = A.y - r.Sy * Akz;
    const float Bx = B.x - r.Sx * Bkz, By = B.y - r.Sy * Bkz;
    const float Cx = C.x - r.Sx * Ckz, Cy = C.y - r.Sy * Ckz;
    float U = Cx * By - Cy * Bx;
    float V = Ax * Cy - Ay * Cx;
    float W = Bx * Ay - By * Ax;
    if (U == 0.f || V == 0.f || W == 0.f) {
        U = (float)((double)Cx * (double)By - (double)Cy * (double)Bx);
        V = (float)((double)Ax * (double)Cy - (double)Ay * (double)Cx);
        W = (float)((double)Bx * (double)Ay - (double)By * (double)Ax);
    }
    if ((U < 0.f || V < 0.f || W < 0.f) && (U > 0.f || V > 0.f || W > 0.f)) return false;
    const float det = U + V + W;
    if (det == 0.f) return false;
    const float Az = r.Sz * Akz, Bz = r.Sz * Bkz, Cz = r.Sz * Ckz;
    const float T = U * Az + V * Bz + W * Cz;
    const float rcp = 1.f / det;
    t = T * rcp;
    if (!(t > r.tmin)) return false;
    u = V * rcp;
    v = W * rcp;
    return true;
}

// LDS addresses as such (address space 3), so that stack accesses compile to
// ds_read/ds_write instead of flat loads through a generic pointer
typedef __attribute__((address_space(3))) uint32_t lds_u32;
typedef __attribute__((address_space(3))) float4 lds_f4;
typedef __attribute__((address_space(3))) const rtx_f4v lds_f4v;
__device__ __forceinline__ float4 lld4(const char __attribute__((address_space(3)))* p) {
    const rtx_f4v v = *(lds_f4v*)p;
    return make_float4(v.x, v.y, v.z, v.w);
}

// an axis's planes of a node (16 B at a multiple of 8) as halves
typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float rtx_f4a8 __attribute__((ext_vector_type(4), aligned(8)));
template <bool G>
__device__ __forceinline__ half8 ld_planes(const char* p) {
    if constexpr (G) return __builtin_bit_cast(half8, (rtx_f4v)*(const RTX_GLOBAL rtx_f4a8*)p);
    else return __builtin_bit_cast(half8, (rtx_f4v)*(const rtx_f4a8*)p);
}
__device__ __forceinline__ half8 lld_planes(const char __attribute__((address_space(3)))* p) {
    return __builtin_bit_cast(half8, (rtx_f4v)*(const rtx_f4a8 __attribute__((address_space(3)))*)p);
}

// the address of an LDS pointer
__device__ __forceinline__ uint32_t lds_addr(const lds_u32* p) { return (uint32_t)(uintptr_t)p; }

// The traversal stack of a lane: a column of SLDS + 1 LDS slots, BLOCK words
// apart, and an overflow column in global memory.  Slot 0 holds kNoChild for
// good, entry i >= 1 is slot i, and the entries above SLDS are in global
// memory.  The stack pointer is the LDS address of the top slot (past the
// column once the top entry is in global memory; only its slot number is used
// then), so a push or pop in LDS needs no address arithmetic beyond moving the
// pointer, and popping an empty stack gives kNoChild without a test.
template <int BLOCK, int SLDS = kStackLDS>
struct LaneStack {
    static constexpr uint32_t kRowBytes = 4u * BLOCK;
    lds_u32* bottom;   // slot 0 of this lane: the pointer of the empty stack
    uint32_t fast;     // with the pointer at or below this, three pushes stay in LDS
    uint32_t* glob;    // overflow column: slot i at glob[(i - SLDS - 1) * gstride]
    uint32_t gstride;
    // s_stack: (SLDS + 1) * BLOCK words of LDS
    __device__ __forceinline__ void init(uint32_t* s_stack, uint32_t* glob_column, uint32_t stride) {
        lds_u32* row0 = (lds_u32*)s_stack;
        bottom = row0 + threadIdx.x;
        fast = lds_addr(row0) + (SLDS - 3) * kRowBytes + (kRowBytes - 1u);
        glob = glob_column;
        gstride = stride;
        *bottom = kNoChild;
    }
    __device__ __forceinline__ uint32_t slot(const lds_u32* sp) const {
        return (lds_addr(sp) - lds_addr(bottom)) / kRowBytes;
    }
    // whether slot sp is in LDS
    __device__ __forceinline__ bool in_lds(const lds_u32* sp) const { return lds_addr(sp) <= fast + 3u * kRowBytes; }
    __device__ __forceinline__ void put(lds_u32* sp, uint32_t v) {
        if (in_lds(sp)) *sp = v;
        else glob[(size_t)(slot(sp) - SLDS - 1) * gstride] = v;
    }
    // the entry at sp (the top one; kNoChild at the bottom)
    __device__ __forceinline__ uint32_t peek(const lds_u32* sp) const {
        if (in_lds(sp)) return *sp;
        return glob[(size_t)(slot(sp) - SLDS - 1) * gstride];
    }
    __device__ __forceinline__ void push(lds_u32*& sp, uint32_t v) {
        sp += BLOCK;
        put(sp, v);
    }
    __device__ __forceinline__ uint32_t pop(lds_u32*& sp) {
        const uint32_t v = peek(sp);
        sp -= BLOCK;
        return v;
    }
    // pushes v[0..N-1] (v[N-1] ends on top) with one range check when all N
    // slots are in LDS
    template <int N>
    __device__ __forceinline__ void push_n(lds_u32*& sp, const uint32_t (&v)[N]) {
        if (in_lds(sp + N * BLOCK)) {
#pragma unroll
            for (int i = 0; i < N; i++) sp[(i + 1) * BLOCK] = v[i];
            sp += N * BLOCK;
        } else {
#pragma unroll
            for (int i = 0; i < N; i++) push(sp, v[i]);
        }
    }
    // pops N entries into v[0..N-1] (v[N-1] is the old top), the inverse of push_n
    template <int N>
    __device__ __forceinline__ void pop_n(lds_u32*& sp, uint32_t (&v)[N]) {
        if (in_lds(sp)) {
            sp -= N * BLOCK;
#pragma unroll
            for (int i = 0; i < N; i++) v[i] = sp[(i + 1) * BLOCK];
        } else {
#pragma unroll
            for (int i = N - 1; i >= 0; i--) v[i] = pop(sp);
        }
    }
    // One node step: pushes the hit ones of children 1..3 of a sorted 4-wide
    // node (h1..h3; the hit children come first, so h3 implies h2 implies h1),
    // the farthest first, and returns the old top entry.  In LDS every child
    // is written, to the slot above a pointer that moves only past hit ones: a
    // child that is not hit is overwritten by the next or stays above the top.
    __device__ __forceinline__ uint32_t step4(lds_u32*& sp, bool h1, bool h2, bool h3, uint32_t r1, uint32_t r2,
                                              uint32_t r3) {
        lds_u32* a = sp;
        uint32_t top;
        if (lds_addr(a) <= fast) {
            top = *a;
            a[BLOCK] = r3;
            a += h3 ? BLOCK : 0;
            a[BLOCK] = r2;
            a += h2 ? BLOCK : 0;
            a[BLOCK] = r1;
            a += h1 ? BLOCK : 0;
        } else {
            top = peek(a);
            if (h3) push(a, r3);
            if (h2) push(a, r2);
            if (h1) push(a, r1);
        }
        sp = a;
        return top;
    }
};

__device__ __forceinline__ float comp4(const float4& v, int j) {
    return j == 0 ? v.x : (j == 1 ? v.y : (j == 2 ? v.z : v.w));
}

// the distance of a plane, half * ds + c (one v_fma_mix_f32)
__device__ __forceinline__ float slab(_Float16 h, float ds, float c) { return __builtin_fmaf((float)h, ds, c); }

// A child of a node step as one double, the entry distance's bits above the
// ref's: doubles order by their high word first, so one v_min_f64 and one
// v_max_f64 exchange a pair where two 32-bit words take a compare and four
// selects, and a 64-bit minimum issues at the rate of a 32-bit one (measured:
// 4.7 against 4.3 clocks per wave and SIMD, 4.4 for a select).  A float's
// infinity, the distance of a child that is not hit, is an ordinary number
// there (exponent 0x7F8), and a distance is never NaN.
__device__ __forceinline__ double child_key(float t, uint32_t ref) {
    return __builtin_bit_cast(double, ((uint64_t)__float_as_uint(t) << 32) | ref);
}
__device__ __forceinline__ uint32_t key_ref(double k) { return (uint32_t)__builtin_bit_cast(uint64_t, k); }
__device__ __forceinline__ bool key_hit(double k) {
    typedef float f2v __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(f2v, k).y < __builtin_inff();
}
// compare-exchange: smaller key first (as instructions, since fmin on doubles
// would quiet its operands first)
__device__ __forceinline__ void sort_ce(double& a, double& b) {
    double lo, hi;
    asm("v_min_f64 %0, %1, %2" : "=v"(lo) : "v"(a), "v"(b));
    asm("v_max_f64 %0, %1, %2" : "=v"(hi) : "v"(a), "v"(b));
    a = lo;
    b = hi;
}

struct HitFull {
    float t, u, v;
    uint32_t tri;    // leaf-ordered triangle, kNoHit on a miss
    uint32_t prim;   // global primitive id (two-level scenes: primitive index within the instance's mesh)
    uint32_t inst;   // instance of the hit (two-level scenes; flat scenes keep it in the triangle)
};

// Resumable traversal state of one ray: the ray, the next node to visit,
// the stack depth and the best hit so far.
struct Trav {
    TRay r;
    HitFull h;
    uint32_t node;    // next node to visit (kNoChild: none left)
    uint32_t leaf;    // a leaf found but not tested yet (kNoChild: none)
    uint32_t leaf2;   // a second one (set only while leaf is)
    lds_u32* sp;      // stack pointer (LaneStack)
    uint32_t inst;    // two-level scenes: the instance the lane is in (kNoHit: top level)
};

__device__ __forceinline__ void trav_reset(Trav& s, const DevScene& sc, lds_u32* bottom, float tmax) {
    s.h.t = tmax;
    s.h.u = s.h.v = 0.f;
    s.h.tri = kNoHit;
    s.h.prim = kNoHit;
    s.h.inst = kNoHit;
    s.node = sc.root;
    s.leaf = kNoChild;
    s.leaf2 = kNoChild;
    s.sp = bottom;
    s.inst = kNoHit;
}

__device__ __forceinline__ void trav_begin(Trav& s, const DevScene& sc, lds_u32* bottom, float3 o, float3 d, float tmin,
                                           float tmax) {
    tray_init(s.r, o, d, tmin);
    trav_reset(s, sc, bottom, tmax);
}

// row . (p, 1) and row . (v, 0) of a 3x4 transform, one rounding per operation
// (the order of the flattening build, so that a two-level scene's world
// vertices are bit for bit those of the flat scene)
__device__ __forceinline__ float xf_point(const float4& row, float3 p) {
    return ((p.x * row.x + p.y * row.y) + p.z * row.z) + row.w;
}
__device__ __forceinline__ float xf_vector(const float4& row, float3 v) {
    return (v.x * row.x + v.y * row.y) + v.z * row.z;
}
// the same products as fused multiply-adds, for the ray an instance entry
// transforms into object space: nothing has to round like the flat scene
// there, and three FMAs per row replace six (five) operations
__device__ __forceinline__ float xf_point_fma(const float4& row, float3 p) {
    return __builtin_fmaf(p.x, row.x, __builtin_fmaf(p.y, row.y, __builtin_fmaf(p.z, row.z, row.w)));
}
__device__ __forceinline__ float xf_vector_fma(const float4& row, float3 v) {
    return __builtin_fmaf(v.x, row.x, __builtin_fmaf(v.y, row.y, v.z * row.z));
}

// two-level scenes: one instance transition of the lanes that call it.  A
// lane with `leave` set has just popped its instance's marker (and has no
// leaf parked): it pops the world ray and the next entry.  A going lane that
// then stands on an instance leaf enters that instance: it pushes the world
// ray and a marker and continues at the instance's bottom-level root with
// the ray in object space.  The lanes that left, entered or both set their
// new ray up together, in one call.
template <bool G, class Stack>
__device__ __forceinline__ void inst_step(const DevScene& sc, Trav& s, bool going, bool leave, Stack& st) {
    float3 o = s.r.o, d = s.r.d;
    if (leave) {
        uint32_t w[6];
        st.pop_n(s.sp, w);
        o = f3(__uint_as_float(w[0]), __uint_as_float(w[1]), __uint_as_float(w[2]));
        d = f3(__uint_as_float(w[3]), __uint_as_float(w[4]), __uint_as_float(w[5]));
        s.inst = kNoHit;
        s.node = st.pop(s.sp);
    }
    const bool enter = going && (s.node & kInstLeaf) == kInstLeaf;
    if (enter) {
        const uint32_t id = s.node & kLeafFirstMask;
        const float4* X = sc.xinst + (size_t)kInstF4 * id;
        const float4 r0 = ld4<G>(X), r1 = ld4<G>(X + 1), r2 = ld4<G>(X + 2), m = ld4<G>(X + 6);
        const uint32_t w[7] = {__float_as_uint(o.x), __float_as_uint(o.y), __float_as_uint(o.z), __float_as_uint(d.x),
                               __float_as_uint(d.y), __float_as_uint(d.z), kInstMarker};
        st.push_n(s.sp, w);
        const float3 wo = o, wd = d;
        o = f3(xf_point_fma(r0, wo), xf_point_fma(r1, wo), xf_point_fma(r2, wo));
        d = f3(xf_vector_fma(r0, wd), xf_vector_fma(r1, wd), xf_vector_fma(r2, wd));
        s.inst = id;
        s.node = __float_as_uint(m.x);
    }
    if (leave || enter) tray_init(s.r, o, d, s.r.tmin);
}

// first active lane of the wave (counts wave-level loop iterations in COUNT mode)
__device__ __forceinline__ bool first_active_lane() {
    const uint64_t e = __builtin_amdgcn_read_exec();
    return (threadIdx.x & 63u) == (uint32_t)(__ffsll((unsigned long long)e) - 1);
}

// LDS words per wave that the compacted leaf phase uses: the owner marks of
// a round (64), the best key per lane (64 x 64 bit) and the lane holding it
// (64)
constexpr uint32_t kLeafScratchWords = 256;
typedef __attribute__((address_space(3))) uint64_t lds_u64;

// orders the LDS accesses of the wave's lanes around it (the lanes of a wave
// run in lockstep and its LDS operations complete in order, so this only
// keeps the compiler from moving them)
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
}

// The leaf phase with the work spread over the wave.  A lane's parked
// leaves hold c = c1 + c2 triangles; the wave's (lane, triangle) pairs are
// numbered by an inclusive prefix sum of c and dealt out 64 at a time, one
// per lane whatever lane parked them.  The lane that tests pair p finds its
// owner (the lane whose pairs hold p) by a max-scan over the wave of the
// round positions that the owners mark in LDS, and reads the owner's ray and
// leaves with ds_bpermute.  A hit goes into the owner's LDS slot as the 64-bit minimum
// of (t, primitive id) -- t > tmin >= 0, so the float's bits order like its
// value; the id is global in a flat scene and within the mesh in a
// two-level one, where all of a lane's parked leaves belong to the instance
// it is in -- and the lane whose key won writes its lane number next
// to it; the owner then takes that hit (t, u, v, triangle) under the rule of
// the per-lane loop: closer, or as close with the lower id.  The minimum of
// (t, id) does not depend on the order of the tests, so the closest hit is
// the one the lane would have found testing its own leaves in order.
// Needs all 64 lanes of the wave in the call (the pairs of an inactive lane
// would never be tested), and a ray with tmin >= 0.  A pair is tested only
// if it lies in its owner's own leaves (q < the owner's count), and read
// from the owner's triangle array, so every triangle read is one the owner
// parked.
// max(v, v of the lane that the DPP control CTRL names); lanes outside the
// rows of ROW_MASK, or without a source lane in their row, keep v
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ uint32_t max_dpp(uint32_t v) {
    const uint32_t t = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROW_MASK, 0xf, false);
    return v > t ? v : t;
}

// v + v of the lane that the DPP control CTRL names (0 where max_dpp keeps v)
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ uint32_t add_dpp(uint32_t v) {
    return v + (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROW_MASK, 0xf, false);
}

template <bool G, bool TL, bool COUNT>
__device__ __forceinline__ void leaves_compact(const DevScene& sc, Trav& s, uint32_t f1, uint32_t c1, uint32_t f2,
                                               uint32_t c2, lds_u32* cl, uint32_t* wi) {
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t c = c1 + c2;
    // inclusive prefix sum of c over the wave (DPP, as the owner scan below)
    uint32_t incl = c;
    incl = add_dpp<0x111, 0xf>(incl);   // row_shr:1
    incl = add_dpp<0x112, 0xf>(incl);   // row_shr:2
    incl = add_dpp<0x114, 0xf>(incl);   // row_shr:4
    incl = add_dpp<0x118, 0xf>(incl);   // row_shr:8
    incl = add_dpp<0x142, 0xa>(incl);   // row_bcast:15 into rows 1 and 3
    incl = add_dpp<0x143, 0xc>(incl);   // row_bcast:31 into rows 2 and 3
    const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
    if (total == 0) return;
    const uint32_t excl = incl - c;
    lds_u32* M = cl;
    lds_u64* K = (lds_u64*)(cl + 64);
    lds_u32* Wn = cl + 192;
    K[lane] = ~0ull;
    // what a helper lane needs of the owner: its ray (object space inside an
    // instance), the first pair's number, and its leaves
    const uint32_t meta = excl | (c1 << 16) | (c << 21) | (s.r.rz0 ? 1u << 30 : 0u) | (s.r.rz1 ? 1u << 31 : 0u);
    wave_sync();
    for (uint32_t base = 0; base < total; base += 64u) {
        if (COUNT && lane == 0) wi[1]++;
        const uint32_t p = base + lane;
        const bool has = p < total;
        // owner: the lane whose pairs [excl, incl) hold p.  Each lane whose
        // pairs meet this round marks the round position of its first one
        // with its lane number; the owner of position j is then the largest
        // mark at or before j (lane numbers grow with the pair numbers), an
        // inclusive max-scan over the wave (DPP: shifts within the 16-lane
        // rows, then broadcasts of the row ends to the rows above)
        M[lane] = 0u;
        wave_sync();
        if (c != 0u && incl > base && excl < base + 64u) M[(excl > base ? excl : base) - base] = lane;
        wave_sync();
        uint32_t i = M[lane];
        i = max_dpp<0x111, 0xf>(i);   // row_shr:1
        i = max_dpp<0x112, 0xf>(i);   // row_shr:2
        i = max_dpp<0x114, 0xf>(i);   // row_shr:4
        i = max_dpp<0x118, 0xf>(i);   // row_shr:8
        i = max_dpp<0x142, 0xa>(i);   // row_bcast:15 into rows 1 and 3
        i = max_dpp<0x143, 0xc>(i);   // row_bcast:31 into rows 2 and 3
        const int ad = (int)(i << 2);
        auto bp = [&](uint32_t v) -> uint32_t { return (uint32_t)__builtin_amdgcn_ds_bpermute(ad, (int)v); };
        auto bpf = [&](float v) -> float { return __uint_as_float(bp(__float_as_uint(v))); };
        TRay hr;
        hr.o = f3(bpf(s.r.o.x), bpf(s.r.o.y), bpf(s.r.o.z));
        hr.Sx = bpf(s.r.Sx);
        hr.Sy = bpf(s.r.Sy);
        hr.Sz = bpf(s.r.Sz);
        hr.tmin = bpf(s.r.tmin);
        const uint32_t om = bp(meta), of1 = bp(f1), of2 = bp(f2);
        hr.rz0 = (om >> 30) & 1u;
        hr.rz1 = (om >> 31) & 1u;
        const uint32_t q = p - (om & 0xFFFFu), oc1 = (om >> 16) & 31u, oc = (om >> 21) & 63u;
        const uint32_t k = q < oc1 ? of1 + q : of2 + (q - oc1);
        float tt = 0.f, uu = 0.f, vv = 0.f;
        bool hit = false;
        uint64_t key = ~0ull;
        // the owner's triangle array: in a batch (G) each lane renders its
        // own job, so the owner's scene need not be this lane's
        const char* tb = (const char*)sc.tris;
        if (G) {
            const uint64_t pt = (uint64_t)sc.tris;
            tb = (const char*)(((uint64_t)bp((uint32_t)(pt >> 32)) << 32) | (uint64_t)bp((uint32_t)pt));
        }
        if (has && q < oc) {
            const uint32_t to = k * 48u;
            typedef const float4 cf4t;
            const float4 t0 = ld4<G>((cf4t*)(tb + to)), t1 = ld4<G>((cf4t*)(tb + (to + 16u))),
                         t2 = ld4<G>((cf4t*)(tb + (to + 32u)));
            hit = watertight(hr, xyz(t0), xyz(t1), xyz(t2), tt, uu, vv);
            if (hit) {
                key = ((uint64_t)__float_as_uint(tt) << 32) | (uint64_t)__float_as_uint(t0.w);
                __hip_atomic_fetch_min(K + i, key, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
            }
        }
        wave_sync();
        if (hit && K[i] == key) Wn[i] = lane;
        wave_sync();
        // the owners of this round's pairs take their best hit
        const uint64_t kk = K[lane];
        const int wa = (int)((Wn[lane] & 63u) << 2);
        const float bu = __uint_as_float((uint32_t)__builtin_amdgcn_ds_bpermute(wa, (int)__float_as_uint(uu)));
        const float bv = __uint_as_float((uint32_t)__builtin_amdgcn_ds_bpermute(wa, (int)__float_as_uint(vv)));
        const uint32_t bk = (uint32_t)__builtin_amdgcn_ds_bpermute(wa, (int)k);
        // (a slot holds a key only if its lane owned a pair of this round
        // that hit: every slot is reset when it is taken)
        if (kk != ~0ull) {
            const float t = __uint_as_float((uint32_t)(kk >> 32));
            const uint32_t prim = (uint32_t)kk;
            const bool lower = TL ? (s.inst < s.h.inst || (s.inst == s.h.inst && prim < s.h.prim)) : prim < s.h.prim;
            if (t < s.h.t || (t == s.h.t && lower)) {
                s.h.t = t;
                s.h.u = bu;
                s.h.v = bv;
                s.h.tri = bk;
                s.h.prim = prim;
                if (TL) s.h.inst = s.inst;
            }
            K[lane] = ~0ull;
        }
        wave_sync();
    }
}

// Advances the traversal of the lanes with `going` set.  A lane clears
// `going` when its ray is done (closest hit final in s.h).
//
// Each round has a node phase and a leaf phase.  The node phase steps the
// lanes that sit on an inner node; a lane that reaches a leaf parks it in
// one of two leaf slots and goes on with the next node from its stack (Aila
// and Laine 2009, "speculative traversal"), and waits only when it reaches a
// third leaf or runs out of nodes.  The phase ends when fewer than
// inner_frac/64 of the going lanes can still step; the leaf phase then tests
// the parked leaves of all lanes together.  inner_frac = 1 runs the node
// phase until no lane can step.  The function
// returns once no lane is going, or -- with `batch` < 64 -- as soon as at
// least `batch` of the wave's `busy` lanes have finished, so that the caller
// can shade them while the others keep their state and resume later.
// COUNT adds node-visit and triangle-test counts (statistics launches only).
// TOPN > 0: the first TOPN nodes of the node array (the top levels: the
// array is breadth-first) are read from a copy in LDS at `top` instead of
// global memory.
// CL: the leaf phase spreads the parked leaves' triangles over the wave
// (leaves_compact, with the wave's kLeafScratchWords of LDS at `cl`);
// otherwise each lane tests its own leaves.
// NN: the lane's node visits are counted in *nn (COUNT: so are more).
template <int BLOCK, bool COUNT = false, bool TL = false, bool G = false, int TOPN = 0, bool CL = false,
          bool NN = false, class Stack>
__device__ __forceinline__ void trav_run(const DevScene& sc, Trav& s, bool& going, bool busy, int batch,
                                         int inner_frac, Stack& st, uint32_t* nn = nullptr,
                                         uint32_t* nt = nullptr, uint32_t* wi = nullptr,
                                         const lds_f4* top = nullptr, lds_u32* cl = nullptr) {
    if (going && s.node == kEmptyRoot) going = false;
    for (;;) {
        // node phase (no lane starts or stops going in it)
        const uint64_t m_going = __ballot(going);
        const uint32_t n_going = (uint32_t)__popcll(m_going);
        // (one scalar condition ends the loop and guards its step, and the step
        // is a block at its end: the loop's branch is then a scalar one, with
        // no mask of lanes that left; 2 % on every frame)
        const uint32_t least = n_going ? ((uint32_t)inner_frac * n_going + 63u) >> 6 : 1u;
        bool step;
        do {
            if (TL) {
                // Instance transitions: leave a finished instance (not while
                // one of its leaves is parked), then enter the instance the
                // lane stands on, if any.  A transition costs several node
                // steps of instructions, so a lane that needs one waits
                // (without stepping) until kTlFrac/64 of the going lanes do,
                // or until the round's transition step after the leaf phase.
                const bool leave = going && s.node == kInstMarker && s.leaf == kNoChild;
                const bool enter = going && (s.node & kInstLeaf) == kInstLeaf;
                const uint64_t need = __ballot(leave || enter);
                if (need && (uint32_t)__popcll(need) * 64u >= (uint32_t)kTlFrac * n_going)
                    inst_step<G>(sc, s, going, leave, st);
            }
            // a lane that reached a leaf parks it (two slots) and goes on
            // with the next node from its stack, so it keeps stepping while
            // the others do; the parked leaves are tested together below
            // (an instance leaf waits for its transition instead)
            if (going && (s.node & kLeafFlag) && (!TL || (s.node & kInstLeaf) != kInstLeaf) &&
                (s.leaf == kNoChild || s.leaf2 == kNoChild)) {
                if (s.leaf == kNoChild) s.leaf = s.node;
                else s.leaf2 = s.node;
                s.node = st.pop(s.sp);
            }
            // no leaf flag, not kNoChild (nor the instance marker): one unsigned
            // compare, balloted as it is and masked with the going lanes
            const bool below = s.node < (TL ? kInstMarker : kNoChild);
            const bool inner = going && below;
            const uint32_t n_inner = (uint32_t)__popcll(__ballot(below) & m_going);
            step = n_inner >= least;
            if (inner && step) {
                if (COUNT || NN) (*nn)++;
                if (COUNT && first_active_lane()) wi[0]++;
                // one 4-wide node: five loads.  The ray reads each axis's
                // entry and exit planes by its direction signs, so the slab
                // test needs no min/max per axis; the halves go into the FMAs
                // as they are (v_fma_mix_f32).
                // (32-bit byte offsets: the builder keeps the node array below 4 GiB)
                const uint32_t no = s.node * (16u * kWideNodeF4);
                const TRay& r = s.r;
                half8 px, py, pz;
                float4 og, rf;
                if (TOPN > 0 && s.node < (uint32_t)TOPN) {
                    typedef const char __attribute__((address_space(3))) lchar;
                    lchar* lb = (lchar*)top;
                    px = lld_planes(lb + (no + r.nx));
                    py = lld_planes(lb + (no + r.ny));
                    pz = lld_planes(lb + (no + r.nz));
                    og = lld4(lb + (no + 16u * kNodeOrigin));
                    rf = lld4(lb + (no + 16u * kNodeRefs));
                } else {
                    typedef const float4 cf4;
                    const char* nb = (const char*)sc.nodes;
                    px = ld_planes<G>(nb + (no + r.nx));
                    py = ld_planes<G>(nb + (no + r.ny));
                    pz = ld_planes<G>(nb + (no + r.nz));
                    og = ld4<G>((cf4*)(nb + (no + 16u * kNodeOrigin)));
                    rf = ld4<G>((cf4*)(nb + (no + 16u * kNodeRefs)));
                }
                // all five in flight before the first is waited for (the
                // compiler would hold some back to reuse registers: the
                // 1080p mixed-level frame 109 ms without, 102 ms with)
                __builtin_amdgcn_sched_barrier(0);
                const float3 ds = f3(og.w * r.idir.x, og.w * r.idir.y, og.w * r.idir.z);
                const float3 oo = f3(og.x - r.o.x, og.y - r.o.y, og.z - r.o.z);
                double key[4];
                const float3 c = f3(oo.x * r.idir.x, oo.y * r.idir.y, oo.z * r.idir.z);
    #pragma unroll
                for (int j = 0; j < 4; j++) {
                    const float x0 = slab(px[j], ds.x, c.x), x1 = slab(px[4 + j], ds.x, c.x);
                    const float y0 = slab(py[j], ds.y, c.y), y1 = slab(py[4 + j], ds.y, c.y);
                    const float z0 = slab(pz[j], ds.z, c.z), z1 = slab(pz[4 + j], ds.z, c.z);
                    const float tn = fmaxf(fmaxf(x0, y0), fmaxf(z0, r.tmin));
                    const float tf = fminf(fminf(x1, y1), fminf(z1, s.h.t));
                    const bool hit = tn <= __builtin_fmaf(fabsf(tf), kBoxPad, tf);   // (tf may be negative)
                    key[j] = child_key(hit ? tn : __builtin_inff(), __float_as_uint(comp4(rf, j)));
                }
                // ascending by entry distance (misses last): 5 compare-exchanges
                sort_ce(key[0], key[1]);
                sort_ce(key[2], key[3]);
                sort_ce(key[0], key[2]);
                sort_ce(key[1], key[3]);
                sort_ce(key[1], key[2]);
                // visit the nearest; push the others farthest first, so the
                // next nearest is on top.  With no hit the top of the stack
                // (kNoChild when it is empty) is next.
                const uint32_t top = st.step4(s.sp, key_hit(key[1]), key_hit(key[2]), key_hit(key[3]),
                                              key_ref(key[1]), key_ref(key[2]), key_ref(key[3]));
                const bool any = key_hit(key[0]);
                s.node = any ? key_ref(key[0]) : top;
                s.sp -= any ? 0 : BLOCK;
            }
        } while (step);
        // leaf phase (compacted when the whole wave is here)
        if (CL && __builtin_amdgcn_read_exec() == ~0ull) {
            uint32_t f1 = 0, c1 = 0, f2 = 0, c2 = 0;
            if (going && s.leaf != kNoChild) {
                f1 = s.leaf & kLeafFirstMask;
                c1 = ((s.leaf >> kLeafCountShift) & 15u) + 1u;
                if (s.leaf2 != kNoChild) {
                    f2 = s.leaf2 & kLeafFirstMask;
                    c2 = ((s.leaf2 >> kLeafCountShift) & 15u) + 1u;
                }
                s.leaf = kNoChild;
                s.leaf2 = kNoChild;
            }
            if (COUNT) *nt += c1 + c2;
            leaves_compact<G, TL, COUNT>(sc, s, f1, c1, f2, c2, cl, wi);
        } else if (going && s.leaf != kNoChild) {
            const uint32_t lf = s.leaf;
            s.leaf = kNoChild;
            const uint32_t first = lf & kLeafFirstMask;
            const uint32_t cnt = ((lf >> kLeafCountShift) & 15u) + 1u;
            const uint32_t lf2 = s.leaf2;
            s.leaf2 = kNoChild;
            const uint32_t first2 = lf2 & kLeafFirstMask;
            const uint32_t cnt2 = lf2 == kNoChild ? 0u : ((lf2 >> kLeafCountShift) & 15u) + 1u;
            if (COUNT) *nt += cnt + cnt2;
            // the triangles of both parked leaves in one loop
            for (uint32_t q = 0; q < cnt + cnt2; q++) {
                const uint32_t k = q < cnt ? first + q : first2 + (q - cnt);
                if (COUNT && first_active_lane()) wi[1]++;
                // (32-bit byte offsets: the builder keeps the triangle array below 4 GiB)
                const char* tb = (const char*)sc.tris;
                const uint32_t to = k * 48u;
                typedef const float4 cf4t;
                const float4 t0 = ld4<G>((cf4t*)(tb + to)), t1 = ld4<G>((cf4t*)(tb + (to + 16u))),
                             t2 = ld4<G>((cf4t*)(tb + (to + 32u)));
                float tt, uu, vv;
                if (watertight(s.r, xyz(t0), xyz(t1), xyz(t2), tt, uu, vv)) {
                    const uint32_t prim = __float_as_uint(t0.w);
                    const bool lower = TL ? (s.inst < s.h.inst || (s.inst == s.h.inst && prim < s.h.prim))
                                          : prim < s.h.prim;
                    if (tt < s.h.t || (tt == s.h.t && lower)) {
                        s.h.t = tt;
                        s.h.u = uu;
                        s.h.v = vv;
                        s.h.tri = k;
                        s.h.prim = prim;
                        if (TL) s.h.inst = s.inst;
                    }
                }
            }
        }
        if (TL) {
            // the round's transition step: every lane waiting for one (no
            // leaf is parked after the leaf phase)
            const bool leave = going && s.node == kInstMarker;
            const bool enter = going && (s.node & kInstLeaf) == kInstLeaf;
            if (__ballot(leave || enter)) inst_step<G>(sc, s, going, leave, st);
        }
        if (going && s.node == kNoChild && s.leaf == kNoChild) going = false;
        const uint64_t g = __ballot(going);
        if (g == 0) return;
        if (batch < 64 && __popcll(__ballot(busy && !going)) >= batch) return;
    }
}

// closest hit, run to completion (query kernels and the picker)
template <int BLOCK, bool TL = false, class Stack>
__device__ __forceinline__ void traverse(const DevScene& sc, const TRay& r, float tmax, HitFull& h, Stack& st) {
    Trav s;
    s.r = r;
    trav_reset(s, sc, st.bottom, tmax);
    bool going = true;
    trav_run<BLOCK, false, TL>(sc, s, going, true, 64, 32, st);
    h = s.h;
}

}  // namespace rtx
