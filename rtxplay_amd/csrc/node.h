// node.h -- writing a 4-wide node (layout in rtx_internal.h).
//
// The traversal is bound by the vector L1 cache, which serves one distinct
// line per clock and CU whatever a lane reads of it (measured: 64 clocks for
// one load instruction of 64 lanes on 64 lines, from 4 to 16 B per lane), and
// the lanes of a wave are on different nodes: a visit costs one access per
// load.  With float planes that was seven (six plane vectors and the refs:
// 0.97 accesses per clock and CU on the 1080p level-6 frame); with the planes
// of an axis in halves, entry and exit side by side, it is five.  Byte planes
// (four loads) were slower: a node that holds the ground and some small things
// has a quantum of 1/255 of the ground, up to 20 % more visits.  Halves are
// finest around the node's origin, which is put at the smallest child.
//
// Rounding is outwards: a plane at p is stored at or beyond p moved out by
// 2^-20 of its distance from the origin, in exact arithmetic.  That margin
// covers the rounding of the traversal's (origin - o) * idir where it cancels
// against half * (scale * idir) (up to 2^-22 of that distance); the
// error relative to the distance itself is covered by kBoxPad in
// traverse.h.  The origin lies a little below the smallest child's lo plane,
// so that no plane of a box is at distance 0 of it and a ray that runs within
// a face of a box (parallel to an axis, through vertices) still meets the box.
#pragma once

#include "rtx_internal.h"

namespace rtx {

// the half (as bits) at or below v, at or above v
__device__ inline uint32_t half_down(double v) {
    uint32_t b = __builtin_bit_cast(uint16_t, (_Float16)(float)v);
    while ((double)__builtin_bit_cast(_Float16, (uint16_t)b) > v)
        b = b == 0u ? 0x8001u : (b & 0x8000u ? b + 1u : b - 1u);
    return b;
}
__device__ inline uint32_t half_up(double v) { return half_down(-v) ^ 0x8000u; }

// The scale of a node whose planes are `reach` from its origin at most: they
// fill 2^15 of the halves' 2^16 range.  (Each node has its own, beside its
// origin: with one scale for a scene a refit that moved things 32 times as far
// apart had infinite planes, and geometry below 2^-35 of the extent had one
// plane step for a whole subtree.)
__device__ inline float node_scale(double reach) {
    int e = 0;
    (void)frexp(reach, &e);
    return ldexpf(1.f, max(e - 15, -126));
}

// lo, hi: the children's boxes; used: which slots hold one
__device__ inline void encode_node(float4* o, const float (&lo)[4][3], const float (&hi)[4][3], const bool (&used)[4],
                                   const uint32_t (&ref)[4]) {
    float org[3] = {0.f, 0.f, 0.f};
    uint2* w = (uint2*)o;
    double reach = 0.0;
    for (int a = 0; a < 3; a++) {
        float least = __builtin_inff();
        float mn = __builtin_inff(), mx = -__builtin_inff();
        for (int k = 0; k < 4; k++) {
            if (!used[k]) continue;
            const float e = hi[k][a] - lo[k][a];
            mn = fminf(mn, lo[k][a]);
            mx = fmaxf(mx, hi[k][a]);
            if (e < least) {
                least = e;
                org[a] = lo[k][a];
            }
        }
        if (mx >= mn && mx - mn < 1e37f) org[a] -= fabsf(org[a]) * 0x1p-21f + (mx - mn) * 0x1p-22f + 1e-36f;
        for (int k = 0; k < 4; k++) {
            if (!used[k]) continue;
            // (infinite planes are infinite halves at any scale)
            const double l = fabs((double)lo[k][a] - (double)org[a]), h = fabs((double)hi[k][a] - (double)org[a]);
            if (l < 1e39) reach = fmax(reach, l);
            if (h < 1e39) reach = fmax(reach, h);
        }
    }
    const float scale = node_scale(reach);
    const double inv = 1.0 / (double)scale;
    for (int a = 0; a < 3; a++) {
        const double O = (double)org[a];
        uint32_t bl[4], bh[4];
        for (int k = 0; k < 4; k++) {
            const double l = (double)lo[k][a] - O, h = (double)hi[k][a] - O;
            bl[k] = used[k] ? half_down((l - fabs(l) * 0x1p-20) * inv) : 0x7C00u;
            bh[k] = used[k] ? half_up((h + fabs(h) * 0x1p-20) * inv) : 0xFC00u;
        }
        const uint2 L = make_uint2(bl[0] | (bl[1] << 16), bl[2] | (bl[3] << 16));
        uint2* p = w + kNodePlanes[a] / 8u;
        p[0] = L;
        p[1] = make_uint2(bh[0] | (bh[1] << 16), bh[2] | (bh[3] << 16));
        p[2] = L;
    }
    o[kNodeOrigin] = make_float4(org[0], org[1], org[2], scale);
    o[kNodeRefs] = make_float4(__uint_as_float(ref[0]), __uint_as_float(ref[1]), __uint_as_float(ref[2]),
                               __uint_as_float(ref[3]));
}

}  // namespace rtx
