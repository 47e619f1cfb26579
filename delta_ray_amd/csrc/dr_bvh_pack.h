// Packing of BVH nodes for ray walks (DrPackedNode).
#pragma once

#include "dr_math.h"
#include "dr_types.h"

// The grid over the root's box: 16-bit coordinate q = (v - lo) * scale + 2, so
// that the box spans 2 .. 65533 and rounding outward stays within 16 bits.
// Axes without extent get a thousandth of the largest one's.
struct BvhGrid {
    float lo[3], scale[3], rscale[3];
};
DR_INLINE BvhGrid bvh_grid(const DrNode &root) {
    const float l[2][3] = {{root.a[0], root.a[1], root.a[2]}, {root.b[2], root.b[3], root.c[0]}};
    const float h[2][3] = {{root.a[3], root.b[0], root.b[1]}, {root.c[1], root.c[2], root.c[3]}};
    BvhGrid g;
    float ext[3], most = 0.f;
    for (int k = 0; k < 3; k++) {
        g.lo[k] = fminf(l[0][k], l[1][k]);
        ext[k] = fmaxf(h[0][k], h[1][k]) - g.lo[k];
        most = fmaxf(most, ext[k]);
    }
    for (int k = 0; k < 3; k++) {
        float e = fmaxf(fmaxf(ext[k], 1e-3f * most), 1e-18f);
        g.scale[k] = fminf(65531.f / e, 1e20f);
        g.rscale[k] = 1.f / g.scale[k];
    }
    return g;
}
// a lower / upper plane on the grid, at least one step outward (not-a-number:
// the grid's end); an empty slot (lo = +inf, hi = -inf) stays empty
DR_INLINE uint32_t pack_lo(float v, float lo, float scale) {
    float q = (v - lo) * scale + 2.f;
    if (!(q >= 1.f)) return 0u;
    return q >= 65536.f ? 65535u : (uint32_t)(floorf(q) - 1.f);
}
DR_INLINE uint32_t pack_hi(float v, float lo, float scale) {
    float q = (v - lo) * scale + 2.f;
    if (!(q <= 65534.f)) return 65535u;
    return q <= -1.f ? 0u : (uint32_t)(ceilf(q) + 1.f);
}
DR_INLINE DrPackedNode pack_node(const DrNode &n, const BvhGrid &g) {
    const float l[2][3] = {{n.a[0], n.a[1], n.a[2]}, {n.b[2], n.b[3], n.c[0]}};
    const float h[2][3] = {{n.a[3], n.b[0], n.b[1]}, {n.c[1], n.c[2], n.c[3]}};
    DrPackedNode p;
    for (int k = 0; k < 3; k++) {
        p.w[k] = pack_lo(l[0][k], g.lo[k], g.scale[k]) | pack_lo(l[1][k], g.lo[k], g.scale[k]) << 16;
        p.w[3 + k] = pack_hi(h[0][k], g.lo[k], g.scale[k]) | pack_hi(h[1][k], g.lo[k], g.scale[k]) << 16;
    }
    for (int c = 0; c < 2; c++)
        p.w[6 + c] = (uint32_t)(n.d[2 + c] > 0 ? ~(2 * n.d[c] + (n.d[2 + c] - 1)) : n.d[c]);
    return p;
}
// element `i` of the head: the grid's nine floats
DR_INLINE DrPackedNode pack_head(const BvhGrid &g, int i) {
    const float f[16] = {g.lo[0], g.lo[1], g.lo[2], g.scale[0], g.scale[1], g.scale[2], g.rscale[0], g.rscale[1],
                         g.rscale[2], 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    DrPackedNode p;
    for (int k = 0; k < 8; k++) p.w[k] = __float_as_uint(f[8 * i + k]);
    return p;
}
