// Packing of BVH nodes for ray walks (DrPackedNode).
#pragma once

#include "dr_math.h"
#include "dr_types.h"

// One axis of a node's frame: planes at origin + q * step, q = 0 .. 255, with the
// origin below the boxes and a positive step, or above them and a negative one.  A
// box's plane on the origin's side lies there (`near`), its other one
// DR_PACK_FAR of a step further (`far`).  The step is 2^k or 1.5 * 2^k, the least of
// which 253 span both boxes, and at least four units in the last place of the
// largest coordinate; the origin lies half of DR_PACK_FAR outside the boxes (or four
// such units).  So a box without extent at the origin's end, a floor or a light below
// the ceiling, stays thin: rays that leave it or end shortly before it do not meet it.
// An axis with coordinates that are not finite, or too large for its distances, has the
// origin not-a-number: so are all of its distances, and it does not constrain a ray.
#define DR_PACK_SLACK (0.25f * DR_PACK_FAR)
struct PackAxis {
    float origin, rstep;
    uint32_t step;  // the top 9 bits below the sign of the step as a float
};
DR_INLINE PackAxis pack_axis(float lo, float hi, bool above) {
    float most = fmaxf(fabsf(lo), fabsf(hi)), ext = hi - lo;
    if (!(lo <= hi && most < 1e18f)) return PackAxis{__uint_as_float(0x7fc00000u), 0.f, 127u << 1};
    const float ulps = most * 4.76837158203125e-7f;
    uint32_t b = __float_as_uint(fmaxf(fmaxf(ext * (1.f / 253.f), ulps), 1e-30f));
    b = (b >> 22) + ((b & 0x3fffffu) != 0);
    const float step = __uint_as_float(b << 22), out = fmaxf(step * (0.5f * DR_PACK_FAR), ulps);
    // (the origin's lowest bit: the step's sign)
    const uint32_t o = __float_as_uint(above ? hi + out : lo - out);
    return PackAxis{__uint_as_float((o & ~1u) | (above ? 1u : 0u)), (above ? -1.f : 1.f) / step, b};
}
// a near / far plane on the axis, at least DR_PACK_SLACK of a step outside v: the
// walk's rounding is at most 1e-4 of a step near the box (not-a-number: any)
DR_INLINE uint32_t pack_near(float v, const PackAxis &a) {
    return (uint32_t)fminf(fmaxf(floorf((v - a.origin) * a.rstep - DR_PACK_SLACK), 0.f), 255.f);
}
DR_INLINE uint32_t pack_far(float v, const PackAxis &a) {
    return (uint32_t)fminf(fmaxf(ceilf((v - a.origin) * a.rstep - (DR_PACK_FAR - DR_PACK_SLACK)), 0.f), 255.f);
}
// Node i of a tree in depth-first order (drh::bvh_in_order()): an interior left
// child is node i + 1, as is an interior right one beside a leaf (the two then
// change places: the first child is a leaf only if both are), and sibling
// leaves' triangles lie side by side.
DR_INLINE DrPackedNode pack_node(const DrNode &n, int i) {
    const bool leaf0 = n.d[2] > 0, leaf1 = n.d[3] > 0;
    // a root that is a leaf has no sibling: the second leaf has no triangles
    const bool none = !leaf1 && n.d[1] == 0;
    const bool swap = leaf0 && !leaf1 && !none;
    DrPackedNode p;
    uint32_t steps = 0;
    auto boxes = [&](int k, float l0, float h0, float l1, float h1) {
        if (none) {
            l1 = l0;
            h1 = h0;
        }
        // (not-a-number in either box: `lo <= hi` fails)
        const float lo = l1 < l0 || l1 != l1 ? l1 : l0, hi = h1 > h0 || h1 != h1 ? h1 : h0;
        const PackAxis a = pack_axis(lo, hi, false), b = pack_axis(lo, hi, true);
        const uint32_t an0 = pack_near(l0, a), af0 = pack_far(h0, a), an1 = pack_near(l1, a), af1 = pack_far(h1, a);
        const uint32_t bn0 = pack_near(h0, b), bf0 = pack_far(l0, b), bn1 = pack_near(h1, b), bf1 = pack_far(l1, b);
        // the end at which the boxes are thinner
        const bool above = bf0 - bn0 + (bf1 - bn1) < af0 - an0 + (af1 - an1);
        const uint32_t c0 = above ? bn0 | bf0 << 8 : an0 | af0 << 8, c1 = above ? bn1 | bf1 << 8 : an1 | af1 << 8;
        p.w[k] = __float_as_uint(above ? b.origin : a.origin);
        p.w[4 + k] = swap ? c1 | c0 << 16 : c0 | c1 << 16;
        steps |= a.step << (22 - 9 * k);
    };
    boxes(0, n.a[0], n.a[3], n.b[2], n.c[1]);
    boxes(1, n.a[1], n.b[0], n.b[3], n.c[2]);
    boxes(2, n.a[2], n.b[1], n.c[0], n.c[3]);
    const uint32_t n0 = leaf0 && !swap ? (uint32_t)n.d[2] : 0u, n1 = leaf1 ? (uint32_t)n.d[3] : (swap ? (uint32_t)n.d[2] : 0u);
    p.w[3] = steps | (leaf0 || leaf1 ? 0x80000000u : 0u) | n0 | n1 << 2;
    p.w[7] = (uint32_t)(leaf0 ? n.d[0] : n.d[1]);
    return p;
}
