// The quantized boxes of the 8-wide tree and the conservative test of a ray against
// them: plain FP32 / FP64 arithmetic that the collapse and the traversal share, and that
// a host program can run against the reference's slab test (box_hit).
#pragma once

#include "pbrtm_geometry.h"

namespace pbrtm {

// 2^e for e in [-126, 127], exactly.
PBRTM_HD float pow2f(int e) { return __builtin_bit_cast(float, uint32_t(e + 127) << 23); }

// Exponent of a node's step along an axis of extent ext: the smallest power of two with
// ext / step <= 253.
PBRTM_HD int box_step_exp(float ext) {
    int e = -126;
    if (ext > 0.f) {
        int e2;
        frexpf(ext / 253.0f, &e2);
        e = e2;
        if (ldexpf(1.0f, e2 - 1) * 253.0f >= ext) e = e2 - 1;
    }
    return e < -126 ? -126 : (e > 126 ? 126 : e);
}

// Quantized lower / upper plane of a coordinate v in a node of origin org and step 2^e
// (inv_step = 2^-e, so the divisions are exact products). The plane lies outside the
// coordinate as a real number, org + q * step, not only after rounding, so that a
// traversal which does not round planes to FP32 needs no allowance for it: far from the
// world's origin such an allowance outgrows the boxes. q * step is exact, and compared
// with v - org as the rounded difference and what it lost. The byte from the rounded
// difference is off by one at most, so there is no loop: the collapse does this 48 times a
// node, and with loops (on the rounded plane, or in FP64) a rebuild of 10M triangles with
// its two traces takes 7.67 and 7.71 ms, so 7.47.
PBRTM_HD float sub_lost(float a, float b, float d) {  // a - b - d, d = fl(a - b): Knuth's TwoSum
    const float t = d - a;
    return (a - (d - t)) - (b + t);
}
PBRTM_HD int box_quant_lo(float v, float org, float step, float inv_step) {
    const float d = v - org, e = sub_lost(v, org, d);
    const int q = int(fminf(255.f, fmaxf(0.f, floorf(d * inv_step))));
    return q - int(q > 0 && (float(q) * step > d || (float(q) * step == d && e < 0.f)));
}
PBRTM_HD int box_quant_hi(float v, float org, float step, float inv_step) {
    const float d = v - org, e = sub_lost(v, org, d);
    const int q = int(fminf(255.f, fmaxf(0.f, ceilf(d * inv_step))));
    return q + int(q < 255 && (float(q) * step < d || (float(q) * step == d && e > 0.f)));
}

// Conservative slab test of the quantized boxes. In a node, the distance to the
// plane with byte q is q * A + B, A = step * inv and B = (org - o) * inv: one
// conversion and one fmaf per plane instead of decoding the plane, subtracting the
// origin and multiplying. It must never miss a box whose exact box the reference's
// test (box_hit) enters, so the near distances are lowered and the far ones raised
// by err = 16u (|B| + 255 |A|), u = 2^-24. In units of u (|B| + 255 |A|), which bounds
// the distance to every plane of the node, what separates the two is at most 13.01:
//   - box_hit's difference and product: 2.01, and its widening of the far distances,
//     2 gamma(3) + u: 7.01 (the near distances are not widened);
//   - the roundings of B (2.01), of B -+ err (1.01) and of the fmaf (1.01);
//   - the quantized planes contain the exact ones as real numbers and A is exact (a power
//     of two times inv): nothing. In particular nothing here grows with the distance of
//     the scene from the world's origin.
// A component of d that is zero or tiny has a reciprocal that is infinite or very large:
// it is clamped to 2^32 times the least |inv| of the ray, and err of that axis raised by
// four times the distance at which the axis of the least |inv| has left the tree's box.
// That covers every distance that the other axes can hold against it (a plane that
// touches o has t = 0 or NaN in the reference), and moves its planes outwards by 2^-30
// of the size of the tree and the ray's distance from it, whatever their scale.
// Rays without a direction, with NaNs or far outside any scene (BoxRay::generic) take
// the reference's own test on the decoded planes. So do rays from so far away that err,
// which grows with |B|, is no longer small against the tree's boxes: it widens them by
// 2^-20 of the distance, and were the nodes of equal squares on a face of the tree's box
// their edge would be extent / sqrt(num_nodes). A ray is conservative up to a distance of
// 3 * 2^16 such edges, where it widens by 3/16 of one. The reference's test makes a visit
// a fourth dearer. 524,288 closest hits without and with the rule, in ms:
//   height field of 3.9M triangles, 500 / 1000 extents away: 0.42 / 0.68, with it 0.33 / 0.36
//   the same with 320,000 triangles, 1000 / 2000: 0.29 / 0.35, with it 0.28 / 0.27
//   10M random triangles, 500 / 2000 / 30,000: 1.28 / 10.9 / 497, with it 1.46 / 8.3 / 54
//   20,000 random triangles, 4000 / 30,000: 0.66 / 1.99, with it 0.77 / 1.35
// Random triangles fill the box, so their nodes are larger than on a face. A line by the
// cube root of num_nodes saves what they lose at the first distances, and leaves the height
// fields as they are without the rule.
constexpr float kBoxErr = 16.0f * 5.9604644775390625e-08f;

// A ray's reciprocal direction for the box tests (clamped; as it is if generic) and its
// clamped axes' constant error term (else 0).
struct BoxRay {
    f3 inv, err;
    bool generic;
};
// What a ray's start needs to know of a tree: the lower corner of its box, the box's largest
// extent, and the distance from the corner along an axis up to which rays are conservative.
struct TreeBox {
    f3 lo;
    float extent, reach;
};
inline TreeBox tree_box(const float bounds[6], uint32_t num_nodes) {
    float extent = 0.f;
    for (int a = 0; a < 3; ++a) {
        const float e = bounds[3 + a] - bounds[a];
        extent = e > extent || e != e ? e : extent;  // a NaN stays: every ray is generic
    }
    return {{bounds[0], bounds[1], bounds[2]}, extent, extent * (0x1.8p17f / sqrtf(float(num_nodes)))};
}
PBRTM_HD BoxRay box_ray(f3 o, f3 d, f3 inv, TreeBox tree) {
    const f3 a = abs3(inv);
    const float least = fminf(fminf(a.x, a.y), a.z), cap = least * 0x1p32f;
    BoxRay r{inv, {0.f, 0.f, 0.f}, false};
    const float span = fabsf(o.x) + fabsf(o.y) + fabsf(o.z) + fabsf(d.x) + fabsf(d.y) + fabsf(d.z);
    const f3 to = abs3(sub3(tree.lo, o));
    const float far = fmaxf(fmaxf(to.x, to.y), to.z);
    if (!(least <= 0x1p20f && span <= 0x1p60f && far <= tree.reach)) {
        r.generic = true;
    } else if (!(fmaxf(fmaxf(a.x, a.y), a.z) <= cap)) {
        const float err = 4.0f * (far + tree.extent) * least;
        if (!(a.x <= cap)) r.inv.x = copysignf(cap, inv.x), r.err.x = err;
        if (!(a.y <= cap)) r.inv.y = copysignf(cap, inv.y), r.err.y = err;
        if (!(a.z <= cap)) r.inv.z = copysignf(cap, inv.z), r.err.z = err;
    }
    return r;
}

// One axis of a node for a ray: near distance fmaf(q, a, bn), far distance fmaf(q, a, bf).
struct BoxAxis {
    float a, bn, bf;
};
PBRTM_HD BoxAxis box_axis(float org, float step, float o, float inv, float ray_err) {
    const float a = step * inv, b = (org - o) * inv;
    const float err = fmaf(fabsf(a), 255.0f * kBoxErr, fmaf(fabsf(b), kBoxErr, ray_err));
    return {a, b - err, b + err};
}
// Negative when the box of near bytes qn and far bytes qf is missed up to t_max.
PBRTM_HD float box_gap(const BoxAxis ax[3], const uint32_t qn[3], const uint32_t qf[3], float t_max) {
    const float lo = fmaxf(fmaxf(fmaxf(fmaf(float(qn[0]), ax[0].a, ax[0].bn), fmaf(float(qn[1]), ax[1].a, ax[1].bn)),
                                 fmaf(float(qn[2]), ax[2].a, ax[2].bn)),
                           0.0f);
    const float hi = fminf(fminf(fminf(fmaf(float(qf[0]), ax[0].a, ax[0].bf), fmaf(float(qf[1]), ax[1].a, ax[1].bf)),
                                 fmaf(float(qf[2]), ax[2].a, ax[2].bf)),
                           t_max);
    return hi - lo;
}

}  // namespace pbrtm
