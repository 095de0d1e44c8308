// Host run of the 8-wide tree's box arithmetic (csrc/wide_box.h) against the reference's
// slab test (box_hit): random and adversarial boxes and rays. Prints per form of rays
//   <form> rays <n> entered <exact> missed <m> extra <e> generic <g>
// where "entered" counts children whose exact box box_hit enters, "missed" those of them
// that the conservative test rejects, and "extra" the children it enters although box_hit
// rejects their decoded quantized box, and "generic" rays that take box_hit itself. Exits 1 if a quantized box does not contain its box.
#include <cmath>
using std::isfinite;
using std::isinf;
using std::isnan;

#define __HIP_PLATFORM_AMD__ 1
#include "wide_box.h"

#include <cstdio>
#include <cstdlib>
#include <cstring>

using namespace pbrtm;

static uint64_t g_state;
static uint32_t u32() {
    g_state = g_state * 6364136223846793005ull + 1442695040888963407ull;
    const uint32_t x = uint32_t(((g_state >> 18) ^ g_state) >> 27), r = uint32_t(g_state >> 59);
    return (x >> r) | (x << ((32 - r) & 31));
}
static double uni() { return u32() * (1.0 / 4294967296.0); }
static double range(double a, double b) { return a + (b - a) * uni(); }
static float sgn() { return u32() & 1 ? 1.f : -1.f; }

int main(int argc, char **argv) {
    const char *form = argv[1];
    const int n = atoi(argv[2]);
    const double scale = atof(argv[3]), offset = atof(argv[4]);
    g_state = strtoull(argv[5], nullptr, 10);
    const uint32_t nodes = uint32_t(atoi(argv[6]));  // of the tree
    // "clear-<form>": no planes or distances that coincide on purpose, no t_max
    const bool clear = !strncmp(form, "clear-", 6);
    const char *kind = clear ? form + 6 : form;
    auto is = [&](const char *f) { return !strcmp(kind, f); };
    uint64_t entered = 0, missed = 0, extra = 0, generic = 0;
    for (int it = 0; it < n; ++it) {
        // the tree's box, a node in it and a child of the node, each at times flat or flush
        double rl[3], rh[3], nl[3], nh[3];
        float lo[3], hi[3], ulo[3], uhi[3], root_lo[3], root_hi[3];
        const double depth = std::exp2(-range(0, 16));
        for (int a = 0; a < 3; ++a) {
            rl[a] = offset + scale * range(-0.1, 0.1);
            rh[a] = rl[a] + scale;
            const double w = scale * depth * (u32() % 8 ? range(0.1, 1) : std::exp2(-range(0, 20)));
            nl[a] = range(rl[a], rh[a] - w);
            nh[a] = nl[a] + w;
            ulo[a] = float(nl[a]);
            uhi[a] = std::fmax(float(nh[a]), ulo[a]);
            double l = range(ulo[a], uhi[a]), h = range(l, uhi[a]);
            if (!clear && u32() % 4 == 0) l = ulo[a];
            if (!clear && u32() % 4 == 0) h = uhi[a];
            if (!clear && u32() % 16 == 0) h = l;
            lo[a] = std::fmin(std::fmax(float(l), ulo[a]), uhi[a]);
            hi[a] = std::fmin(std::fmax(float(h), lo[a]), uhi[a]);
            root_lo[a] = std::fmin(float(rl[a]), ulo[a]);
            root_hi[a] = std::fmax(float(rh[a]), uhi[a]);
        }
        float step[3];
        uint32_t ql[3], qh[3];
        for (int a = 0; a < 3; ++a) {
            const int e = box_step_exp(uhi[a] - ulo[a]);
            step[a] = pow2f(e);
            ql[a] = uint32_t(box_quant_lo(lo[a], ulo[a], step[a], pow2f(-e)));
            qh[a] = uint32_t(box_quant_hi(hi[a], ulo[a], step[a], pow2f(-e)));
            const long double pl = (long double)ulo[a] + (long double)ql[a] * step[a];
            const long double ph = (long double)ulo[a] + (long double)qh[a] * step[a];
            if (ql[a] > 255 || qh[a] > 255 || pl > lo[a] || ph < hi[a] || fmaf(float(ql[a]), step[a], ulo[a]) > lo[a] ||
                fmaf(float(qh[a]), step[a], ulo[a]) < hi[a]) {
                printf("not contained: axis %d box [%a, %a] node [%a, %a] bytes %u %u\n", a, lo[a], hi[a], ulo[a],
                       uhi[a], ql[a], qh[a]);
                return 1;
            }
        }
        // the ray: towards a point in or near the child, from in or around the tree
        double o[3], d[3], p[3], len = 0;
        const double out = is("far") ? std::exp2(range(2, 12)) : 1.5;
        for (int a = 0; a < 3; ++a) {
            o[a] = rl[a] + scale * range(-out, 1 + out);
            p[a] = u32() % 3 ? range(lo[a], hi[a]) : range(nl[a], nh[a]);
            if (!clear && u32() % 8 == 0) p[a] = u32() & 1 ? lo[a] : hi[a];
        }
        for (int a = 0; a < 3; ++a) d[a] = p[a] - double(float(o[a]));
        if (is("axis") || is("plane") || is("tiny")) {
            const int keep = int(u32() % 3);
            for (int a = 0; a < 3; ++a) {
                if (is("axis") ? a == keep : a != keep) continue;
                // beside or inside the slab, or on one of its planes
                o[a] = clear || u32() % 3 ? p[a] : (u32() & 1 ? double(u32() & 1 ? lo[a] : hi[a]) : p[a] + scale * range(-.1, .1));
                d[a] = is("tiny") ? sgn() * std::exp2(-range(10, 148)) : sgn() * 0.0;
            }
        }
        for (int a = 0; a < 3; ++a) len += d[a] * d[a];
        if (len == 0) continue;
        const double unit = is("scaled") ? std::exp2(range(-60, 60)) : (is("short") ? std::exp2(-range(18, 60)) : 1.0);
        f3 ro{float(o[0]), float(o[1]), float(o[2])};
        const double k = unit / std::sqrt(len);
        f3 rd{float(is("tiny") && std::fabs(d[0]) < 1e-3 ? d[0] : d[0] * k), float(is("tiny") && std::fabs(d[1]) < 1e-3 ? d[1] : d[1] * k),
              float(is("tiny") && std::fabs(d[2]) < 1e-3 ? d[2] : d[2] * k)};
        const f3 inv{1.0f / rd.x, 1.0f / rd.y, 1.0f / rd.z};
        const int neg[3] = {inv.x < 0.f, inv.y < 0.f, inv.z < 0.f};
        float t_max = __builtin_inff();
        if (!clear && u32() % 3 == 0) {  // at the box's own entry distance, and a few units around it
            float tn = 0.f;
            const float ov[3] = {ro.x, ro.y, ro.z}, iv[3] = {inv.x, inv.y, inv.z};
            for (int a = 0; a < 3; ++a) tn = std::fmax(tn, ((neg[a] ? hi[a] : lo[a]) - ov[a]) * iv[a]);
            for (uint32_t s = u32() % 4; s > 0; --s) tn = std::nextafterf(tn, __builtin_inff());
            if (tn > 0.f) t_max = tn;
        }
        const bool exact = box_hit(lo, hi, ro, inv, neg, t_max);
        const float bounds[6] = {root_lo[0], root_lo[1], root_lo[2], root_hi[0], root_hi[1], root_hi[2]};
        const BoxRay R = box_ray(ro, rd, inv, tree_box(bounds, nodes));
        generic += R.generic;
        float dl[3], dh[3];
        uint32_t qn[3], qf[3];
        BoxAxis ax[3];
        const float ov[3] = {ro.x, ro.y, ro.z}, iv[3] = {R.inv.x, R.inv.y, R.inv.z}, ev[3] = {R.err.x, R.err.y, R.err.z};
        for (int a = 0; a < 3; ++a) {
            dl[a] = fmaf(float(ql[a]), step[a], ulo[a]);
            dh[a] = fmaf(float(qh[a]), step[a], ulo[a]);
            qn[a] = neg[a] ? qh[a] : ql[a];
            qf[a] = neg[a] ? ql[a] : qh[a];
            ax[a] = box_axis(ulo[a], step[a], ov[a], iv[a], ev[a]);
        }
        const bool decoded = box_hit(dl, dh, ro, inv, neg, t_max);
        const bool pass = R.generic ? decoded : !std::signbit(box_gap(ax, qn, qf, t_max));
        entered += exact;
        if (exact && !pass && missed++ < 3)
            printf("missed: o %a %a %a d %a %a %a t_max %a box %a %a %a - %a %a %a\n", ro.x, ro.y, ro.z, rd.x, rd.y, rd.z,
                   t_max, lo[0], lo[1], lo[2], hi[0], hi[1], hi[2]);
        extra += pass && !decoded;
    }
    printf("%s rays %d entered %llu missed %llu extra %llu generic %llu\n", form, n, (unsigned long long)entered,
           (unsigned long long)missed, (unsigned long long)extra, (unsigned long long)generic);
    return 0;
}
