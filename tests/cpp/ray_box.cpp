// The traversal's slab and watertight tests on host-given rays: for ray i
// against triangle i, hit[i] bit 0: the watertight test hits within [tmin,
// tmax]; bit 1: the slab test enters the triangle's box within it; bit 2: it
// enters the box given in `boxes`.
#include <algorithm>

#include "../../btrc_amd/csrc/core/traverse.h"

using namespace btrc;

static bool enters(const RayBoxPre &rb, const float *lo, const float *hi, float tmin, float tmax)
{
    float te;
    return raybox_nf(rb, rb.neg_x ? hi[0] : lo[0], rb.neg_x ? lo[0] : hi[0], rb.neg_y ? hi[1] : lo[1],
                     rb.neg_y ? lo[1] : hi[1], rb.neg_z ? hi[2] : lo[2], rb.neg_z ? lo[2] : hi[2], tmin, tmax, &te);
}

extern "C" void ray_box(const float *rays, const float *tris, const float *boxes, int n, unsigned char *hit)
{
    for(int i = 0; i < n; ++i)
    {
        const float *r = rays + 8 * i, *p = tris + 9 * i, *b = boxes + 6 * i;
        const V3 o = v3(r[0], r[1], r[2]), d = v3(r[4], r[5], r[6]);
        const WatertightPre w = watertight_pre(o, d);
        const RayBoxPre rb = raybox_pre(o, d);
        auto axis = [&](int k) { return v3(p[k], p[3 + k], p[6 + k]); };
        float t, b1, b2, lo[3], hi[3];
        for(int k = 0; k < 3; ++k)
        {
            lo[k] = std::min({ p[k], p[3 + k], p[6 + k] });
            hi[k] = std::max({ p[k], p[3 + k], p[6 + k] });
        }
        hit[i] = (watertight_hit(w, axis(w.kx), axis(w.ky), axis(w.kz), r[3], r[7], &t, &b1, &b2) ? 1 : 0) |
                 (enters(rb, lo, hi, r[3], r[7]) ? 2 : 0) | (enters(rb, b, b + 3, r[3], r[7]) ? 4 : 0);
    }
}
