// Ray/box and ray/triangle tests of the software traversal that replaces the
// OptiX trace and shadow programs (renderer/wavefront/trace.cpp:38-78,
// shadow.cpp:24-76). Host and device share this header so that a closest hit
// computed anywhere has the same (t, b1, b2) bits.
//
// Two triangle tests are provided:
//  * watertight (Woop, Benthin, Wald, "Watertight Ray/Triangle Intersection",
//    JCGT 2013), single precision only, used by the renderer;
//  * Moeller-Trumbore in the exact operation order of lib/bvh's Triangle
//    (lib/bvh/include/bvh/triangle.hpp:26-115), so that hits can be compared
//    bit for bit with the reference's CPU traversal on the same rays.
// The closest hit is the lexicographic minimum of (t, flattened triangle
// index), which makes it independent of the BVH layout and visit order.
#pragma once

#include "vecmath.h"

namespace btrc {

enum : int32_t
{
    TRI_WATERTIGHT = 0,
    TRI_MOLLER_TRUMBORE = 1,
};

// 4-wide BVH node, 128 bytes: one 128-byte cache line of gfx950's L2.
// Slot j holds the box of child j. child[j] >= 0 names an inner node;
// child[j] < 0 is a leaf whose triangles start at ~child[j] and number
// count[j]. Unused slots carry an empty box (lo = +inf, hi = -inf).
struct alignas(16) BvhNode4
{
    float lo_x[4], hi_x[4];
    float lo_y[4], hi_y[4];
    float lo_z[4], hi_z[4];
    // as built: inner child index, or ~first triangle of a leaf with
    // count[j] triangles (count 0: empty slot); the device copy holds the
    // traversal codes instead (inner index, leaf code, or all ones)
    int32_t child[4];
    int32_t count[4];
};
static_assert(sizeof(BvhNode4) == 128, "BvhNode4 must be one 128-byte line");

// A ray as the slab test reads it: the distance to a plane is one fused
// multiply-add b * inv + c, with the rounding of c paid for in advance.
struct RayBoxPre
{
    V3 inv;   // 1 / d, bounded (raybox_axis)
    V3 near_c; // -o / d, lowered: entry distances never come out late
    V3 far_c;  // -o / d, raised: exit distances never come out early
    bool neg_x, neg_y, neg_z;
};

// One axis, inv = |1 / d|. With v = 1/d (1 + e1) and oi = o v (1 + e2), |e| <=
// 2^-24, the plane distance fma(b, v, -oi) differs from (b - o) / d by at most
// 2^-23 of itself plus 2^-24 |oi|. near_c and far_c move by 2^-22 |oi| (and
// their own rounding takes at most 2^-24 of it), so only the relative part is
// left, which raybox_nf pays on the exit side; then by the distance along the
// ray of `out` units on this axis.
BTRC_HD void raybox_axis(float o, float d, float inv, float big, float out, float *v_out, float *near_c, float *far_c)
{
    const float m = fmaxf(fminf(inv, big), 2.9387359e-39f); // 2^-128, never 0: an empty slot's planes stay infinite
    const float v = u2f(f2u(m) | (f2u(d) & 0x80000000u));
    const float oi = o * v;
    *v_out = v;
    *near_c = fmaf(m, -out, fmaf(fabsf(oi), -2.3841858e-7f, -oi)); // 2^-22
    *far_c = fmaf(m, out, fmaf(fabsf(oi), 2.3841858e-7f, -oi));
}

BTRC_HD RayBoxPre raybox_pre(V3 o, V3 d)
{
    RayBoxPre p;
    const float ix = fabsf(1.0f / d.x), iy = fabsf(1.0f / d.y), iz = fabsf(1.0f / d.z);
    // An axis on which the ray hardly moves (zero directions among them)
    // counts as 1 / |d| = big = 2^120 / max(|o|, 1), to a power of two, which
    // keeps o v finite for every origin. That pulls its planes towards the
    // origin: a plane on the other side of it stays there; the planes around an
    // origin inside the slab, or on one of them, are moved out past every hit
    // by out = 2^-56 max(|o|, 1) / the largest |d| (out * big exceeds any t
    // that 2^63 units can take, where the triangle tests overflow). On other
    // axes that is next to nothing. Without any |d| there is no hit.
    const float mo = fmaxf(fmaxf(fabsf(o.x), fabsf(o.y)), fmaxf(fabsf(o.z), 1.0f));
    const uint32_t exponent = f2u(mo) & 0x7f800000u;
    const float big = u2f((374u << 23) - exponent);
    const float slow = fminf(ix, fminf(iy, iz)); // 1 / the largest |d|
    const float out = slow <= MAX_FLOAT ? slow * u2f(exponent - (56u << 23)) : 0.0f;
    raybox_axis(o.x, d.x, ix, big, out, &p.inv.x, &p.near_c.x, &p.far_c.x);
    raybox_axis(o.y, d.y, iy, big, out, &p.inv.y, &p.near_c.y, &p.far_c.y);
    raybox_axis(o.z, d.z, iz, big, out, &p.inv.z, &p.near_c.z, &p.far_c.z);
    p.neg_x = (f2u(d.x) >> 31) != 0;
    p.neg_y = (f2u(d.y) >> 31) != 0;
    p.neg_z = (f2u(d.z) >> 31) != 0;
    return p;
}

// Conservative slab test of one box, its near and far planes already chosen
// by the ray's direction signs; the entry distance goes to *tentry. Six
// fused multiply-adds: half the arithmetic of (b - o) * inv per plane. The
// maxNum / minNum chains drop NaN operands (0 * inf planes), as the robust
// max / min of lib/bvh do (lib/bvh/include/bvh/utilities.hpp:62-71); tmin and
// tmax are never NaN. The exit side is widened by 2^-21, more than the two
// sides' 2^-23 each (Ize, "Robust BVH Ray Traversal", JCGT 2013).
BTRC_HD bool raybox_nf(const RayBoxPre &p, float nx, float fx, float ny, float fy, float nz, float fz,
                       float tmin, float tmax, float *tentry)
{
    const float t0x = fmaf(nx, p.inv.x, p.near_c.x);
    const float t0y = fmaf(ny, p.inv.y, p.near_c.y);
    const float t0z = fmaf(nz, p.inv.z, p.near_c.z);
    const float t1x = fmaf(fx, p.inv.x, p.far_c.x);
    const float t1y = fmaf(fy, p.inv.y, p.far_c.y);
    const float t1z = fmaf(fz, p.inv.z, p.far_c.z);
    const float te = fmaxf(t0x, fmaxf(t0y, fmaxf(t0z, tmin)));
    const float tx = fminf(t1x, fminf(t1y, fminf(t1z, tmax)));
    *tentry = te;
    return te <= fmaf(fabsf(tx), 4.7683716e-7f, tx);
}

// Box culling distance for the current closest hit. A box's entry distance
// and a triangle's t come from different arithmetic: the slab entry carries
// ~2 ulps of rounding, the watertight t an error of order 2^-24 times the
// distance from the ray origin to the triangle's vertices (it works on
// v - o), which for a ray starting close to a large triangle is many ulps of
// t (11 ulps were seen for a hit at t = 0.037 on a 2-unit floor). Culling
// therefore keeps every box whose entry lies within best_t (1 + 2^-20) +
// margin, with margin = 2^-18 (scene extent + |o|) from cull_margin: a hit
// no farther than the current one (a tie included) is never culled, so the
// (t, index) minimum does not depend on the visit order.
BTRC_HD float cull_margin(float scene_extent, V3 o)
{
    const float m = fmaxf(fabs_(o.x), fmaxf(fabs_(o.y), fabs_(o.z)));
    return (scene_extent + m) * (1.0f / 262144.0f);
}

BTRC_HD float cull_distance(float best_t, float margin)
{
    return best_t < MAX_FLOAT ? best_t * 1.00000095f + margin : best_t;
}

// ---- watertight test ----

// The ray as the watertight test reads it: its axes permuted so that z is the
// largest direction component, and the shear to it. Triangle coordinates
// come in the same permutation.
struct WatertightPre
{
    int32_t kx, ky, kz;
    float ox, oy, oz; // origin components kx, ky, kz
    float Sx, Sy, Sz;
};

BTRC_HD WatertightPre watertight_pre(V3 o, V3 d)
{
    WatertightPre w;
    const float ax = fabs_(d.x), ay = fabs_(d.y), az = fabs_(d.z);
    int32_t kz = ax > ay ? (ax > az ? 0 : 2) : (ay > az ? 1 : 2);
    int32_t kx = kz + 1 == 3 ? 0 : kz + 1;
    int32_t ky = kx + 1 == 3 ? 0 : kx + 1;
    if(comp(d, kz) < 0.0f)
    {
        const int32_t t = kx;
        kx = ky;
        ky = t;
    }
    w.kx = kx;
    w.ky = ky;
    w.kz = kz;
    w.ox = comp(o, kx);
    w.oy = comp(o, ky);
    w.oz = comp(o, kz);
    const float dz = comp(d, kz);
    w.Sx = comp(d, kx) / dz;
    w.Sy = comp(d, ky) / dz;
    w.Sz = 1.0f / dz;
    return w;
}

// Returns true on a hit with t in [tmin, tmax]; (b1, b2) are the barycentric
// weights of v1 and v2. vx, vy, vz: components kx, ky, kz of v0, v1, v2.
BTRC_HD bool watertight_hit(const WatertightPre &w, V3 vx, V3 vy, V3 vz, float tmin, float tmax,
                            float *t_out, float *b1_out, float *b2_out)
{
    const float Akz = vz.x - w.oz, Bkz = vz.y - w.oz, Ckz = vz.z - w.oz;
    const float Ax = (vx.x - w.ox) - w.Sx * Akz;
    const float Ay = (vy.x - w.oy) - w.Sy * Akz;
    const float Bx = (vx.y - w.ox) - w.Sx * Bkz;
    const float By = (vy.y - w.oy) - w.Sy * Bkz;
    const float Cx = (vx.z - w.ox) - w.Sx * Ckz;
    const float Cy = (vy.z - w.oy) - w.Sy * Ckz;
    const float U = Cx * By - Cy * Bx;
    const float V = Ax * Cy - Ay * Cx;
    const float W = Bx * Ay - By * Ax;
    if((U < 0.0f || V < 0.0f || W < 0.0f) && (U > 0.0f || V > 0.0f || W > 0.0f))
        return false;
    const float det = U + V + W;
    if(det == 0.0f)
        return false;
    const float Az = w.Sz * Akz;
    const float Bz = w.Sz * Bkz;
    const float Cz = w.Sz * Ckz;
    const float T = U * Az + V * Bz + W * Cz;
    const float rcp = 1.0f / det;
    const float t = T * rcp;
    if(!(t >= tmin && t <= tmax))
        return false;
    *t_out = t;
    *b1_out = V * rcp;
    *b2_out = W * rcp;
    return true;
}

// ---- lib/bvh Moeller-Trumbore (triangle.hpp:95-115) ----

struct MTPre
{
    V3 o, d;
};

BTRC_HD MTPre mt_pre(V3 o, V3 d)
{
    MTPre m;
    m.o = o;
    m.d = d;
    return m;
}

// Returns lib/bvh's (t, u, v) for the triangle (p0, p1, p2).
BTRC_HD bool mt_hit(const MTPre &m, V3 v0, V3 v1, V3 v2, float tmin, float tmax,
                    float *t_out, float *u_out, float *v_out)
{
    const V3 e1 = v0 - v1;
    const V3 e2 = v2 - v0;
    const V3 n = cross(e1, e2);
    const V3 c = v0 - m.o;
    const V3 r = cross(m.d, c);
    const float inv_det = 1.0f / dot(n, m.d);
    const float u = dot(r, e2) * inv_det;
    const float v = dot(r, e1) * inv_det;
    const float w = 1.0f - u - v;
    if(u >= 0.0f && v >= 0.0f && w >= 0.0f)
    {
        const float t = dot(n, c) * inv_det;
        if(t >= tmin && t <= tmax)
        {
            *t_out = t;
            *u_out = u;
            *v_out = v;
            return true;
        }
    }
    return false;
}

} // namespace btrc
