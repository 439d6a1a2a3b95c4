/*
 * clpt_pack.h -- the BVH4 node's packed form (host and device; the device
 * packs whole trees, the host form serves checks).
 */
#ifndef CLPT_PACK_H
#define CLPT_PACK_H

#include "clpt_scene.h"

#include <math.h>
#include <string.h>

/* The largest half not above x, as its bits: 10 bits of fraction, exponents
 * -14..15 (no subnormals: values in (-2^-14, 2^-14) go to -2^-14 or 0), and
 * -inf below the half range and for NaN.  Values above it give the largest
 * half. */
__host__ __device__ inline uint16_t half_floor(double x)
{
    if (!(x >= -65504.0))
        return 0xfc00u;
    if (x >= 65504.0)
        return 0x7bffu;
    if (fabs(x) < 6.103515625e-05) /* 2^-14 */
        return x < 0.0 ? 0x8400u : 0u;
    uint64_t b;
    memcpy(&b, &x, sizeof(b));
    /* truncated towards zero; a negative value with a remainder is the next
     * one away from it, a carry out of the fraction the next exponent */
    uint32_t h = ((uint32_t)(b >> 52 & 0x7ffu) - 1008u) << 10 | (uint32_t)(b >> 42 & 0x3ffu);
    if (b >> 63 && (b & ((1ull << 42) - 1u)))
        ++h;
    return (uint16_t)((uint32_t)(b >> 63) << 15 | h);
}
__host__ __device__ inline uint16_t half_ceil(double x) { return (uint16_t)(half_floor(-x) ^ 0x8000u); }

__host__ __device__ inline void pack_node4(const Node4& in, Node4P& out)
{
    const float* lo[3] = {in.lox, in.loy, in.loz};
    const float* hi[3] = {in.hix, in.hiy, in.hiz};
    float        p[3]  = {0.0f, 0.0f, 0.0f};
    double       ext   = 0.0;
    for (int a = 0; a < 3; ++a)
    {
        /* over the planes that are finite; the others pack to infinities */
        float l = INFINITY, h = -INFINITY;
        for (int c = 0; c < 4; ++c)
            for (int k = 0; k < 2; ++k)
            {
                const float x = k ? hi[a][c] : lo[a][c];
                if (in.child[c] != CLPT_CHILD_EMPTY && fabsf(x) < INFINITY)
                {
                    l = fminf(l, x);
                    h = fmaxf(h, x);
                }
            }
        if (l <= h)
        {
            p[a] = l;
            ext  = fmax(ext, (double)h - (double)l);
        }
    }
    /* s = 2^k with the extent at most 2^14 s */
    int k = -60;
    if (ext > 0.0)
    {
        (void)frexp(ext, &k); /* ext < 2^k */
        k -= 14;
        k = k < -60 ? -60 : k;
    }
    /* From 2^60 on, (p - o) inv can overflow (|inv| is at most 1e20) for a
     * ray that lies in a child's box: such boxes take every ray. */
    const bool   open = ext >= 1.152921504606847e18;
    const double r = ldexp(1.0, -k), w = ext * 9.5367431640625e-07; /* 2^-20 */
    for (int a = 0; a < 3; ++a)
        for (int c = 0; c < 4; ++c)
        {
            if (in.child[c] == CLPT_CHILD_EMPTY)
            {
                out.pl[a][0][c] = 0x7c00u; /* +inf */
                out.pl[a][1][c] = 0xfc00u; /* -inf */
                continue;
            }
            out.pl[a][0][c] = open ? 0xfc00u : half_floor(((double)lo[a][c] - w - (double)p[a]) * r);
            out.pl[a][1][c] = open ? 0x7c00u : half_ceil(((double)hi[a][c] + w - (double)p[a]) * r);
        }
    for (int a = 0; a < 3; ++a)
        out.p[a] = p[a];
    out.s = open ? 1.0f : (float)ldexp(1.0, k);
    for (int c = 0; c < 4; ++c)
        out.child[c] = in.child[c];
}

/* The slab test on packed planes.  On each axis the plane of half q lies at
 * p + q s, at the ray's t = q (s inv) + (p - o) inv, one fused multiply-add:
 * the ray in the node's units is (i, b) = (s inv, (p - o) inv). */
struct PackRay
{
    float bx, ix, by, iy, bz, iz;
};

__host__ __device__ inline PackRay pack_ray(float px, float py, float pz, float s, float ox, float oy, float oz, float invx,
                                            float invy, float invz)
{
    PackRay r;
    r.bx = (px - ox) * invx;
    r.ix = s * invx;
    r.by = (py - oy) * invy;
    r.iy = s * invy;
    r.bz = (pz - oz) * invz;
    r.iz = s * invz;
    return r;
}

/* A child by its near and far planes (lo and hi by the sign of inv): the
 * entry distance, padded by 2e-5 relative (all on the near side), and whether
 * the ray meets the box in [tmin, tmax].  An empty slot (inverted infinite
 * box) gives +inf > far, but where every slab overflows to NaN. */
__host__ __device__ inline bool pack_slab(const PackRay& r, float nx, float ny, float nz, float fx, float fy, float fz,
                                          float tmin, float tmax, float& tnear)
{
    const float tnx = __builtin_fmaf(nx, r.ix, r.bx), tfx = __builtin_fmaf(fx, r.ix, r.bx);
    const float tny = __builtin_fmaf(ny, r.iy, r.by), tfy = __builtin_fmaf(fy, r.iy, r.by);
    const float tnz = __builtin_fmaf(nz, r.iz, r.bz), tfz = __builtin_fmaf(fz, r.iz, r.bz);
    tnear             = fmaxf(fmaxf(tnx, tny), fmaxf(tnz, tmin)) * 0.99998f;
    const float tfar  = fminf(fminf(tfx, tfy), fminf(tfz, tmax));
    return tnear <= tfar;
}

#endif
