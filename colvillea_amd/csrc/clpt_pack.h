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
 * -inf below the half range.  Values above it give the largest half. */
__host__ __device__ inline uint16_t half_floor(double x)
{
    const double tiny = 6.103515625e-05; /* 2^-14 */
    if (x >= 0.0 && x < tiny)
        return 0u;
    if (x < 0.0 && x > -tiny)
        return (uint16_t)(0x8000u | (1u << 10));
    if (x >= 65504.0)
        return 0x7bffu;
    if (x < -65504.0)
        return 0xfc00u;
    int          e;
    const double f = frexp(fabs(x), &e);    /* |x| = f 2^e, f in [1/2, 1) */
    const double m = f * 2048.0;            /* 11 significant bits: [1024, 2048) */
    uint32_t     k = (uint32_t)m;           /* towards zero */
    if (x < 0.0 && (double)k != m)
        ++k;                                /* away from zero */
    if (k == 2048u)
    {
        k = 1024u;
        ++e;
    }
    return (uint16_t)((x < 0.0 ? 0x8000u : 0u) | ((uint32_t)(e + 14) << 10) | (k - 1024u));
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
        float l = INFINITY, h = -INFINITY;
        for (int c = 0; c < 4; ++c)
            if (in.child[c] != CLPT_CHILD_EMPTY)
            {
                l = fminf(l, lo[a][c]);
                h = fmaxf(h, hi[a][c]);
            }
        if (l <= h && l >= -3.0e38f && h <= 3.0e38f)
        {
            p[a] = l;
            ext  = fmax(ext, (double)h - (double)l);
        }
    }
    /* s = 2^k with the extent at most 2^14 s; far out of range, planes
     * beyond the halves become infinite */
    int k = -60;
    if (ext > 0.0)
    {
        (void)frexp(ext, &k); /* ext < 2^k */
        k -= 14;
        k = k < -60 ? -60 : (k > 60 ? 60 : k);
    }
    const double s = ldexp(1.0, k), w = ext * 9.5367431640625e-07; /* 2^-20 */
    for (int a = 0; a < 3; ++a)
        for (int c = 0; c < 4; ++c)
        {
            if (in.child[c] == CLPT_CHILD_EMPTY)
            {
                out.pl[a][0][c] = 0x7c00u; /* +inf */
                out.pl[a][1][c] = 0xfc00u; /* -inf */
                continue;
            }
            out.pl[a][0][c] = half_floor(((double)lo[a][c] - w - (double)p[a]) / s);
            out.pl[a][1][c] = half_ceil(((double)hi[a][c] + w - (double)p[a]) / s);
        }
    for (int a = 0; a < 3; ++a)
        out.p[a] = p[a];
    out.s = (float)s;
    for (int c = 0; c < 4; ++c)
        out.child[c] = in.child[c];
}

#endif
