/* Host check of the packed BVH4 node (colvillea_amd/csrc/clpt_pack.h): over
 * nodes of many extents and places (flat, tiny, huge beyond what halves and
 * the slab test's products hold, far from the origin, with planes that are
 * not finite, with empty slots), every packed box contains the float box, empty slots
 * are inverted and infinite, and the packed slab test passes every child
 * that the float slab test passes, for rays that graze and miss boxes,
 * start inside, far away and along axes.  Prints "ok" or the failures. */
#include "../colvillea_amd/csrc/clpt_pack.h"

#include <cmath>
#include <cstdio>
#include <cstring>
#include <random>

static int failures = 0;
static void fail(const char* what, double a, double b)
{
    if (failures++ < 10)
        std::printf("%s: %.17g %.17g\n", what, a, b);
}

static double half_value(uint16_t h)
{
    const int    e = (h >> 10) & 31, m = h & 1023;
    const double s = h & 0x8000u ? -1.0 : 1.0;
    if (e == 31)
        return m ? NAN : s * INFINITY;
    return e ? s * std::ldexp(1024.0 + m, e - 25) : s * std::ldexp((double)m, -24);
}

static float rcp(float d)
{
    const float tiny = 1e-20f;
    return 1.0f / (std::fabs(d) > tiny ? d : (d < 0.0f ? -tiny : tiny));
}

/* the slab test on float boxes (the packed one is the kernels' own) */
static bool pass_float(const float lo[3], const float hi[3], const float o[3], const float inv[3], float tmin, float tmax)
{
    float n = tmin, f = tmax;
    for (int a = 0; a < 3; ++a)
    {
        const float t0 = (lo[a] - o[a]) * inv[a], t1 = (hi[a] - o[a]) * inv[a];
        n = std::fmax(n, inv[a] < 0.0f ? t1 : t0);
        f = std::fmin(f, inv[a] < 0.0f ? t0 : t1);
    }
    return n * 0.99999f <= f * 1.00001f;
}

static bool pass_packed(const Node4P& p, int c, const float o[3], const float inv[3], float tmin, float tmax)
{
    const PackRay r = pack_ray(p.p[0], p.p[1], p.p[2], p.s, o[0], o[1], o[2], inv[0], inv[1], inv[2]);
    float         n[3], f[3], t;
    for (int a = 0; a < 3; ++a)
    {
        const bool g = inv[a] < 0.0f;
        n[a]         = (float)half_value(p.pl[a][g ? 1 : 0][c]);
        f[a]         = (float)half_value(p.pl[a][g ? 0 : 1][c]);
    }
    return pack_slab(r, n[0], n[1], n[2], f[0], f[1], f[2], tmin, tmax, t);
}

int main()
{
    std::mt19937                           rng(7);
    std::uniform_real_distribution<double> U(-1.0, 1.0);
    const double sizes[]  = {1e-30, 1e-12, 1e-6, 1e-3, 0.03, 1.0, 40.0, 1e5, 1e12, 1e21, 1e25, 1e37};
    const double places[] = {0.0, 1e-4, 1.0, 30.0, 1e4, 1e9, 1e22};
    long         passes = 0, both = 0;
    for (double size : sizes)
        for (double place : places)
            for (int it = 0; it < 60; ++it)
            {
                Node4 nd;
                std::memset(&nd, 0, sizeof(nd));
                float* lo[3] = {nd.lox, nd.loy, nd.loz};
                float* hi[3] = {nd.hix, nd.hiy, nd.hiz};
                double at[3];
                for (double& x : at)
                    x = place * U(rng);
                const int empties = it % 4;
                for (int c = 0; c < 4; ++c)
                {
                    nd.child[c] = c < 4 - empties ? (uint32_t)c : CLPT_CHILD_EMPTY;
                    for (int a = 0; a < 3; ++a)
                    {
                        const double u = at[a] + size * U(rng), v = it % 5 == 0 && a == it % 3 ? u : at[a] + size * U(rng);
                        lo[a][c] = c < 4 - empties ? (float)std::fmin(u, v) : INFINITY;
                        hi[a][c] = c < 4 - empties ? (float)std::fmax(u, v) : -INFINITY;
                    }
                }
                /* boxes of vertices that are not finite */
                const int odd = it % 10, oa = it / 10 % 3;
                if (odd == 7)
                    hi[oa][0] = INFINITY;
                if (odd == 8)
                {
                    lo[oa][0] = -INFINITY;
                    hi[oa][0] = INFINITY;
                }
                if (odd == 9)
                    (it % 4 < 2 ? lo : hi)[oa][0] = NAN;
                Node4P p;
                pack_node4(nd, p);
                for (int c = 0; c < 4; ++c)
                    for (int a = 0; a < 3; ++a)
                    {
                        const double l = (double)p.p[a] + half_value(p.pl[a][0][c]) * (double)p.s;
                        const double h = (double)p.p[a] + half_value(p.pl[a][1][c]) * (double)p.s;
                        if (nd.child[c] == CLPT_CHILD_EMPTY)
                        {
                            if (!(l == INFINITY && h == -INFINITY))
                                fail("empty slot", l, h);
                        }
                        else if (l > lo[a][c] || h < hi[a][c] || l != l || h != h)
                            fail("box", l - lo[a][c], hi[a][c] - h);
                    }
                for (int r = 0; r < 200; ++r)
                {
                    const double away = std::pow(10.0, 3.0 * U(rng));
                    float        o[3], d[3], inv[3];
                    const int    c = (int)(rng() % (unsigned)(4 - empties));
                    for (int a = 0; a < 3; ++a)
                        o[a] = (float)(at[a] + size * away * U(rng));
                    /* towards a corner, an edge or the inside of a child's box */
                    for (int a = 0; a < 3; ++a)
                    {
                        const int    k = (int)(rng() % 3u);
                        const double x = k == 0 ? lo[a][c] : (k == 1 ? hi[a][c] : 0.5 * ((double)lo[a][c] + hi[a][c]));
                        d[a]           = (float)(x - o[a]);
                        if (rng() % 8u == 0u)
                            d[a] = 0.0f;
                    }
                    const double len = std::sqrt((double)d[0] * d[0] + (double)d[1] * d[1] + (double)d[2] * d[2]);
                    if (!(len > 0.0 && len < INFINITY))
                        continue;
                    /* half of the rays are not of unit length, as inside a scaled instance */
                    const double mag = r % 4 < 2 ? 1.0 : std::pow(10.0, 20.0 * U(rng));
                    for (int a = 0; a < 3; ++a)
                    {
                        d[a]   = (float)(d[a] / len * mag);
                        inv[a] = rcp(d[a]);
                    }
                    const float tmin = r % 2 ? 0.001f : 0.0f, tmax = r % 3 ? 3.402823466e+38f : (float)len;
                    for (int k = 0; k < 4 - empties; ++k)
                    {
                        const float l[3] = {lo[0][k], lo[1][k], lo[2][k]}, h[3] = {hi[0][k], hi[1][k], hi[2][k]};
                        const bool  was = pass_float(l, h, o, inv, tmin, tmax);
                        passes += was;
                        if (was && !pass_packed(p, k, o, inv, tmin, tmax))
                            fail("slab test lost a box, size and place", size, place);
                        both += was;
                    }
                }
            }
    if (passes < 100000)
        fail("too few boxes passed", (double)passes, (double)both);
    if (!failures)
        std::printf("ok %ld\n", passes);
    return failures != 0;
}
