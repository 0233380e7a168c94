// The polygon tests of the head geometry (gegs_amd/csrc/mlc.hpp) against their
// plain forms: every edge divided and every distance rooted, as the
// reference writes them (geom.cu:310-327, :442-484, :1152-1191).  Results
// must be equal bit for bit.  argv[1]: number of random polygons; argv[2]: how
// many ULP the reciprocals that the selections use are off at most (0: none).
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>
#include <vector>

// a reciprocal as far off as the device's, up or down, another way each call
static unsigned rcp_ulps = 0;
static float rcp_off(float x) {
    const float y = 1.0f / x;
    if (!rcp_ulps || !(fabsf(y) >= 1.17549435e-38f && fabsf(y) <= 1e38f)) return y;
    static uint32_t state = 12345u;
    state = state * 1664525u + 1013904223u;
    const int d = (int)((state >> 16) % (2u * rcp_ulps + 1u)) - (int)rcp_ulps;
    return __uint_as_float((uint32_t)((int64_t)__float_as_uint(y) + d));
}
#define GEGS_RCP_NEAR rcp_off
#include "../../gegs_amd/csrc/event.hpp"

namespace gegs {
float lds_env[LDS_FLOATS];
}
using namespace gegs;

static bool plain_in(P2 p, const gegs_float2 *poly, int n) {
    bool odd = false;
    int j = n - 1;
    for (int i = 0; i < n; ++i) {
        const P2 a = vtx(poly, i), b = vtx(poly, j);
        if (((a.y < p.y && b.y >= p.y) || (b.y < p.y && a.y >= p.y)) && (a.x <= p.x || b.x <= p.x))
            if (a.x + (p.y - a.y) / (b.y - a.y) * (b.x - a.x) < p.x) odd = !odd;
        j = i;
    }
    return odd;
}

static float plain_ray(P2 p0, P2 v, const gegs_float2 *poly, int n, bool &inside) {
    float best = INFI_DIST + 1.0f;
    int hits = 0;
    for (int i = 0; i < n; ++i) {
        const int j = i + 1 < n ? i + 1 : 0;
        const P2 a = vtx(poly, i), b = vtx(poly, j);
        const float den = v.x * (b.y - a.y) - v.y * (b.x - a.x);
        if (den != 0.0f) {
            const float d = ((b.x - a.x) * (p0.y - a.y) - (b.y - a.y) * (p0.x - a.x)) / den;
            const float u = ((a.x - p0.x) * v.y - (a.y - p0.y) * v.x) / den;
            if (d >= 0.0f && u >= 0.0f && u < 1.0f) {
                hits++;
                if (d < best) best = d;
            }
        }
    }
    inside = (hits & 1) != 0;
    return best;
}

static float plain_seg(P2 p, P2 v, P2 w) {
    const float l2 = (v.x - w.x) * (v.x - w.x) + (v.y - w.y) * (v.y - w.y);
    if (l2 == 0.0f) return sqrtf((p.x - v.x) * (p.x - v.x) + (p.y - v.y) * (p.y - v.y));
    const float t = ((p.x - v.x) * (w.x - v.x) + (p.y - v.y) * (w.y - v.y)) / l2;
    if (t < 0.0f) return sqrtf((p.x - v.x) * (p.x - v.x) + (p.y - v.y) * (p.y - v.y));
    if (t > 1.0f) return sqrtf((p.x - w.x) * (p.x - w.x) + (p.y - w.y) * (p.y - w.y));
    const float ax = v.x + t * (w.x - v.x), ay = v.y + t * (w.y - v.y);
    return sqrtf((p.x - ax) * (p.x - ax) + (p.y - ay) * (p.y - ay));
}

static float plain_dist(P2 p, const gegs_float2 *poly, int n) {
    float best = 1e9f;
    for (int i = 0; i < n; ++i) {
        const float d = plain_seg(p, vtx(poly, i), vtx(poly, i + 1 < n ? i + 1 : 0));
        if (d < best) best = d;
    }
    return best;
}

static bool same(float a, float b) { return memcmp(&a, &b, 4) == 0 || (a == 0.0f && b == 0.0f); }

int main(int argc, char **argv) {
    const int polys = argc > 1 ? atoi(argv[1]) : 1000;
    rcp_ulps = argc > 2 ? (unsigned)atoi(argv[2]) : 0u;
    std::mt19937 rng(5);
    auto uni = [&](float lo, float hi) { return lo + (hi - lo) * (float)(rng() >> 8) * (1.0f / 16777216.0f); };
    size_t checks = 0, hits = 0;
    for (int k = 0; k < polys; ++k) {
        const int kind = k % 6;
        int n = kind == 0 ? 4 : (kind == 1 ? 14 : (kind == 2 ? 17 : (kind == 3 ? 30 : 3 + (int)(rng() % 28))));
        std::vector<gegs_float2> v(n);
        const float scale = kind == 5 ? powf(10.0f, uni(-3.0f, 4.0f)) : 1.0f;
        const float cx = uni(-20.0f, 20.0f), cy = uni(20.0f, 60.0f);
        for (int i = 0; i < n; ++i) {
            if (kind == 0) {            // a slab, sides on the axes
                v[i] = {(i == 0 || i == 3) ? -25.0f : 25.0f, i < 2 ? 48.0f : 54.75f};
            } else if (kind == 1) {     // a leaf: near-vertical sides with steps
                const float s = i < 7 ? 0.0f : 0.5f, z = i < 7 ? i : 13 - i;
                v[i] = {cx + s + 0.04f * (float)((i * 5) % 3), 48.0f + z};
            } else if (kind == 2) {     // a leaf end: an arc closed by a far edge
                const float f = 0.4f * ((float)(i - 8) / 8.0f);
                v[i] = i < 2 ? gegs_float2{-25.0f, i ? 54.75f : 48.0f}
                             : gegs_float2{cx + 8.0f * cosf(f), 51.0f + 8.0f * sinf(f)};
            } else {
                v[i] = {cx + scale * uni(-5.0f, 5.0f), cy + scale * uni(-5.0f, 5.0f)};
            }
        }
        if (kind == 4 && n > 4) v[2] = v[1];              // an edge of no length
        for (int q = 0; q < 400; ++q) {
            P2 p = p2(cx + scale * uni(-8.0f, 8.0f), (kind == 0 || kind == 1 || kind == 2 ? 51.0f : cy) + scale * uni(-8.0f, 8.0f));
            const int i = (int)(rng() % n), j = i + 1 < n ? i + 1 : 0;
            const int place = q % 8;
            const float f = uni(0.0f, 1.0f);
            if (place == 1) p = vtx(v.data(), i);                                     // on a vertex
            if (place == 2) p = p2(v[i].x + f * (v[j].x - v[i].x), v[i].y + f * (v[j].y - v[i].y));   // on an edge
            if (place == 3) p = p2(v[i].x + uni(-1e-4f, 1e-4f), v[i].y + uni(-1e-4f, 1e-4f));
            if (place == 4) p.y = v[i].y;                                             // level with a vertex
            if (place == 5) p.x = v[i].x;
            if (place == 6) p = p2(0.5f * (v[i].x + v[j].x) + uni(-0.1f, 0.1f), 0.5f * (v[i].y + v[j].y) + uni(-0.1f, 0.1f));
            P2 d;
            const float phi = uni(0.0f, 6.2831853f), ln = uni(0.0f, 1.0f);
            d = p2(ln * cosf(phi), ln * sinf(phi));
            if (q % 16 == 0) d = p2(0.0f, 1.0f);
            if (q % 16 == 5) d = p2(uni(-1e-3f, 1e-3f), 1.0f);
            if (q % 16 == 9) d = p2(v[i].x - p.x, v[i].y - p.y);                      // aimed at a vertex
            if (q % 16 == 13) d = p2(1e-30f * uni(-1.0f, 1.0f), 0.0f);
            bool in0, in1;
            const float r0 = plain_ray(p, d, v.data(), n, in0), r1 = ray_polygon(p, d, v.data(), n, in1);
            const float s0 = plain_dist(p, v.data(), n), s1 = poly_dist(p, v.data(), n);
            const bool c0 = plain_in(p, v.data(), n), c1 = point_in_polygon(p, v.data(), n);
            checks++;
            hits += r0 < INFI_DIST;
            if (!same(r0, r1) || in0 != in1 || !same(s0, s1) || c0 != c1) {
                printf("polygon %d kind %d n %d query %d: ray %.9g %.9g (%d %d) distance %.9g %.9g inside %d %d\n", k, kind, n,
                       q, r0, r1, in0, in1, s0, s1, c0, c1);
                return 1;
            }
        }
    }
    printf("checks %zu hits %zu\n", checks, hits);
    return 0;
}
