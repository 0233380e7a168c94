// mlc.hpp -- multileaf collimator module (DYNVMLC-type, 60 leaf pairs).
//
// The MLC is a slab z in [zmin, zmin + zthick] of the head frame (z from the
// source).  Across the leaves (x-z plane) every leaf is a 14-vertex polygon
// with source-focused sides (cross_xz, leaf i at [16 i, 16 i + 14)); along the
// leaf travel (y-z plane) a leaf pair's ends are a 34-vertex profile
// (endnode: [0,1] the -rmax edge, [2,16] the bank A end, [17,31] the bank B
// end, [32,33] the +rmax edge) shifted to the field's leaf positions.  A
// particle in the module carries its leaf index (>= 0: inside leaf i's
// cross-section; -(i+1): in the air gap next to leaf i; OUTMLC: not yet
// located; PASSMLC: has left the MLC towards the next module) and its bank
// (0 field opening, 1 bank A, 2 bank B, -1 not yet located).
// Geometry of the reference: geom.cu:310-790 (howfar), :1152-1286 (hownear),
// init.cu:345-611 (polygons), :1594-1662 (leaf ends per field).
#pragma once
// Included by transport.hpp after Env, Part and the phantom geometry.

namespace gegs {

constexpr int MLC_LEAVES = GEGS_MLC_LEAVES;
constexpr int OUTMLC = -99;
constexpr int PASSMLC = -98;
constexpr uint32_t REG_AIR = 1;          // default_reg
constexpr uint32_t REG_MLC = 3;          // MLC_region

struct P2 {
    float x, y;
};

__device__ __forceinline__ P2 p2(float x, float y) {
    P2 q;
    q.x = x;
    q.y = y;
    return q;
}

__device__ __forceinline__ P2 vtx(const gegs_float2 *poly, int i) { return p2(poly[i].x, poly[i].y); }

// The polygon tests below run at every step in the head: an electron in a
// leaf measures its distance to up to 44 edges and traces its ray through up
// to 52.  They were bound by the divisions and square roots of every edge,
// executed for the whole wavefront wherever one lane took that branch.  Each
// now decides with cheap arithmetic whose error is bounded which edge the
// result comes from, and evaluates only that one as the reference does, so
// the results are the reference's bit for bit.  The 5-field MLC plan of 2e6
// histories went from 73.3 to 64.7 ms with them (and with the slab's distance and the
// exit leaf left to the branches that use them), jaws and MLC 1e5 from 25.6 to
// 22.9 ms.

// 1/x to about 1 ULP, for the selections only (no result depends on it).
// The CPU check of the selections gives its own, as far off as the device's.
__device__ __forceinline__ float rcp_near(float x) {
#if defined(__HIP_DEVICE_COMPILE__) && __HIP_DEVICE_COMPILE__
    return __builtin_amdgcn_rcpf(x);
#elif defined(GEGS_RCP_NEAR)
    return GEGS_RCP_NEAR(x);
#else
    return 1.0f / x;
#endif
}

// crossing-number test (geom.cu:310-327): a horizontal ray from p to -x.
// Where both ends of a crossed edge are to the left of p by more than the
// interpolation's rounding (a few ULP of their coordinates), the crossing is
// to the left without the division.
__device__ __forceinline__ bool point_in_polygon(P2 p, const gegs_float2 *poly, int n) {
    bool odd = false;
    P2 b = vtx(poly, n - 1);
    for (int i = 0; i < n; ++i) {
        const P2 a = vtx(poly, i);
        if (((a.y < p.y && b.y >= p.y) || (b.y < p.y && a.y >= p.y)) && (a.x <= p.x || b.x <= p.x)) {
            const float hi = fmaxf(a.x, b.x);
            const float slack = 1e-5f * (fabsf(a.x) + fabsf(b.x) + fabsf(p.x));
            if (hi + slack < p.x) odd = !odd;
            else if (a.x + (p.y - a.y) / (b.y - a.y) * (b.x - a.x) < p.x) odd = !odd;
        }
        b = a;
    }
    return odd;
}

// bank of a point in the y-z plane of leaf pair `en` (geom.cu:330-344)
__device__ __forceinline__ int point_in_leaf(P2 p, const gegs_float2 *en) {
    if (point_in_polygon(p, en, 17)) return 1;
    if (point_in_polygon(p, en + 17, 17)) return 2;
    return 0;
}

// leaf whose cross-section holds p (x across the leaves, y = z); -(i+1) in
// the gap after leaf i, OUTMLC outside the leaf rows (geom.cu:346-410)
__device__ __forceinline__ int index_of_leaf(const gegs_mlc &m, P2 p) {
    const float x = p.x / p.y * m.zmin;
    const float z = p.y - m.zmin;
    if (z < 0.0f || z > m.zthick) return OUTMLC;
    if (x < m.x_start || x > m.x_end) return OUTMLC;
    int i = OUTMLC;
    if (x < m.x_start + m.wt) {
        i = 0;
    } else if (x < m.x_mid_1 + m.wt) {
        i = (int)((x - m.x_start - m.wt) / (m.wl_full + m.air_gap));
    } else if (x < m.x_mid_2 + m.wt) {
        const float pair = m.wl_target + m.wl_isocenter + m.air_gap * 2.0f;
        i = (int)((x - m.x_mid_1 - m.wt) / pair);
        if (x - m.x_mid_1 - m.wt - pair * (float)i < m.wl_target + m.air_gap) i = 10 + i * 2;
        else i = 11 + i * 2;
    } else if (x < m.x_end - m.wl_full) {
        i = (int)((x - m.x_mid_2 - m.wt) / (m.wl_full + m.air_gap)) + 50;
    } else if (x <= m.x_end) {
        i = 58;
    }
    int index = OUTMLC;
    if (i >= 0) {
        if (point_in_polygon(p, m.cross_xz + i * 16, 14)) index = i;
        else if (i < MLC_LEAVES - 1) index = point_in_polygon(p, m.cross_xz + (i + 1) * 16, 14) ? i + 1 : -(i + 1);
    }
    return index;
}

// distance along v (not normalised: the result is in units of |v|) to the
// nearest polygon edge, and whether p0 is inside (odd number of crossings);
// an edge is hit for u in [0, 1) so that a vertex counts once (geom.cu:442-484).
// d = nd / den >= 0 and u = nu / den in [0, 1) are decided by signs and
// |nu| < |den|: a quotient of binary32 numbers rounds to 1 or more exactly
// when |nu| >= |den|, and to a value >= 0 when the signs agree.  (It also
// does when a negative quotient underflows to -0: numerators of opposite sign
// below 1e-36 in size are divided.)  Rounding keeps order, so the nearest
// hit's distance is the one quotient of the smallest fraction; two fractions
// closer than the reciprocals' error are compared by their quotients.
__device__ __forceinline__ float ray_polygon(P2 p0, P2 v, const gegs_float2 *poly, int n, bool &inside) {
    float bn = 0.0f, bd = 0.0f, bq = 0.0f;   // nearest hit: nd, |den|, nd / |den| approximately
    int hits = 0, kept = 0;
    const P2 first = vtx(poly, 0);
    P2 a = first;
    float wx = p0.x - a.x, wy = p0.y - a.y;
#pragma unroll 2
    for (int i = 0; i < n; ++i) {
        const P2 b = i + 1 < n ? vtx(poly, i + 1) : first;
        const float ex = b.x - a.x, ey = b.y - a.y;
        const float den = v.x * ey - v.y * ex;
        const float nd0 = ex * wy - ey * wx;
        const float nu0 = wy * v.x - wx * v.y;
        const float ad = fabsf(den);
        const float nd = den < 0.0f ? -nd0 : nd0, nu = den < 0.0f ? -nu0 : nu0;
        if (den != 0.0f && nd > -1e-36f && nu > -1e-36f && nu < ad) {
            if (!(nd < 0.0f || nu < 0.0f) || (nd / ad >= 0.0f && nu / ad >= 0.0f)) {
                hits++;
                const float q = nd * rcp_near(ad);
                const bool clear = ad >= 1e-30f && bd >= 1e-30f;   // normal reciprocals
                bool take = kept == 0 || (clear && q < bq * 0.999999f);
                if (!take && !(clear && q > bq * 1.000001f)) take = nd / ad < bn / bd;
                if (take) {
                    bn = nd;
                    bd = ad;
                    bq = q;
                    kept = 1;
                }
            }
        }
        a = b;
        wx = p0.x - a.x;
        wy = p0.y - a.y;
    }
    inside = (hits & 1) != 0;
    float best = INFI_DIST + 1.0f;
    if (kept) {
        const float d = bn / bd;
        if (d < best) best = d;
    }
    return best;
}

// squared distance of p to the segment v-w, as the reference's distance
// before its square root (geom.cu:1152-1170)
__device__ __forceinline__ float seg_dist2(P2 p, P2 v, P2 w) {
    const float l2 = (v.x - w.x) * (v.x - w.x) + (v.y - w.y) * (v.y - w.y);
    const float t = l2 == 0.0f ? -1.0f : ((p.x - v.x) * (w.x - v.x) + (p.y - v.y) * (w.y - v.y)) / l2;
    // the nearest point: an end, or the foot at t (NaN takes the foot, as `t < 0`, `t > 1` both false)
    const float ax = t < 0.0f ? v.x : (t > 1.0f ? w.x : v.x + t * (w.x - v.x));
    const float ay = t < 0.0f ? v.y : (t > 1.0f ? w.y : v.y + t * (w.y - v.y));
    return (p.x - ax) * (p.x - ax) + (p.y - ay) * (p.y - ay);
}

// perpendicular distance to the nearest edge (geom.cu:1152-1191).  The square
// root keeps order, so it is taken once, of the smallest squared distance.
// A first pass estimates every edge's squared distance (reciprocal instead of
// the division, no branches) and keeps the two nearest; both estimates and
// the reference's values are within 32 units of 2^-24 of the lengths
// involved (|p|, the distance and the longest edge: seg_dist2's and the
// estimate's roundings add up to 26), so only edges within that of the
// nearest estimate can hold the smallest value.  Usually the two nearest do
// (neighbours that share the nearest vertex); with a third one as near,
// every edge is evaluated.
__device__ __forceinline__ float poly_dist(P2 p, const gegs_float2 *poly, int n) {
    float b1 = 3.0e38f, b2 = 3.0e38f, b3 = 3.0e38f, lmax = 0.0f;
    int i1 = -1, i2 = -1;
    const P2 first = vtx(poly, 0);
    P2 a = first;
#pragma unroll 2
    for (int i = 0; i < n; ++i) {
        const P2 b = i + 1 < n ? vtx(poly, i + 1) : first;
        const float ex = b.x - a.x, ey = b.y - a.y, wx = p.x - a.x, wy = p.y - a.y;
        const float l2 = ex * ex + ey * ey;
        // a degenerate edge (0 x inf) takes its first end
        const float t = fminf(fmaxf((wx * ex + wy * ey) * rcp_near(l2), 0.0f), 1.0f);
        const float rx = wx - t * ex, ry = wy - t * ey;
        const float x = rx * rx + ry * ry;
        lmax = fmaxf(lmax, l2);
        const bool n1 = x < b1, n2 = x < b2;
        b3 = n2 ? b2 : fminf(b3, x);
        b2 = n1 ? b1 : (n2 ? x : b2);
        i2 = n1 ? i1 : (n2 ? i : i2);
        b1 = n1 ? x : b1;
        i1 = n1 ? i : i1;
        a = b;
    }
    float x = 1.0e38f;
    if (i1 >= 0) {
        const float s = sqrtf(b1);
        const float slack = 1.9073486e-6f * (fabsf(p.x) + fabsf(p.y) + s + sqrtf(lmax));   // 32 x 2^-24
        const float reach = (s + 2.0f * slack) * (s + 2.0f * slack);
        if (b3 <= reach || !(reach < 1.0e37f)) {
            i1 = -1;
        } else {
            x = seg_dist2(p, vtx(poly, i1), vtx(poly, i1 + 1 < n ? i1 + 1 : 0));
            if (b2 <= reach) {
                const float y = seg_dist2(p, vtx(poly, i2), vtx(poly, i2 + 1 < n ? i2 + 1 : 0));
                if (y < x) x = y;
            }
        }
    }
    if (i1 < 0) {
        x = __builtin_inff();
        for (int i = 0; i < n; ++i) {
            const float y = seg_dist2(p, vtx(poly, i), vtx(poly, i + 1 < n ? i + 1 : 0));
            if (y < x) x = y;
        }
    }
    const float d = sqrtf(x);
    return d < 1e9f ? d : 1e9f;
}

// the y-z polygon a particle in leaf pair `en` with bank `bank` is bounded by
__device__ __forceinline__ const gegs_float2 *yz_polygon(const gegs_float2 *en, int bank, int &n) {
    if (bank == 0) { n = 30; return en + 2; }
    n = 17;
    return bank == 2 ? en + 17 : en;
}

// region of a point in the MLC: W inside a leaf, air otherwise (geom.cu:486-516)
__device__ __forceinline__ uint32_t inwhere_mlc(const gegs_mlc &m, const gegs_float2 *endnodes, float qx, float qy,
                                                float qz, int &index, int &bank) {
    uint32_t inew = REG_AIR;
    if (index == OUTMLC) index = index_of_leaf(m, p2(qx, qz));
    if (index >= 0) {
        bank = point_in_leaf(p2(qy, qz), endnodes + index * 34);
        inew = bank > 0 ? REG_MLC : REG_AIR;
    }
    return inew;
}

// distance to the next MLC boundary along the flight and the region entered;
// updates the particle's leaf index, bank and, on leaving, its module
// (geom.cu:518-790)
__device__ __forceinline__ uint32_t howfar_mlc(const Env &env, Part &p, float &t) {
    const gegs_mlc &m = *env.mlc;
    const gegs_float2 *endnodes = env.endnodes + (size_t)p.job * MLC_LEAVES * 34;
    uint32_t inew = p.region;
    int bank = p.bank;
    int index = p.leaf;
    float dis_out = 0.0f;   // distance to the slab's exit in the x-z plane
    if (p.y < -m.rmax || p.y > m.rmax) return 0u;
    const P2 p1 = p2(p.x, p.z), pyz = p2(p.y, p.z);
    const P2 d1 = p2(p.u, p.w), d2 = p2(p.v, p.w);
    bool in_xz, in_yz;
    float dis_xz = ray_polygon(p1, d1, m.boundary_xz, 4, in_xz);
    float dis_yz = ray_polygon(pyz, d2, m.boundary_yz, 4, in_yz);
    if (dis_xz >= INFI_DIST || dis_yz >= INFI_DIST) return 0u;
    const float bound = dis_xz < dis_yz ? dis_xz : dis_yz;
    bool new_region = false;
    if (in_xz && in_yz) {
        dis_out = dis_xz;
    } else {
        // outside the MLC: step to its boundary
        inew = 0u;
        if (bound >= INFI_DIST) return inew;
        if (t > bound) {
            t = bound + EPSTEP;
            new_region = true;
        } else {
            return inew;
        }
    }
    if (!new_region) {
        index = p.leaf > -MLC_LEAVES ? p.leaf : index_of_leaf(m, p1);
        if (index >= 0) {
            dis_xz = ray_polygon(p1, d1, m.cross_xz + index * 16, 14, in_xz);
            int nyz;
            const gegs_float2 *yz = yz_polygon(endnodes + index * 34, p.bank, nyz);
            dis_yz = ray_polygon(pyz, d2, yz, nyz, in_yz);
            if (dis_yz > dis_xz) {
                // the side of the leaf comes first: the particle goes into the gap
                if (d1.x < 0.0f && index > 0) index = -index;
                else if (index < MLC_LEAVES - 1) index = -(index + 1);
            }
        } else if (index > -MLC_LEAVES) {
            // in a gap: search the leaves the ray can reach, those between
            // here and the exit point
            const P2 p3 = p2(p1.x + dis_out * d1.x, p1.y + (dis_out - 0.001f) * d1.y);
            int lim1 = index_of_leaf(m, p3), lim2;
            if (lim1 < 0) lim1 = -lim1;
            int sx = 1, sl = 16;
            if (d1.x < 0.0f) {
                sx = -1;
                sl = -16;
                if (lim1 > 0) lim1 -= 1;
                lim2 = -index + 1;
            } else {
                lim2 = lim1;
                lim1 = -index - 1;
            }
            int i = -index - sx;
            if (lim1 < 0) lim1 = 0;
            if (lim2 > MLC_LEAVES - 1) lim2 = MLC_LEAVES - 1;
            if (i < 0) i = 0;
            if (i > MLC_LEAVES - 1) i = MLC_LEAVES - 1;
            const gegs_float2 *leaf = m.cross_xz + i * 16;
            float tmp;
            do {
                tmp = ray_polygon(p1, d1, leaf, 14, in_xz);
                i += sx;
                leaf += sl;
            } while (i >= lim1 && i <= lim2 && tmp >= INFI_DIST);
            if (tmp < dis_xz) {
                dis_xz = tmp;
                index = i - sx;
            } else {
                index = PASSMLC;
                p.module = env.mlc_next;
            }
        }
        float dmin = dis_xz < dis_yz ? dis_xz : dis_yz;
        bool stepping_out = false;
        if (dmin + EPSTEP >= bound) {
            dmin = bound;
            stepping_out = true;
        }
        if (t > dmin) {
            t = dmin + EPSTEP;
            if (stepping_out) {
                p.leaf = PASSMLC;
                p.module = env.mlc_next;
                return REG_AIR;
            }
        } else {
            return inew;
        }
    }
    // the region at the end of the step
    const float qx = p.x + t * p.u, qy = p.y + t * p.v, qz = p.z + t * p.w;
    inew = inwhere_mlc(m, endnodes, qx, qy, qz, index, bank);
    p.leaf = index;
    p.bank = bank;
    return inew;
}

// distance to the nearest MLC boundary (geom.cu:1193-1286)
__device__ __forceinline__ float hownear_mlc(const Env &env, Part &p) {
    const gegs_mlc &m = *env.mlc;
    const gegs_float2 *endnodes = env.endnodes + (size_t)p.job * MLC_LEAVES * 34;
    const P2 p1 = p2(p.x, p.z), pyz = p2(p.y, p.z);
    float tp_xz = INFI_DIST + 1.0f, tp_yz = INFI_DIST + 1.0f;
    bool in_xz = true, in_yz = true;
    if (p.leaf < -MLC_LEAVES) {
        in_xz = point_in_polygon(p1, m.boundary_xz, 4);
        in_yz = point_in_polygon(pyz, m.boundary_yz, 4);
    }
    if (!(in_xz && in_yz)) {
        const float bxz = poly_dist(p1, m.boundary_xz, 4);
        const float byz = poly_dist(pyz, m.boundary_yz, 4);
        return bxz < byz ? bxz : byz;
    }
    int index;
    if (p.leaf > PASSMLC) {
        index = p.leaf;
    } else {
        index = index_of_leaf(m, p1);
        p.leaf = index;
    }
    if (index >= 0) {
        tp_xz = poly_dist(p1, m.cross_xz + index * 16, 14);
        if (p.bank < 0) p.bank = point_in_leaf(pyz, endnodes + index * 34);
        int nyz;
        const gegs_float2 *yz = yz_polygon(endnodes + index * 34, p.bank, nyz);
        tp_yz = poly_dist(pyz, yz, nyz);
    } else if (index > -MLC_LEAVES) {
        const int i = -index;
        const float a = poly_dist(p1, m.cross_xz + i * 16, 14);
        tp_xz = poly_dist(p1, m.cross_xz + (i - 1) * 16, 14);
        if (a < tp_xz) tp_xz = a;
    }
    return tp_xz < tp_yz ? tp_xz : tp_yz;
}

}  // namespace gegs
