/*
 * BVH2 closest-hit and any-hit traversal over 64-byte wide nodes with a per-lane LDS stack: two walks with
 * the same results, and the triangle tests and stacks that they share.
 *
 * The step-exact walk (traverse_begin / _pop / _leaf / _node) takes every step of the reference's
 * (CudaSceneClosestHit.cu:407-1186), for launches that count steps and for scenes and cameras outside
 * the other walk's range:
 *  - the slab test is the binary64 quotient widened by one ulp (:407-455);
 *  - children are pushed far-then-near with the first (lower canonical index) child winning ties
 *    (:466-512); the first child of an internal node always has the lower pre-order index;
 *  - triangles use the watertight binary32 test with binary64 re-decision of ambiguous edges
 *    (:583-824); candidates are ordered by (t, instance id, primitive id) (:873-881).
 * The reference re-tests a node's own box with the current t_max when it is popped. A node's box
 * passed its push-time test, so that pop test reduces to near <= t_max; the stack stores near
 * rounded UP to binary32 (exactly equivalent for a binary32 t_max), which lets a popped leaf go
 * straight to its triangle without fetching a node. The reference keeps one 64-entry stack per
 * structure; here TLAS and BLAS share one stack of BF_STACK_DEPTH entries, each part held to the
 * reference's 64, so a lane reports stack overflow exactly where the reference's would. Slab quotients are formed from a per-ray
 * binary64 reciprocal with one correction step, which yields the correctly rounded quotient.
 *
 * The bound walk (bound_begin / _pop / _leaf / _node), which every other launch takes, is described
 * where it begins, under "traversal on binary32 bounds".
 */
#ifndef BF_TRAVERSAL_H
#define BF_TRAVERSAL_H

#include "bf_device_math.h"
#include "bf_device_scene.h"

struct trav_ray {
    v3f o, d;
    float t_min, t_max;
    uint32_t mask;
};

struct trav_hit {
    bool present;
    float t, b0, b1, b2;
    uint32_t instance_id, primitive, scene_instance, leaf;
};

struct trav_counters {
    uint32_t nodes, triangles, instances;
};

/* Shear of the watertight triangle test for one direction (CudaSceneClosestHit.cu:694-740): the
 * dominant axis kz, the other two in winding order, and rz = 1 / d_kz, sx = d_kx rz, sy = d_ky rz.
 * `ok` is false when one of them is not finite (every triangle test then fails numerically). */
struct trav_shear {
    uint32_t kx, ky, kz;
    float rz, sx, sy;
    bool ok;
};

BF_D void make_shear(v3f d, trav_shear& s) {
    uint32_t kz = 0;
    float maxd = fabsf(d.x);
    if (fabsf(d.y) > maxd) {
        kz = 1;
        maxd = fabsf(d.y);
    }
    if (fabsf(d.z) > maxd) kz = 2;
    uint32_t kx = kz + 1;
    if (kx == 3) kx = 0;
    uint32_t ky = kx + 1;
    if (ky == 3) ky = 0;
    if (comp3(d, kz) < 0.0f) {
        const uint32_t t = kx;
        kx = ky;
        ky = t;
    }
    s.kx = kx;
    s.ky = ky;
    s.kz = kz;
    s.rz = 1.0f / comp3(d, kz);
    s.sx = comp3(d, kx) * s.rz;
    s.sy = comp3(d, ky) * s.rz;
    s.ok = bf_isfinite(s.rz) && bf_isfinite(s.sx) && bf_isfinite(s.sy);
}

/* A ray expressed in one space (world for the TLAS, an instance's object space for its BLAS),
 * with the correctly rounded binary64 reciprocal of every non-zero direction component and the
 * binary32 roundings the slab filter uses (finv, and efloor = 2^-147 max |finv|), formed once
 * instead of per node. (Keeping the triangle test's shear here as well measured slower: the
 * extra live registers spill in the traversal kernels.) */
struct trav_space {
    v3f o, d;
    double inv[3];
    float finv[3];
    float efloor;
};

/* The derived binary32 constants of a space whose o, d and inv are set. */
BF_D void finish_space(trav_space& s) {
    float inv_max = 0.0f;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        s.finv[a] = (float)s.inv[a];
        inv_max = fmaxf(inv_max, fabsf(s.finv[a]));
    }
    s.efloor = 0x1p-147f * inv_max;
}

BF_D void make_space(v3f o, v3f d, trav_space& s) {
    s.o = o;
    s.d = d;
    s.inv[0] = d.x != 0.0f ? 1.0 / (double)d.x : 0.0;
    s.inv[1] = d.y != 0.0f ? 1.0 / (double)d.y : 0.0;
    s.inv[2] = d.z != 0.0f ? 1.0 / (double)d.z : 0.0;
    finish_space(s);
}

/* a / b rounded to nearest from y = RN(1/b): q0 = RN(a y), r = a - b q0 (exact through the fma),
 * q0 + r y rounded once is RN(a / b) (Markstein's quotient correction), i.e. the same binary64
 * quotient the reference's division returns, for three fused operations instead of a division. */
BF_D double quotient(double a, double b, double y) {
    const double q0 = a * y;
    const double r = fma(-q0, b, a);
    return fma(r, y, q0);
}

/* CudaSceneClosestHit.cu:407-455 (boxes are validated finite and ordered by the host builder):
 * per axis the binary64 plane distances (lo - o) / d and (hi - o) / d, widened by one ulp. */
BF_D uint32_t slab_exact(float lx, float ly, float lz, float hx, float hy, float hz, const trav_space& s, float t_min,
                         float t_max, bool& hit, double& near_value) {
    double nv = (double)t_min;
    double fv = (double)t_max;
    const float lo[3] = {lx, ly, lz};
    const float hi[3] = {hx, hy, hz};
    const float oo[3] = {s.o.x, s.o.y, s.o.z};
    const float dd[3] = {s.d.x, s.d.y, s.d.z};
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        if (dd[a] == 0.0f) {
            if (oo[a] < lo[a] || oo[a] > hi[a]) {
                hit = false;
                return BF_HIT_MISS;
            }
            continue;
        }
        const double db = (double)dd[a];
        const double first = quotient((double)lo[a] - (double)oo[a], db, s.inv[a]);
        const double second = quotient((double)hi[a] - (double)oo[a], db, s.inv[a]);
        if (bf_isnand(first) || bf_isnand(second)) return BF_HIT_NUMERICAL_FAILURE;
        nv = fmax(nv, bf_next_down(fmin(first, second)));
        fv = fmin(fv, bf_next_up(fmax(first, second)));
        if (nv > fv) {
            hit = false;
            return BF_HIT_MISS;
        }
    }
    hit = true;
    near_value = nv;
    return BF_HIT_MISS;
}

/* A child a node step pushes: its stack entry and bounds [key_lo, key_hi] of the binary32 rounding
 * of its binary64 near value (the reference orders siblings by that rounding). */
struct child_near {
    uint2 entry;
    float key_lo, key_hi;
    uint32_t tie_axis; /* 0-2: that axis's near plane alone sets the binary64 near value; 3: t_min
                        * does; 4: not known */
    float tie_plane;   /* that plane's coordinate */
};

BF_D float round_up_float(double v) {
    float f = (float)v;
    if ((double)f < v) f = bf_next_up_f(f);
    return f;
}

/* An entry whose near word is the exact binary64 near value rounded up to binary32: visited iff it
 * is <= the current t_max, exactly the reference's pop test. */
BF_D void exact_child(uint32_t ref, double v, child_near& c) {
    c.entry = make_uint2(ref | BF_NEAR_EXACT, __float_as_uint(round_up_float(v)));
    c.key_lo = c.key_hi = (float)v;
    c.tie_axis = 4u;
    c.tie_plane = 0.0f;
}

/*
 * An entry that keeps bounds lo <= near <= hi of the binary64 near value (0 <= lo): bits 8-31 of
 * the near word hold hi rounded up to a multiple of 256 ulps (still an upper bound) and bits 0-7
 * k with 2^(k-127) >= hi' - lo, so that hi' - 2^(k-127) is a lower bound (k = 255: none kept).
 * With E the exponent field of RN(hi' - lo), 2^(E+1-127) exceeds hi' - lo itself.
 */
BF_D void bounded_child(uint32_t ref, float lo, float hi, child_near& c) {
    const uint32_t hb = (__float_as_uint(hi) + 0xFFu) & ~0xFFu;
    const uint32_t k = min((__float_as_uint(__uint_as_float(hb) - lo) >> 23) + 1u, 255u);
    c.entry = make_uint2(ref, hb | k);
    c.key_lo = lo;
    c.key_hi = hi;
}

/*
 * The same decision with a binary32 filter in front. Each binary32 plane distance
 * q~ = RN32(RN32(plane - o) * RN32(1/d)) is within 3 binary32 roundings of the exact quotient
 * (relative 3u, u = 2^-24), and the binary64 quotient and its one-ulp widening add under 2^-51
 * relative; subnormal differences add at most |1/d| 2^-149 absolutely. So every binary64
 * interval end lies within e = 4u max|q~| + max |1/d| 2^-147 + 2^-126 of its binary32 estimate,
 * and when the estimated interval is empty (or non-empty) by more than 2e the binary64 test
 * reaches the same verdict. Only a box within that band takes binary64 arithmetic; a certain hit
 * returns its near value as the binary32 interval [nv - en, nv + en], en = 4u nv + the absolute
 * terms (widened outward by one ulp each side, and never below t_min, which bounds the binary64
 * value from below).
 */
BF_D uint32_t slab(float lx, float ly, float lz, float hx, float hy, float hz, const trav_space& s, float t_min,
                   float t_max, uint32_t ref, bool& hit, child_near& near) {
    const float lo[3] = {lx, ly, lz};
    const float hi[3] = {hx, hy, hz};
    const float oo[3] = {s.o.x, s.o.y, s.o.z};
    const float dd[3] = {s.d.x, s.d.y, s.d.z};
    /* nv: the largest near estimate (t_min included), second: the next one, axis: nv's source */
    float nv = t_min, second = -BF_INFINITY_F, fv = t_max, scale = 0.0f, plane = 0.0f;
    uint32_t axis = 3u;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        if (dd[a] == 0.0f) {
            if (oo[a] < lo[a] || oo[a] > hi[a]) {
                hit = false;
                return BF_HIT_MISS;
            }
            continue;
        }
        const float inv = s.finv[a];
        const float q1 = (lo[a] - oo[a]) * inv;
        const float q2 = (hi[a] - oo[a]) * inv;
        const float qn = fminf(q1, q2);
        if (qn > nv) {
            second = nv;
            nv = qn;
            axis = (uint32_t)a;
            plane = dd[a] > 0.0f ? lo[a] : hi[a];
        } else {
            second = fmaxf(second, qn);
        }
        fv = fminf(fv, fmaxf(q1, q2));
        scale = fmaxf(scale, fmaxf(fabsf(q1), fabsf(q2)));
    }
    const float e = 4.0f * 0x1p-24f * scale + s.efloor + 0x1p-126f;
    if (bf_isfinite(e) && bf_isfinite(nv) && bf_isfinite(scale)) {
        if (nv - fv > 2.0f * e) {
            hit = false;
            return BF_HIT_MISS;
        }
        /* The near value alone has a tighter bound than the interval test: an axis whose near
         * estimate lies below t_min by more than its own error contributes t_min exactly, and every
         * other axis's near quotient is at most nv (or tiny), so its error is under 4u nv plus the
         * absolute terms. A ray nearly parallel to an axis (huge quotients there) keeps tight near
         * bounds this way. */
        const float en = 4.0f * 0x1p-24f * nv + s.efloor + 0x1p-126f;
        const float up = nv + en; /* > 0: nv >= t_min >= 0, en > 0 */
        if (fv - nv > 2.0f * e && up < 0x1p127f) {
            const float low = nv - en;
            hit = true;
            /* one ulp outward on each side (both positive where they bind) */
            bounded_child(ref, low > t_min ? __uint_as_float(__float_as_uint(low) - 1u) : t_min,
                          __uint_as_float(__float_as_uint(up) + 1u), near);
            /* every estimate is within en of its binary64 term, so a lead of more than 2 en makes
             * the source of nv the source of the binary64 near value too */
            near.tie_axis = nv - second > 2.0f * en ? axis : 4u;
            near.tie_plane = plane;
            return BF_HIT_MISS;
        }
    }
    double v = 0.0;
    const uint32_t st = slab_exact(lx, ly, lz, hx, hy, hz, s, t_min, t_max, hit, v);
    exact_child(ref, v, near);
    return st;
}

/* The binary64 near value of a box the ray is known to meet: per axis the near plane (lo for
 * d > 0, hi for d < 0; rounding is monotone) widened down by one ulp, and t_min. */
BF_D double near_exact(const float* box, const trav_space& s, float t_min) {
    const float oo[3] = {s.o.x, s.o.y, s.o.z};
    const float dd[3] = {s.d.x, s.d.y, s.d.z};
    double n = (double)t_min;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        if (dd[a] == 0.0f) continue;
        const float plane = dd[a] > 0.0f ? box[a] : box[3 + a];
        n = fmax(n, bf_next_down(quotient((double)plane - (double)oo[a], (double)dd[a], s.inv[a])));
    }
    return n;
}

/* 1: the entry's near value is <= t (visit), 0: it is > t (skip), 2: its bounds cannot tell */
BF_D uint32_t near_decision(uint2 entry, float t) {
    if (entry.x & BF_NEAR_EXACT) return __uint_as_float(entry.y) <= t ? 1u : 0u;
    const float hi = __uint_as_float(entry.y & ~0xFFu);
    if (hi <= t) return 1u;
    const uint32_t k = entry.y & 0xFFu;
    if (k != 255u && bf_next_down_f(hi - __uint_as_float(k << 23)) > t) return 0u;
    return 2u;
}

struct tri_result {
    bool hit;
    float t, b0, b1, b2;
};

/* CudaSceneClosestHit.cu:583-692 */
template <bool BARY>
BF_D uint32_t refine_edges(v3f v0, v3f v1, v3f v2, v3f o, v3f d, uint32_t kx, uint32_t ky, uint32_t kz, float t_min,
                           float t_max, tri_result& r) {
    const double dx = (double)comp3(d, kx), dy = (double)comp3(d, ky), dz = (double)comp3(d, kz);
    if (dz == 0.0) return BF_HIT_NUMERICAL_FAILURE;
    const double p0x = (double)comp3(v0, kx) - (double)comp3(o, kx);
    const double p0y = (double)comp3(v0, ky) - (double)comp3(o, ky);
    const double p0z = (double)comp3(v0, kz) - (double)comp3(o, kz);
    const double p1x = (double)comp3(v1, kx) - (double)comp3(o, kx);
    const double p1y = (double)comp3(v1, ky) - (double)comp3(o, ky);
    const double p1z = (double)comp3(v1, kz) - (double)comp3(o, kz);
    const double p2x = (double)comp3(v2, kx) - (double)comp3(o, kx);
    const double p2y = (double)comp3(v2, ky) - (double)comp3(o, ky);
    const double p2z = (double)comp3(v2, kz) - (double)comp3(o, kz);
    const double ax = p0x * dz - dx * p0z;
    const double ay = p0y * dz - dy * p0z;
    const double bx = p1x * dz - dx * p1z;
    const double by = p1y * dz - dy * p1z;
    const double cx = p2x * dz - dx * p2z;
    const double cy = p2y * dz - dy * p2z;
    const double e0 = bx * cy - by * cx;
    const double e1 = cx * ay - cy * ax;
    const double e2 = ax * by - ay * bx;
    if (!bf_isfinited(e0) || !bf_isfinited(e1) || !bf_isfinited(e2)) return BF_HIT_NUMERICAL_FAILURE;
    const bool neg = e0 < 0.0 || e1 < 0.0 || e2 < 0.0;
    const bool pos = e0 > 0.0 || e1 > 0.0 || e2 > 0.0;
    if (neg && pos) return BF_HIT_MISS;
    const double det = e0 + e1 + e2;
    if (!bf_isfinited(det)) return BF_HIT_NUMERICAL_FAILURE;
    if (det == 0.0) return BF_HIT_MISS;
    const double num = fma(e0, p0z, fma(e1, p1z, e2 * p2z));
    const double den = det * dz;
    if (!bf_isfinited(num) || !bf_isfinited(den) || den == 0.0) return BF_HIT_NUMERICAL_FAILURE;
    const double t = num / den;
    if (!BARY) {
        if (!bf_isfinited(t)) return BF_HIT_NUMERICAL_FAILURE;
        if (t < (double)t_min || t > (double)t_max) return BF_HIT_MISS;
        const float ft = (float)t;
        if (!bf_isfinite(ft)) return BF_HIT_NUMERICAL_FAILURE;
        r.hit = true;
        r.t = ft == 0.0f ? 0.0f : ft;
        return BF_HIT_MISS;
    }
    const double b0 = e0 / det, b1 = e1 / det, b2 = e2 / det;
    if (!bf_isfinited(t) || !bf_isfinited(b0) || !bf_isfinited(b1) || !bf_isfinited(b2)) return BF_HIT_NUMERICAL_FAILURE;
    if (t < (double)t_min || t > (double)t_max) return BF_HIT_MISS;
    const float ft = (float)t, f0 = (float)b0, f1 = (float)b1, f2 = (float)b2;
    if (!bf_isfinite(ft) || !bf_isfinite(f0) || !bf_isfinite(f1) || !bf_isfinite(f2)) return BF_HIT_NUMERICAL_FAILURE;
    r.hit = true;
    r.t = ft == 0.0f ? 0.0f : ft;
    r.b0 = f0 == 0.0f ? 0.0f : f0;
    r.b1 = f1 == 0.0f ? 0.0f : f1;
    r.b2 = f2 == 0.0f ? 0.0f : f2;
    return BF_HIT_MISS;
}

/* CudaSceneClosestHit.cu:694-824, with the direction's shear formed by make_shear */
template <bool BARY>
BF_D uint32_t watertight(v3f v0, v3f v1, v3f v2, v3f o, v3f d, const trav_shear& sh, float t_min, float t_max,
                         tri_result& r) {
    const uint32_t kx = sh.kx, ky = sh.ky, kz = sh.kz;
    const v3f t0 = sub3(v0, o), t1 = sub3(v1, o), t2 = sub3(v2, o);
    if (!fin3(t0) || !fin3(t1) || !fin3(t2)) return BF_HIT_NUMERICAL_FAILURE;
    const float rz = sh.rz, sx = sh.sx, sy = sh.sy;
    if (!sh.ok) return BF_HIT_NUMERICAL_FAILURE;
    const float ax = fmaf(-sx, comp3(t0, kz), comp3(t0, kx));
    const float ay = fmaf(-sy, comp3(t0, kz), comp3(t0, ky));
    const float bx = fmaf(-sx, comp3(t1, kz), comp3(t1, kx));
    const float by = fmaf(-sy, comp3(t1, kz), comp3(t1, ky));
    const float cx = fmaf(-sx, comp3(t2, kz), comp3(t2, kx));
    const float cy = fmaf(-sy, comp3(t2, kz), comp3(t2, ky));
    const float az = comp3(t0, kz) * rz;
    const float bz = comp3(t1, kz) * rz;
    const float cz = comp3(t2, kz) * rz;
    if (!bf_isfinite(ax) || !bf_isfinite(ay) || !bf_isfinite(bx) || !bf_isfinite(by) || !bf_isfinite(cx) ||
        !bf_isfinite(cy) || !bf_isfinite(az) || !bf_isfinite(bz) || !bf_isfinite(cz))
        return BF_HIT_NUMERICAL_FAILURE;
    const float e0 = bx * cy - by * cx;
    const float e1 = cx * ay - cy * ax;
    const float e2 = ax * by - ay * bx;
    if (!bf_isfinite(e0) || !bf_isfinite(e1) || !bf_isfinite(e2)) return BF_HIT_NUMERICAL_FAILURE;
    const bool neg = e0 < 0.0f || e1 < 0.0f || e2 < 0.0f;
    const bool pos = e0 > 0.0f || e1 > 0.0f || e2 > 0.0f;
    if (neg && pos) {
        /* Binary32 filter in front of the binary64 re-decision. Each sheared coordinate is within
         * 4u (u = 2^-24) of its exact value relative to m = |t_x| + |s t_z|, so each edge function
         * is within 10.001u (m_b m_c' + m_b' m_c) of the exact one, while the binary64
         * re-decision is accurate to about 2^-50 of the same terms. When one edge is negative and
         * another positive by more than 12u of that (plus subnormal floors), the binary64 signs
         * are mixed too and the ray misses exactly as refine_edges would decide. */
        const float fl = 0x1p-120f;
        const float max_ = fabsf(comp3(t0, kx)) + fabsf(sx * comp3(t0, kz)) + fl;
        const float may = fabsf(comp3(t0, ky)) + fabsf(sy * comp3(t0, kz)) + fl;
        const float mbx = fabsf(comp3(t1, kx)) + fabsf(sx * comp3(t1, kz)) + fl;
        const float mby = fabsf(comp3(t1, ky)) + fabsf(sy * comp3(t1, kz)) + fl;
        const float mcx = fabsf(comp3(t2, kx)) + fabsf(sx * comp3(t2, kz)) + fl;
        const float mcy = fabsf(comp3(t2, ky)) + fabsf(sy * comp3(t2, kz)) + fl;
        const float k = 12.0f * 0x1p-24f;
        const float b0 = k * (mbx * mcy + mby * mcx) + 0x1p-100f;
        const float b1 = k * (mcx * may + mcy * max_) + 0x1p-100f;
        const float b2 = k * (max_ * mby + may * mbx) + 0x1p-100f;
        const bool sure_neg = e0 < -b0 || e1 < -b1 || e2 < -b2;
        const bool sure_pos = e0 > b0 || e1 > b1 || e2 > b2;
        if (sure_neg && sure_pos && bf_isfinite(b0) && bf_isfinite(b1) && bf_isfinite(b2)) return BF_HIT_MISS;
    }
    if (e0 == 0.0f || e1 == 0.0f || e2 == 0.0f || (neg && pos))
        return refine_edges<BARY>(v0, v1, v2, o, d, kx, ky, kz, t_min, t_max, r);
    const float det = e0 + e1 + e2;
    if (!bf_isfinite(det)) return BF_HIT_NUMERICAL_FAILURE;
    if (det == 0.0f) return BF_HIT_MISS;
    const float sp = fmaf(e0, az, fmaf(e1, bz, e2 * cz));
    if (!bf_isfinite(sp)) return BF_HIT_NUMERICAL_FAILURE;
    const float smin = t_min * det, smax = t_max * det;
    if (bf_isnan(smin) || bf_isnan(smax)) return BF_HIT_NUMERICAL_FAILURE;
    if ((det > 0.0f && (sp < smin || sp > smax)) || (det < 0.0f && (sp > smin || sp < smax))) return BF_HIT_MISS;
    const float inv = 1.0f / det;
    const float t = sp * inv;
    if (!BARY) {
        if (!bf_isfinite(t)) return BF_HIT_NUMERICAL_FAILURE;
        if (t < t_min || t > t_max) return BF_HIT_MISS;
        r.hit = true;
        r.t = t == 0.0f ? 0.0f : t;
        return BF_HIT_MISS;
    }
    const float b0 = e0 * inv, b1 = e1 * inv, b2 = e2 * inv;
    if (!bf_isfinite(t) || !bf_isfinite(b0) || !bf_isfinite(b1) || !bf_isfinite(b2)) return BF_HIT_NUMERICAL_FAILURE;
    if (t < t_min || t > t_max) return BF_HIT_MISS;
    r.hit = true;
    r.t = t == 0.0f ? 0.0f : t;
    r.b0 = b0 == 0.0f ? 0.0f : b0;
    r.b1 = b1 == 0.0f ? 0.0f : b1;
    r.b2 = b2 == 0.0f ? 0.0f : b2;
    return BF_HIT_MISS;
}

/* CudaSceneClosestHit.cu:873-881 */
BF_D bool precedes(float t, uint32_t inst, uint32_t prim, const trav_hit& c) {
    return !c.present || t < c.t || (t == c.t && (inst < c.instance_id || (inst == c.instance_id && prim < c.primitive)));
}

/* A lane's column of a global spill area. */
struct column_spill {
    uint2* area;
    uint32_t stride;
    BF_D void put(uint32_t k, uint2 e) { area[(size_t)k * stride] = e; }
    BF_D uint2 get(uint32_t k) const { return area[(size_t)k * stride]; }
    BF_D void put(uint32_t k, uint32_t e) { area[(size_t)k * stride].x = e; }
    BF_D void get(uint32_t k, uint2& e) const { e = area[(size_t)k * stride]; }
    BF_D void get(uint32_t k, uint32_t& e) const { e = area[(size_t)k * stride].x; }
};

/* A spill area in the lane's scratch, for launches without a workspace. */
struct scratch_spill {
    uint32_t *ref, *near_word; /* BF_STACK_DEPTH words each, the lane's own */
    BF_D void put(uint32_t k, uint2 e) {
        ref[k] = e.x;
        near_word[k] = e.y;
    }
    BF_D void put(uint32_t k, uint32_t e) { ref[k] = e; }
    BF_D void get(uint32_t k, uint2& e) const { e = make_uint2(ref[k], near_word[k]); }
    BF_D void get(uint32_t k, uint32_t& e) const { e = ref[k]; }
};

/*
 * The step-exact walk's stack of (node reference, near bits) pairs. The top S entries live in LDS,
 * laid out [entry][lane] so that a wave's pushes and pops touch consecutive banks; when a push
 * finds them full, the lower half moves to the lane's spill area and comes back when the LDS part
 * runs empty (stack_refill). A lane whose cap is S never spills.
 */
template <uint32_t S, uint32_t LANES, typename Spill = column_spill>
struct trav_stack {
    uint2* lds;             /* entry k at lds[k * LANES] (LANES = lanes of the workgroup) */
    Spill spill;
    uint32_t sp, gsp;       /* entries in LDS, entries spilled */
    uint32_t cap;           /* entries the lane may hold in all: S without a spill area */
};

template <uint32_t S, uint32_t LANES, typename Spill>
BF_D uint32_t stack_depth(const trav_stack<S, LANES, Spill>& s) { return s.sp + s.gsp; }

template <uint32_t S, uint32_t LANES, typename Spill>
BF_D void stack_push(trav_stack<S, LANES, Spill>& s, uint2 entry) {
    if (S < BF_STACK_DEPTH && s.sp == S) {
#pragma unroll
        for (uint32_t k = 0; k < S / 2; ++k) s.spill.put(s.gsp + k, s.lds[k * LANES]);
#pragma unroll
        for (uint32_t k = 0; k < S / 2; ++k) s.lds[k * LANES] = s.lds[(k + S / 2) * LANES];
        s.gsp += S / 2;
        s.sp = S / 2;
    }
    s.lds[s.sp * LANES] = entry;
    ++s.sp;
}

template <uint32_t S, uint32_t LANES, typename Spill>
BF_D void stack_refill(trav_stack<S, LANES, Spill>& s) {
    if (S < BF_STACK_DEPTH && s.sp == 0u && s.gsp != 0u) {
        s.gsp -= S / 2;
#pragma unroll
        for (uint32_t k = 0; k < S / 2; ++k) s.lds[k * LANES] = s.spill.get(s.gsp + k);
        s.sp = S / 2;
    }
}

template <uint32_t S, uint32_t LANES, typename Spill>
BF_D uint2 stack_pop(trav_stack<S, LANES, Spill>& s) {
    stack_refill(s);
    --s.sp;
    return s.lds[s.sp * LANES];
}

/* Loop state of one ray's traversal between steps (the stack lives in trav_stack). */
struct trav_state {
    trav_space space;
    float t_min, t_max;
    uint32_t mask;
    uint32_t in_blas, blas_base;
    uint32_t inst_id, scene_inst;
};

/* Starts a ray: empties the stack and pushes the TLAS root when the ray meets its box. On a normal
 * return an empty stack means the ray is already done. */
template <uint32_t S, uint32_t LANES, typename Spill>
BF_D uint32_t traverse_begin(const bf_dev_scene& S_, const trav_ray& ray, trav_stack<S, LANES, Spill>& stack, trav_state& ts,
                             trav_hit& best, bool& occluded, trav_counters& ctr) {
    best.present = false;
    best.t = ray.t_max;
    occluded = false;
    stack.sp = 0u;
    stack.gsp = 0u;
    if (S_.tlas_root_ref == BF_INVALID_INDEX) return BF_HIT_MISS;
    ts.t_min = ray.t_min;
    ts.t_max = ray.t_max;
    ts.mask = ray.mask;
    ts.in_blas = 0u;
    ts.blas_base = 0u;
    ts.inst_id = 0u;
    ts.scene_inst = 0u;
    make_space(ray.o, ray.d, ts.space);
    bool h;
    child_near nv;
    const uint32_t st = slab(S_.tlas_root_box[0], S_.tlas_root_box[1], S_.tlas_root_box[2], S_.tlas_root_box[3],
                             S_.tlas_root_box[4], S_.tlas_root_box[5], ts.space, ts.t_min, ts.t_max, S_.tlas_root_ref,
                             h, nv);
    if (st != BF_HIT_MISS) return st;
    if (!h) {
        ctr.nodes++;
        return BF_HIT_MISS;
    }
    stack_push(stack, nv.entry);
    return BF_HIT_MISS;
}

/* True when the next entry is a leaf (a triangle or an instance) rather than an interior node; the
 * stack holds entries and has been refilled. */
template <uint32_t S, uint32_t LANES, typename Spill>
BF_D bool leaf_on_top(const trav_stack<S, LANES, Spill>& stack) {
    return (stack.lds[(stack.sp - 1u) * LANES].x & BF_WIDE_LEAF) != 0u;
}

/* A step is traverse_pop, then traverse_leaf or traverse_node of what it popped; the ray is done when
 * the stack is empty. Pops one entry; false when the reference would skip it. `leave(space)` forms the
 * world space again when a BLAS is left, so that no copy of it stays live between steps. */
template <bool ANY, uint32_t S, uint32_t LANES, typename Spill, typename Leave>
BF_D bool traverse_pop(const bf_dev_scene& S_, Leave leave, trav_stack<S, LANES, Spill>& stack, trav_state& ts,
                       const trav_hit& best, trav_counters& ctr, uint32_t& ref) {
    if (ts.in_blas && stack_depth(stack) <= ts.blas_base) {
        ts.in_blas = 0u;
        leave(ts.space);
    }
    const uint2 entry = stack_pop(stack);
    ref = entry.x & ~BF_NEAR_EXACT;
    ctr.nodes++;
    const float tcur = ANY ? ts.t_max : best.t;
    /* the reference's pop test: the entry's binary64 near value against the current t_max */
    const uint32_t visit = near_decision(entry, tcur);
    if (visit != 2u) return visit != 0u;
    const uint32_t index = ref & BF_REF_MASK;
    const float* box = (ref & BF_WIDE_LEAF) ? (ts.in_blas ? S_.blas_leaf_boxes : S_.tlas_leaf_boxes)
                                            : (ts.in_blas ? S_.blas_node_boxes : S_.tlas_node_boxes);
    return near_exact(box + 6 * (size_t)index, ts.space, ts.t_min) <= (double)tcur;
}

/* A popped instance entry or triangle. Returns a traversal status (BF_HIT_MISS = no error). */
template <bool ANY, uint32_t S, uint32_t LANES, typename Spill>
BF_D uint32_t traverse_leaf(const bf_dev_scene& S_, uint32_t ref, trav_stack<S, LANES, Spill>& stack, trav_state& ts,
                            trav_hit& best, bool& occluded, trav_counters& ctr) {
    const float tcur = ANY ? ts.t_max : best.t;
    const uint32_t leaf = ref & BF_REF_MASK;
    if (!ts.in_blas) {
        const bf_dev_tlas_leaf L = S_.tlas_leaves[leaf];
        if ((ts.mask & L.visibility_mask) == 0u) return BF_HIT_MISS;
        const v3f lo = xform_point(L.world_to_local, ts.space.o);
        const v3f ld = xform_vector(L.world_to_local, ts.space.d);
        if (!fin3(lo) || !fin3(ld) || (ld.x == 0.0f && ld.y == 0.0f && ld.z == 0.0f)) return BF_HIT_NUMERICAL_FAILURE;
        ctr.instances++;
        const bf_dev_blas B = S_.blases[L.blas_index];
        trav_space local;
        make_space(lo, ld, local);
        bool h;
        child_near nv;
        const uint32_t st = slab(B.root_box[0], B.root_box[1], B.root_box[2], B.root_box[3], B.root_box[4],
                                 B.root_box[5], local, ts.t_min, tcur, B.root_ref, h, nv);
        if (st != BF_HIT_MISS) return st;
        if (!h) {
            ctr.nodes++;
            return BF_HIT_MISS;
        }
        /* the BLAS root opens the BLAS part of the stack (a fresh stack in the reference) */
        if (stack_depth(stack) + 1u > stack.cap) return BF_HIT_STACK_OVERFLOW;
        ts.inst_id = L.instance_id;
        ts.scene_inst = L.scene_instance;
        ts.in_blas = 1u;
        ts.blas_base = stack_depth(stack);
        ts.space = local;
        stack_push(stack, nv.entry);
        return BF_HIT_MISS;
    }
    const float4 q0 = S_.leaf_triangles[3 * (size_t)leaf + 0];
    const float4 q1 = S_.leaf_triangles[3 * (size_t)leaf + 1];
    const float4 q2 = S_.leaf_triangles[3 * (size_t)leaf + 2];
    const uint32_t prim = __float_as_uint(q0.w);
    ctr.triangles++;
    tri_result tr;
    tr.hit = false;
    trav_shear sh;
    make_shear(ts.space.d, sh);
    const uint32_t st = watertight<false>(mk(q0.x, q0.y, q0.z), mk(q1.x, q1.y, q1.z), mk(q2.x, q2.y, q2.z), ts.space.o,
                                          ts.space.d, sh, ts.t_min, tcur, tr);
    if (st != BF_HIT_MISS) return st;
    if (!tr.hit) return BF_HIT_MISS;
    if (ANY) {
        occluded = true;
        stack.sp = 0;
        stack.gsp = 0;
        return BF_HIT_MISS;
    }
    if (!precedes(tr.t, ts.inst_id, prim, best)) return BF_HIT_MISS;
    best.present = true;
    best.t = tr.t;
    best.instance_id = ts.inst_id;
    best.primitive = prim;
    best.scene_instance = ts.scene_inst;
    best.leaf = leaf;
    return BF_HIT_MISS;
}

/* The two child boxes of a popped interior node. */
template <bool ANY, uint32_t S, uint32_t LANES, typename Spill>
BF_D uint32_t traverse_node(const bf_dev_scene& S_, uint32_t ref, trav_stack<S, LANES, Spill>& stack, trav_state& ts,
                            const trav_hit& best) {
    const float tcur = ANY ? ts.t_max : best.t;
    const bf_wide_node* nodes = ts.in_blas ? S_.blas_nodes : S_.tlas_nodes;
    const bf_wide_node N = nodes[ref];
    bool h0, h1;
    child_near n0, n1;
    uint32_t st = slab(N.lo_x[0], N.lo_y[0], N.lo_z[0], N.hi_x[0], N.hi_y[0], N.hi_z[0], ts.space, ts.t_min, tcur,
                       N.child[0], h0, n0);
    if (st != BF_HIT_MISS) return st;
    st = slab(N.lo_x[1], N.lo_y[1], N.lo_z[1], N.hi_x[1], N.hi_y[1], N.hi_z[1], ts.space, ts.t_min, tcur, N.child[1], h1,
              n1);
    if (st != BF_HIT_MISS) return st;
    if (!h0 && !h1) return BF_HIT_MISS;
    /* entries of the current structure (TLAS, or the BLAS above blas_base) against its own cap */
    const uint32_t depth = stack_depth(stack), used = ts.in_blas ? depth - ts.blas_base : depth;
    const uint32_t pushes = h0 && h1 ? 2u : 1u;
    if (used + pushes > BF_STRUCTURE_STACK || depth + pushes > stack.cap) return BF_HIT_STACK_OVERFLOW;
    if (h0 && h1) {
        /* near child first: RN32 of the binary64 near values, ties to the first child (the lower
         * canonical index). Bounds of both roundings decide it unless they overlap; then both
         * near values are formed exactly. */
        bool first_near;
        if (n0.key_hi <= n1.key_lo) first_near = true;
        else if (n0.key_lo > n1.key_hi) first_near = false;
        else if (n0.tie_axis < 4u && n0.tie_axis == n1.tie_axis && (n0.tie_axis == 3u || n0.tie_plane == n1.tie_plane))
            first_near = true; /* both near values are t_min, or the same plane's quotient: a tie */
        else {
            const float b0[6] = {N.lo_x[0], N.lo_y[0], N.lo_z[0], N.hi_x[0], N.hi_y[0], N.hi_z[0]};
            const float b1[6] = {N.lo_x[1], N.lo_y[1], N.lo_z[1], N.hi_x[1], N.hi_y[1], N.hi_z[1]};
            exact_child(N.child[0], near_exact(b0, ts.space, ts.t_min), n0);
            exact_child(N.child[1], near_exact(b1, ts.space, ts.t_min), n1);
            first_near = n0.key_lo <= n1.key_lo;
        }
        stack_push(stack, first_near ? n1.entry : n0.entry);
        stack_push(stack, first_near ? n0.entry : n1.entry);
    } else {
        stack_push(stack, h0 ? n0.entry : n1.entry);
    }
    return BF_HIT_MISS;
}

/*
 * Traverses TLAS then BLASes depth-first in the reference's order. Returns a traversal status
 * (BF_HIT_MISS = no error). The stack must be empty on entry and is empty on a normal return.
 * The winning candidate keeps (t, ids, leaf); its barycentrics are re-derived by
 * closest_hit_barycentrics from the same deterministic triangle test.
 */
template <bool ANY, uint32_t S, uint32_t LANES, typename Spill, typename Leave>
BF_D uint32_t traverse(const bf_dev_scene& S_, const trav_ray& ray, Leave leave, trav_stack<S, LANES, Spill>& stack, trav_hit& best,
                       bool& occluded, trav_counters& ctr) {
    trav_state ts;
    uint32_t st = traverse_begin(S_, ray, stack, ts, best, occluded, ctr);
    while (st == BF_HIT_MISS && stack_depth(stack) != 0u) {
        uint32_t ref;
        if (!traverse_pop<ANY>(S_, leave, stack, ts, best, ctr, ref)) continue;
        st = (ref & BF_WIDE_LEAF) ? traverse_leaf<ANY>(S_, ref, stack, ts, best, occluded, ctr)
                                  : traverse_node<ANY>(S_, ref, stack, ts, best);
    }
    return st;
}

/* ---- traversal on binary32 bounds ------------------------------------------------------------
 * The engine of every launch that does not count its steps. It returns the reference's result bit
 * for bit with far fewer operations per step than the step-exact walk above, because the exact
 * binary64 decisions are only needed where they can reach the result:
 *
 *  - A box is tested with binary32 bounds that never reject what the binary64 test accepts, so the
 *    walk enters a superset of the reference's nodes. A triangle's ancestors contain its box, and
 *    the binary64 plane distances are monotone in the plane, so a triangle the reference reaches is
 *    exactly one whose own box passes the binary64 test against [t_min, current t], inside an
 *    instance whose world box passed when it was popped. Both are decided exactly: the instance's
 *    when it is entered, the triangle's only when its test reports a hit or a failure (a
 *    triangle's box is the bounds of the vertices already in registers). Most triangle tests miss
 *    and never ask.
 *  - The order of two siblings is the reference's: RN32 of their binary64 near values, ties to the
 *    first. Bounds decide it unless they overlap; then equal planes (a tie), and last binary64.
 *
 * Error of the bounds: q~ = RN(RN(plane - o) * RN(1 / d)) is within 3u (u = 2^-24) of the exact
 * quotient plus at most 2^-149 of underflow, the binary64 quotient and its one-ulp widening add
 * less than 2^-51 relative, and x -> x (1 +- 4u) is monotone, so the bound carries over to the
 * maximum of near and the minimum of far distances. BF_SLAB_REL = 8u and BF_SLAB_ABS leave room
 * for the rounding of the comparisons themselves. An axis the ray does not move along has
 * RN(1 / d) = +-inf: its near and far quotients are -inf and +inf inside the slab, (+inf, +inf) or
 * (-inf, -inf) outside, NaN on a plane, which fmaxf / fminf ignore. A space whose numbers leave
 * the range of this analysis (subnormal or huge direction components, origins past 2^126) gets NaN
 * reciprocals that keep the direction's signs: every box is then entered, near planes are still told
 * from far ones, and every order of siblings whose near planes differ is decided in binary64.
 *
 * The launchers use this engine where the boxes' coordinates stay within 2^126, no stack can
 * overflow the reference's 64 entries (both checked when the scene is built) and t_min >= 0;
 * counting launches and everything else take the step-exact walk. */
#define BF_SLAB_REL 0x1p-21f
#define BF_SLAB_ABS 0x1p-120f
/* State references beside nodes and leaves: the ray is done (also the root reference of a scene
 * without instances), a BLAS is left, or the next entry has yet to be popped. All have BF_WIDE_LEAF
 * set. */
#define BF_TRAV_DONE 0xFFFFFFFFu
#define BF_TRAV_POP 0xFFFFFFFEu
#define BF_TRAV_LEAVE 0xFFFFFFFDu
struct bound_state {
    v3f o, inv, d;     /* the current space; d is kept for BLAS spaces only */
    float t_min, t;    /* t: the closest hit so far (any-hit: t_max) */
    uint32_t cur;      /* next reference: node, BF_WIDE_LEAF | leaf, or one of the above */
    uint32_t base;     /* stack.sp below the current structure's entries */
    uint32_t tleaf;    /* TLAS leaf of the instance being walked, BF_INVALID_INDEX in the TLAS */
    uint32_t hit_tleaf, hit_leaf; /* the closest hit: TLAS leaf and triangle */
    const bf_wide_node* nodes;
};

/* Stack of the bound walk: entry k of a lane is in LDS slot k mod S of its column while it is among
 * the top ones, in the lane's spill area otherwise. A push into a full column moves the oldest half
 * to the spill area and a pop below the column brings half back (one entry at a time, a lane working
 * around a full column pays a memory access for every push and pop: 1.7 times the vector-memory
 * instructions of a launch). `sp` and `low` (the first entry in LDS) count in units of a slot row's
 * bytes, so that a slot's address is one and-or. */
template <typename Entry, uint32_t S, uint32_t LANES, typename Spill>
struct ring_stack {
    static_assert((S & (S - 1u)) == 0u && (LANES & (LANES - 1u)) == 0u, "slots and lanes are powers of two");
    static constexpr uint32_t ROW = LANES * (uint32_t)sizeof(Entry);
    using entry = Entry;
    uint8_t* column; /* LDS rows, row 0 */
    uint32_t lane;   /* byte offset of the lane in a row */
    Spill spill;
    uint32_t sp, low;

    BF_D Entry* slot(uint32_t at) { return reinterpret_cast<Entry*>(column + ((at & ((S - 1u) * ROW)) | lane)); }
    BF_D void reset() { sp = low = 0u; }
    BF_D void push(Entry e) {
        if (sp - low == S * ROW) {
#pragma unroll
            for (uint32_t k = 0; k < S / 2u; ++k) spill.put(low / ROW + k, *slot(low + k * ROW));
            low += S / 2u * ROW;
        }
        *slot(sp) = e;
        sp += ROW;
    }
    BF_D Entry pop() {
        if (sp == low) {
            low -= S / 2u * ROW;
#pragma unroll
            for (uint32_t k = 0; k < S / 2u; ++k) spill.get(low / ROW + k, *slot(low + k * ROW));
        }
        sp -= ROW;
        return *slot(sp);
    }
};

/* Binary32 reciprocals of a direction, or NaN with the direction's signs where the bounds do not hold. */
BF_D v3f bound_reciprocals(v3f o, v3f d) {
    const float m = fmaxf(fmaxf(fabsf(d.x), fabsf(d.y)), fabsf(d.z));
    const float c = fmaxf(fmaxf(fabsf(o.x), fabsf(o.y)), fabsf(o.z));
    const bool tiny = (fabsf(d.x) < 0x1p-126f && d.x != 0.0f) || (fabsf(d.y) < 0x1p-126f && d.y != 0.0f) ||
                      (fabsf(d.z) < 0x1p-126f && d.z != 0.0f);
    v3f inv = mk(1.0f / d.x, 1.0f / d.y, 1.0f / d.z);
    if (tiny || !(m <= 0x1p126f) || !(c <= 0x1p126f)) {
        const float nan = __builtin_nanf("");
        inv = mk(copysignf(nan, d.x), copysignf(nan, d.y), copysignf(nan, d.z));
    }
    return inv;
}

/* True when an axis's near plane is its upper one: by the sign bit, which NaN reciprocals have too. */
BF_D bool descending(float inv) { return __float_as_int(inv) < 0; }

/* The binary64 verdict on a box against [t_min, t]: the reference's push and pop tests together. */
BF_D bool box_visited_exact(v3f lo, v3f hi, v3f o, v3f d, float t_min, float t) {
    trav_space s;
    make_space(o, d, s);
    bool hit = false;
    double near_value = 0.0;
    (void)slab_exact(lo.x, lo.y, lo.z, hi.x, hi.y, hi.z, s, t_min, t, hit, near_value);
    return hit && near_value <= (double)t;
}

/* True when the binary64 test certainly passes: every near bound at or below every other axis's
 * far bound (an axis's own near never exceeds its far), and the near bounds at or below t. */
BF_D bool box_visited_certain(v3f lo, v3f hi, v3f o, v3f inv, float t_min, float t) {
    const bool sx = inv.x < 0.0f, sy = inv.y < 0.0f, sz = inv.z < 0.0f;
    const float nx = fmaxf(((sx ? hi.x : lo.x) - o.x) * inv.x, -3.402823466e38f);
    const float ny = fmaxf(((sy ? hi.y : lo.y) - o.y) * inv.y, -3.402823466e38f);
    const float nz = fmaxf(((sz ? hi.z : lo.z) - o.z) * inv.z, -3.402823466e38f);
    const float fx = fminf(((sx ? lo.x : hi.x) - o.x) * inv.x, 3.402823466e38f);
    const float fy = fminf(((sy ? lo.y : hi.y) - o.y) * inv.y, 3.402823466e38f);
    const float fz = fminf(((sz ? lo.z : hi.z) - o.z) * inv.z, 3.402823466e38f);
    const float ux = fmaf(fabsf(nx), BF_SLAB_REL, nx) + BF_SLAB_ABS;
    const float uy = fmaf(fabsf(ny), BF_SLAB_REL, ny) + BF_SLAB_ABS;
    const float uz = fmaf(fabsf(nz), BF_SLAB_REL, nz) + BF_SLAB_ABS;
    const float wx = fmaf(fabsf(fx), -BF_SLAB_REL, fx) - BF_SLAB_ABS;
    const float wy = fmaf(fabsf(fy), -BF_SLAB_REL, fy) - BF_SLAB_ABS;
    const float wz = fmaf(fabsf(fz), -BF_SLAB_REL, fz) - BF_SLAB_ABS;
    return !bf_isnan(inv.x) && ux <= fminf(wy, wz) && uy <= fminf(wx, wz) && uz <= fminf(wx, wy) &&
           fmaxf(fmaxf(ux, uy), uz) <= t && t_min <= fminf(fminf(wx, wy), wz) && t_min <= t;
}

/* near_exact of a node's child k, its planes given */
BF_D double child_near_exact(v3f n, const trav_space& s, float t_min) {
    double v = (double)t_min;
    if (s.d.x != 0.0f) v = fmax(v, bf_next_down(quotient((double)n.x - (double)s.o.x, (double)s.d.x, s.inv[0])));
    if (s.d.y != 0.0f) v = fmax(v, bf_next_down(quotient((double)n.y - (double)s.o.y, (double)s.d.y, s.inv[1])));
    if (s.d.z != 0.0f) v = fmax(v, bf_next_down(quotient((double)n.z - (double)s.o.z, (double)s.d.z, s.inv[2])));
    return v;
}

/* A stack entry of a closest-hit walk is (reference, near bound); any-hit walks, whose t never
 * shrinks, keep the reference alone. */
BF_D void push_entry(uint2& e, uint32_t ref, float lo) { e = make_uint2(ref, __float_as_uint(lo)); }
BF_D void push_entry(uint32_t& e, uint32_t ref, float) { e = ref; }
BF_D uint32_t entry_ref(uint2 e) { return e.x; }
BF_D uint32_t entry_ref(uint32_t e) { return e; }
BF_D bool entry_live(uint2 e, float t) { return !(__uint_as_float(e.y) > t); }
BF_D bool entry_live(uint32_t, float) { return true; }

template <typename Stack>
BF_D void push_ref(Stack& stack, uint32_t ref, float lo) {
    typename Stack::entry e;
    push_entry(e, ref, lo);
    stack.push(e);
}

/* Back to world space: `cache` holds the lane's world-space o and 1/d, six floats with the given
 * stride. */
BF_D void bound_leave(const bf_dev_scene& S_, bound_state& ts, const float* cache, uint32_t stride) {
    ts.o = mk(cache[0], cache[stride], cache[2u * stride]);
    ts.inv = mk(cache[3u * stride], cache[4u * stride], cache[5u * stride]);
    ts.nodes = S_.tlas_nodes;
    ts.tleaf = BF_INVALID_INDEX;
    ts.base = 0u;
}

/* Takes the next entry that can still hold a closer hit where one is due (ts.cur is BF_TRAV_POP),
 * leaving the BLAS on the way. Any-hit walks find the ends of the BLAS and of the ray as entries of
 * their own (16 half-size slots have room for them: 49.3 ms of shadow rays in the 1080p x 64 frame,
 * 52.5 with a compare against the structure's first entry); closest-hit walks compare, since two
 * entries more of their 8 slots spill more often (98.3 ms of closest-hit rays, 102.9 with entries). */
template <bool ANY, typename Stack>
BF_D void bound_pop(const bf_dev_scene& S_, Stack& stack, bound_state& ts, const float* cache, uint32_t stride) {
    while (ts.cur == BF_TRAV_POP) {
        if constexpr (ANY) {
            const auto e = stack.pop();
            const uint32_t ref = entry_ref(e);
            if (ref == BF_TRAV_LEAVE) bound_leave(S_, ts, cache, stride);
            else if (entry_live(e, ts.t)) ts.cur = ref;
        } else {
            if (stack.sp == ts.base) {
                if (ts.tleaf == BF_INVALID_INDEX) ts.cur = BF_TRAV_DONE;
                else bound_leave(S_, ts, cache, stride);
            } else {
                const auto e = stack.pop();
                if (entry_live(e, ts.t)) ts.cur = entry_ref(e);
            }
        }
    }
}

/* Starts a ray (its world-space o and 1/d go to the lane's cache). */
template <bool ANY, typename Stack>
BF_D void bound_begin(const bf_dev_scene& S_, v3f o, v3f d, float t_min, float t_max, Stack& stack, bound_state& ts,
                      float* cache, uint32_t stride) {
    stack.reset();
    ts.base = 0u;
    if constexpr (ANY) push_ref(stack, BF_TRAV_DONE, -BF_INFINITY_F);
    ts.o = o;
    ts.inv = bound_reciprocals(o, d);
    cache[0] = o.x;
    cache[stride] = o.y;
    cache[2u * stride] = o.z;
    cache[3u * stride] = ts.inv.x;
    cache[4u * stride] = ts.inv.y;
    cache[5u * stride] = ts.inv.z;
    ts.t_min = t_min;
    ts.t = t_max;
    ts.tleaf = BF_INVALID_INDEX;
    ts.hit_leaf = BF_INVALID_INDEX;
    ts.hit_tleaf = BF_INVALID_INDEX;
    ts.nodes = S_.tlas_nodes;
    ts.cur = S_.tlas_root_ref; /* BF_INVALID_INDEX (no instances) is BF_TRAV_DONE */
}

/* The two child boxes of node ts.cur: the near child becomes ts.cur, the far one is pushed. */
template <typename Stack, typename WorldRay>
BF_D void bound_node(WorldRay world, Stack& stack, bound_state& ts) {
    const float4* p = reinterpret_cast<const float4*>(ts.nodes + ts.cur);
    const float4 a = p[0], b = p[1], c = p[2];
    const uint2 child = *reinterpret_cast<const uint2*>(p + 3);
    const bool sx = descending(ts.inv.x), sy = descending(ts.inv.y), sz = descending(ts.inv.z);
    /* a: lo_x lo_y, b: lo_z hi_x, c: hi_y hi_z, each for both children */
    const v3f n0 = mk(sx ? b.z : a.x, sy ? c.x : a.z, sz ? c.z : b.x);
    const v3f n1 = mk(sx ? b.w : a.y, sy ? c.y : a.w, sz ? c.w : b.y);
    const v3f f0 = mk(sx ? a.x : b.z, sy ? a.z : c.x, sz ? b.x : c.z);
    const v3f f1 = mk(sx ? a.y : b.w, sy ? a.w : c.y, sz ? b.y : c.w);
    const v3f q0 = mk((n0.x - ts.o.x) * ts.inv.x, (n0.y - ts.o.y) * ts.inv.y, (n0.z - ts.o.z) * ts.inv.z);
    const v3f q1 = mk((n1.x - ts.o.x) * ts.inv.x, (n1.y - ts.o.y) * ts.inv.y, (n1.z - ts.o.z) * ts.inv.z);
    const v3f r0 = mk((f0.x - ts.o.x) * ts.inv.x, (f0.y - ts.o.y) * ts.inv.y, (f0.z - ts.o.z) * ts.inv.z);
    const v3f r1 = mk((f1.x - ts.o.x) * ts.inv.x, (f1.y - ts.o.y) * ts.inv.y, (f1.z - ts.o.z) * ts.inv.z);
    const float nv0 = fmaxf(fmaxf(fmaxf(q0.x, q0.y), q0.z), ts.t_min);
    const float nv1 = fmaxf(fmaxf(fmaxf(q1.x, q1.y), q1.z), ts.t_min);
    const float fv0 = fminf(fminf(fminf(r0.x, r0.y), r0.z), ts.t);
    const float fv1 = fminf(fminf(fminf(r1.x, r1.y), r1.z), ts.t);
    const float lo0 = fmaf(nv0, 1.0f - BF_SLAB_REL, -BF_SLAB_ABS);
    const float lo1 = fmaf(nv1, 1.0f - BF_SLAB_REL, -BF_SLAB_ABS);
    const bool h0 = !(lo0 > fmaf(fv0, 1.0f + BF_SLAB_REL, BF_SLAB_ABS));
    const bool h1 = !(lo1 > fmaf(fv1, 1.0f + BF_SLAB_REL, BF_SLAB_ABS));
    const bool both = h0 && h1;
    const float lead = nv1 - nv0;
    bool first = both ? lead > 0.0f : h0;
    if (both && !(fabsf(lead) > fmaf(nv0 + nv1, BF_SLAB_REL, 4.0f * BF_SLAB_ABS))) {
        /* a tie when each axis has equal near planes or lies below both near values */
        const float below = fmaf(fminf(nv0, nv1), 1.0f - 2.0f * BF_SLAB_REL, -4.0f * BF_SLAB_ABS);
        const float up = 1.0f + BF_SLAB_REL;
        const bool tie = (n0.x == n1.x || fmaxf(q0.x, q1.x) * up < below) &&
                         (n0.y == n1.y || fmaxf(q0.y, q1.y) * up < below) &&
                         (n0.z == n1.z || fmaxf(q0.z, q1.z) * up < below);
        first = true;
        if (!tie) {
            v3f d = ts.d;
            uint32_t mask;
            if (ts.tleaf == BF_INVALID_INDEX) world(d, mask);
            trav_space s;
            make_space(ts.o, d, s);
            first = (float)child_near_exact(n0, s, ts.t_min) <= (float)child_near_exact(n1, s, ts.t_min);
        }
    }
    if (both) push_ref(stack, first ? child.y : child.x, first ? lo1 : lo0);
    ts.cur = first ? child.x : child.y;
    if (!h0 && !h1) ts.cur = BF_TRAV_POP;
}

/* watertight<false> with the same verdict and t for fewer operations: non-finite terms are looked
 * for once (an infinite or NaN input makes one of the six values non-finite), and the binary64
 * re-decision of mixed edge signs is filtered with one bound for the three edges. */
BF_D uint32_t watertight_bound(v3f v0, v3f v1, v3f v2, v3f o, v3f d, v3f inv, float t_min, float t_max, tri_result& r) {
    uint32_t kz = 0u;
    float maxd = fabsf(d.x);
    if (fabsf(d.y) > maxd) {
        kz = 1u;
        maxd = fabsf(d.y);
    }
    if (fabsf(d.z) > maxd) kz = 2u;
    uint32_t kx = kz == 2u ? 0u : kz + 1u;
    uint32_t ky = kx == 2u ? 0u : kx + 1u;
    const float dz = comp3(d, kz);
    if (dz < 0.0f) {
        const uint32_t t = kx;
        kx = ky;
        ky = t;
    }
    /* 1 / d_kz as the space already holds it */
    float rz = comp3(inv, kz);
    if (bf_isnan(rz)) rz = 1.0f / dz;
    const float sx = comp3(d, kx) * rz, sy = comp3(d, ky) * rz;
    const v3f t0 = sub3(v0, o), t1 = sub3(v1, o), t2 = sub3(v2, o);
    const float t0x = comp3(t0, kx), t0y = comp3(t0, ky), t0z = comp3(t0, kz);
    const float t1x = comp3(t1, kx), t1y = comp3(t1, ky), t1z = comp3(t1, kz);
    const float t2x = comp3(t2, kx), t2y = comp3(t2, ky), t2z = comp3(t2, kz);
    const float ax = fmaf(-sx, t0z, t0x), ay = fmaf(-sy, t0z, t0y);
    const float bx = fmaf(-sx, t1z, t1x), by = fmaf(-sy, t1z, t1y);
    const float cx = fmaf(-sx, t2z, t2x), cy = fmaf(-sy, t2z, t2y);
    const float az = t0z * rz, bz = t1z * rz, cz = t2z * rz;
    const float e0 = bx * cy - by * cx;
    const float e1 = cx * ay - cy * ax;
    const float e2 = ax * by - ay * bx;
    if (!__builtin_isfinite(e0) || !__builtin_isfinite(e1) || !__builtin_isfinite(e2) || !__builtin_isfinite(az) ||
        !__builtin_isfinite(bz) || !__builtin_isfinite(cz))
        return BF_HIT_NUMERICAL_FAILURE;
    const float emin = fminf(fminf(e0, e1), e2), emax = fmaxf(fmaxf(e0, e1), e2);
    const bool mixed = emin < 0.0f && emax > 0.0f;
    if (mixed) {
        /* Binary32 filter in front of the binary64 re-decision (u = 2^-24). With M at least every
         * |t_x| + |s t_z| (|s| <= 1 + 3u), a sheared coordinate is within 4.1u M of its exact value;
         * with R the largest of the six, an edge function is then within 4 R 4.1u M + 2 (4.1u M)^2
         * of the exact one for its inputs' errors and 4.1u R^2 for its own roundings, and the
         * binary64 edge functions (the exact ones times d_kz^2) within 2^-48 of the same terms.
         * Signs beyond 25u M (R + 25u M) are therefore the binary64 signs. R, the distance of the
         * triangle's edges from the ray, and not M, the distance of the ray's origin, keeps this
         * tight for small far triangles: with M^2 for R M about half the far tests went to binary64. */
        const float M = fmaxf(fmaxf(fmaxf(fabsf(t0x), fabsf(t1x)), fabsf(t2x)),
                              fmaxf(fmaxf(fabsf(t0y), fabsf(t1y)), fabsf(t2y))) +
                        fmaxf(fmaxf(fabsf(t0z), fabsf(t1z)), fabsf(t2z)) + 0x1p-60f;
        const float R = fmaxf(fmaxf(fmaxf(fabsf(ax), fabsf(bx)), fabsf(cx)), fmaxf(fmaxf(fabsf(ay), fabsf(by)), fabsf(cy)));
        const float m = M * (25.0f * 0x1p-24f);
        const float bound = fmaf(m, R + m, 0x1p-100f);
        if (emin < -bound && emax > bound) return BF_HIT_MISS;
    }
    if (mixed || emin == 0.0f || emax == 0.0f)
        return refine_edges<false>(v0, v1, v2, o, d, kx, ky, kz, t_min, t_max, r);
    const float det = e0 + e1 + e2;
    if (!bf_isfinite(det)) return BF_HIT_NUMERICAL_FAILURE;
    if (det == 0.0f) return BF_HIT_MISS;
    const float sp = fmaf(e0, az, fmaf(e1, bz, e2 * cz));
    if (!bf_isfinite(sp)) return BF_HIT_NUMERICAL_FAILURE;
    const float smin = t_min * det, smax = t_max * det;
    if (bf_isnan(smin) || bf_isnan(smax)) return BF_HIT_NUMERICAL_FAILURE;
    if ((det > 0.0f && (sp < smin || sp > smax)) || (det < 0.0f && (sp > smin || sp < smax))) return BF_HIT_MISS;
    const float rcp = 1.0f / det;
    const float t = sp * rcp;
    if (!bf_isfinite(t)) return BF_HIT_NUMERICAL_FAILURE;
    if (t < t_min || t > t_max) return BF_HIT_MISS;
    r.hit = true;
    r.t = t == 0.0f ? 0.0f : t;
    return BF_HIT_MISS;
}

/* The leaf ts.cur: an instance is entered, a triangle is tested. Returns a traversal status;
 * `occluded` is set by an any-hit walk, whose ray is then done. */
template <bool ANY, typename Stack, typename WorldRay>
BF_D uint32_t bound_leaf(const bf_dev_scene& S_, WorldRay world, Stack& stack, bound_state& ts, bool& occluded) {
    const uint32_t leaf = ts.cur & BF_REF_MASK;
    ts.cur = BF_TRAV_POP;
    if (ts.tleaf == BF_INVALID_INDEX) {
        const bf_dev_tlas_leaf& L = S_.tlas_leaves[leaf];
        v3f d;
        uint32_t mask;
        world(d, mask);
        const v3f lo = mk(L.box[0], L.box[1], L.box[2]), hi = mk(L.box[3], L.box[4], L.box[5]);
        const v3f po = xform_point(L.world_to_local, ts.o), pd = xform_vector(L.world_to_local, d);
        bool enter = (mask & L.visibility_mask) != 0u;
        if (enter && !box_visited_certain(lo, hi, ts.o, ts.inv, ts.t_min, ts.t))
            enter = box_visited_exact(lo, hi, ts.o, d, ts.t_min, ts.t);
        if (enter) {
            if (!fin3(po) || !fin3(pd) || (pd.x == 0.0f && pd.y == 0.0f && pd.z == 0.0f)) return BF_HIT_NUMERICAL_FAILURE;
            ts.o = po;
            ts.d = pd;
            ts.inv = bound_reciprocals(po, pd);
            ts.tleaf = leaf;
            ts.base = stack.sp;
            if constexpr (ANY) push_ref(stack, BF_TRAV_LEAVE, 0.0f);
            ts.nodes = S_.blas_nodes;
            ts.cur = L.root_ref;
            return BF_HIT_MISS;
        }
    } else {
        const float4 w0 = S_.leaf_triangles[3 * (size_t)leaf + 0];
        const float4 w1 = S_.leaf_triangles[3 * (size_t)leaf + 1];
        const float4 w2 = S_.leaf_triangles[3 * (size_t)leaf + 2];
        const v3f v0 = mk(w0.x, w0.y, w0.z), v1 = mk(w1.x, w1.y, w1.z), v2 = mk(w2.x, w2.y, w2.z);
        tri_result tr;
        tr.hit = false;
        const uint32_t st = watertight_bound(v0, v1, v2, ts.o, ts.d, ts.inv, ts.t_min, ts.t, tr);
        if (st != BF_HIT_MISS || tr.hit) {
            const v3f lo = mk(fminf(fminf(v0.x, v1.x), v2.x), fminf(fminf(v0.y, v1.y), v2.y), fminf(fminf(v0.z, v1.z), v2.z));
            const v3f hi = mk(fmaxf(fmaxf(v0.x, v1.x), v2.x), fmaxf(fmaxf(v0.y, v1.y), v2.y), fmaxf(fmaxf(v0.z, v1.z), v2.z));
            if (box_visited_certain(lo, hi, ts.o, ts.inv, ts.t_min, ts.t) ||
                box_visited_exact(lo, hi, ts.o, ts.d, ts.t_min, ts.t)) {
                if (st != BF_HIT_MISS) return st;
                if (ANY) {
                    occluded = true;
                    ts.cur = BF_TRAV_DONE;
                    return BF_HIT_MISS;
                }
                /* precedes(): by t, then instance id, then primitive */
                bool closer = ts.hit_leaf == BF_INVALID_INDEX || tr.t < ts.t;
                if (!closer && tr.t == ts.t) {
                    const uint32_t i0 = S_.tlas_leaves[ts.tleaf].instance_id, i1 = S_.tlas_leaves[ts.hit_tleaf].instance_id;
                    closer = i0 < i1 || (i0 == i1 && __float_as_uint(w0.w) <
                                                         __float_as_uint(S_.leaf_triangles[3 * (size_t)ts.hit_leaf].w));
                }
                if (closer) {
                    ts.t = tr.t;
                    ts.hit_leaf = leaf;
                    ts.hit_tleaf = ts.tleaf;
                }
            }
        }
    }
    return BF_HIT_MISS;
}

/* The closest hit of a finished walk in the form closest_hit_barycentrics takes. */
BF_D void bound_result(const bf_dev_scene& S_, const bound_state& ts, trav_hit& best) {
    best.present = ts.hit_leaf != BF_INVALID_INDEX;
    if (!best.present) return;
    best.t = ts.t;
    best.leaf = ts.hit_leaf;
    best.instance_id = S_.tlas_leaves[ts.hit_tleaf].instance_id;
    best.scene_instance = S_.tlas_leaves[ts.hit_tleaf].scene_instance;
    best.primitive = __float_as_uint(S_.leaf_triangles[3 * (size_t)ts.hit_leaf].w);
}

/* Barycentrics of the winning candidate: the triangle test is a pure function of the triangle, the
 * object-space ray and the parameter range, and the winner passed it within [t_min, t_max] of the
 * ray (re-testing against its own t could fail: the range test compares sp with t_max * det
 * before the division that produces t). */
BF_D uint32_t closest_hit_barycentrics(const bf_dev_scene& S, v3f o, v3f d, float t_min, float t_max, trav_hit& best) {
    const float* m = S.instances[best.scene_instance].world_to_local;
    const v3f lo = xform_point(m, o), ld = xform_vector(m, d);
    const float4 q0 = S.leaf_triangles[3 * (size_t)best.leaf + 0];
    const float4 q1 = S.leaf_triangles[3 * (size_t)best.leaf + 1];
    const float4 q2 = S.leaf_triangles[3 * (size_t)best.leaf + 2];
    tri_result tr;
    tr.hit = false;
    trav_shear sh;
    make_shear(ld, sh);
    const uint32_t st = watertight<true>(mk(q0.x, q0.y, q0.z), mk(q1.x, q1.y, q1.z), mk(q2.x, q2.y, q2.z), lo, ld, sh,
                                         t_min, t_max, tr);
    if (st != BF_HIT_MISS) return st;
    if (!tr.hit || tr.t != best.t) return BF_HIT_NUMERICAL_FAILURE;
    best.b0 = tr.b0;
    best.b1 = tr.b1;
    best.b2 = tr.b2;
    return BF_HIT_MISS;
}

/* CudaSceneClosestHit.cu:826-871 */
BF_D bool world_normal(const float* m, v3f l0, v3f l1, v3f l2, v3f& n) {
    const v3f w0 = xform_point(m, l0), w1 = xform_point(m, l1), w2 = xform_point(m, l2);
    if (!fin3(w0) || !fin3(w1) || !fin3(w2)) return false;
    const v3f f = sub3(w1, w0), s = sub3(w2, w0);
    if (!fin3(f) || !fin3(s)) return false;
    const double cx = (double)f.y * (double)s.z - (double)f.z * (double)s.y;
    const double cy = (double)f.z * (double)s.x - (double)f.x * (double)s.z;
    const double cz = (double)f.x * (double)s.y - (double)f.y * (double)s.x;
    const double mx = fmax(fabs(cx), fmax(fabs(cy), fabs(cz)));
    if (!bf_isfinited(cx) || !bf_isfinited(cy) || !bf_isfinited(cz) || !bf_isfinited(mx) || mx == 0.0) return false;
    const double sx = cx / mx, sy = cy / mx, sz = cz / mx;
    const double len = sqrt(sx * sx + sy * sy + sz * sz);
    if (!bf_isfinited(len) || len == 0.0) return false;
    n = mk((float)(sx / len), (float)(sy / len), (float)(sz / len));
    return fin3(n);
}

/* CudaSceneClosestHit.cu:397-405 */
BF_D bool valid_traversal_ray(const bf_transport_ray& r) {
    const v3f o = mk(r.origin_x, r.origin_y, r.origin_z);
    const v3f d = mk(r.direction_x, r.direction_y, r.direction_z);
    return fin3(o) && fin3(d) && (d.x != 0.0f || d.y != 0.0f || d.z != 0.0f) && bf_isfinite(r.t_min) && r.t_min >= 0.0f &&
           !bf_isnan(r.t_max) && r.t_max >= r.t_min && bf_isfinite(r.time) && r.time >= 0.0f && r.time <= 1.0f &&
           r.reserved == 0u;
}

#endif
