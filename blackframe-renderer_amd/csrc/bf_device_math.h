/*
 * Device scalar library of the HIP wavefront backend: vectors, sampling, checked products, MIS,
 * Russian roulette and the closure lobes. Each function states the reference function whose
 * arithmetic it reproduces operation for operation (file:line relative to the reference root);
 * compiled with -ffp-contract=off so that only the explicit fmaf calls fuse.
 */
#ifndef BF_DEVICE_MATH_H
#define BF_DEVICE_MATH_H

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/blackframe_hip_abi.h"
#include "../../include/blackframe_math.h"

#define BF_D __device__ __forceinline__

#define BF_EPS 0x1p-23f
#define BF_DENORM_MIN 0x1p-149f
#define BF_PI 3.14159265358979323846f
#define BF_INV_PI 0.31830988618379067154f
#define BF_QUARTER_PI 0.78539816339744830962f

#define BF_DIM_RASTER_X 0xA24BAED4963EE407ull
#define BF_DIM_RASTER_Y 0x9FB21C651E98DF25ull

enum { BF_L_OK = 0, BF_L_INVALID = 1, BF_L_NOT_REPRESENTABLE = 2, BF_L_OUTSIDE = 3 };

struct v3f {
    float x, y, z;
};

BF_D v3f mk(float x, float y, float z) { return v3f{x, y, z}; }
BF_D bool fin3(v3f v) { return (bool)(bf_isfinite(v.x) & bf_isfinite(v.y) & bf_isfinite(v.z)); }
BF_D v3f add3(v3f a, v3f b) { return mk(a.x + b.x, a.y + b.y, a.z + b.z); }
BF_D v3f sub3(v3f a, v3f b) { return mk(a.x - b.x, a.y - b.y, a.z - b.z); }
BF_D v3f mul3(v3f a, float s) { return mk(a.x * s, a.y * s, a.z * s); }
/* CudaWavefrontStages.cu:314-324 */
BF_D float dot3(v3f a, v3f b) { return fmaf(a.x, b.x, fmaf(a.y, b.y, a.z * b.z)); }
BF_D v3f cross3(v3f a, v3f b) {
    return mk(fmaf(a.y, b.z, -a.z * b.y), fmaf(a.z, b.x, -a.x * b.z), fmaf(a.x, b.y, -a.y * b.x));
}
BF_D float comp3(v3f v, uint32_t a) { return a == 0 ? v.x : (a == 1 ? v.y : v.z); }
BF_D void set3(v3f& v, uint32_t a, float value) {
    if (a == 0) v.x = value;
    else if (a == 1) v.y = value;
    else v.z = value;
}
/* CudaSceneClosestHit.cu:514-536 */
BF_D v3f xform_point(const float* m, v3f p) {
    return mk(fmaf(m[0], p.x, fmaf(m[1], p.y, fmaf(m[2], p.z, m[3]))),
              fmaf(m[4], p.x, fmaf(m[5], p.y, fmaf(m[6], p.z, m[7]))),
              fmaf(m[8], p.x, fmaf(m[9], p.y, fmaf(m[10], p.z, m[11]))));
}
BF_D v3f xform_vector(const float* m, v3f v) {
    return mk(fmaf(m[0], v.x, fmaf(m[1], v.y, m[2] * v.z)), fmaf(m[4], v.x, fmaf(m[5], v.y, m[6] * v.z)),
              fmaf(m[8], v.x, fmaf(m[9], v.y, m[10] * v.z)));
}

/* ---- sampling: SampleStreamDevice.cuh:12-33, OwenScrambling.cpp:8-43 ----------------------- */
BF_D uint64_t mix_bits(uint64_t v) {
    v ^= v >> 30;
    v *= 0xBF58476D1CE4E5B9ull;
    v ^= v >> 27;
    v *= 0x94D049BB133111EBull;
    return v ^ (v >> 31);
}

struct sample_key {
    uint32_t px, py;
    uint64_t s, seed;
};

BF_D uint64_t indexed_bits(const sample_key& k, uint64_t dim) {
    const uint64_t packed = ((uint64_t)k.px << 32) | (uint64_t)k.py;
    uint64_t state = mix_bits(k.seed ^ 0x9E3779B97F4A7C15ull);
    state = mix_bits(state ^ packed ^ 0xD1B54A32D192ED03ull);
    state = mix_bits(state ^ k.s ^ 0x8CB92BA72F3D8DD7ull);
    return mix_bits(state ^ dim);
}

struct sampler_ctx {
    uint32_t kind;
    uint32_t sobol_dims;
    const uint32_t* directions; /* [dimension][64]: the 24 leading bits of each direction number */
    const uint64_t* dimension_keys; /* [dimension]: mix_bits(dimension + 1) */
};

/*
 * Owen-scrambled Sobol, evaluated only to the 24 leading bits the binary32 sample keeps: the nested
 * scramble of OwenScrambling.cpp:22-36 decides output bit 63-d from input bits above it, so depths
 * 24..63 never reach (bits >> 40), and bits above 24 of the direction numbers suffice. The scramble's
 * flips are what a light or closure sample costs (24 64-bit hashes a dimension, about a fifth of the
 * shade stage's vector cycles), so each is cut to what its one result bit needs.
 */
struct owen_stream {
    uint32_t input;     /* Sobol point, 24 bits */
    uint32_t key_low;   /* the hash input of node n is (key ^ key >> 30) ^ n: n stays in the low word */
    uint64_t product;   /* its high word's share of the first product */
};

BF_D bool owen_open(const sampler_ctx& sc, const sample_key& k, uint64_t sobol_dim, owen_stream& o) {
    if (sobol_dim >= sc.sobol_dims) return false;
    const uint64_t gray = k.s ^ (k.s >> 1);
    const uint32_t* d = sc.directions + (uint32_t)sobol_dim * 64u;
    /* the first eight bits of the index (frames of up to 256 samples) without a loop of dependent loads */
    const uint4 d0 = reinterpret_cast<const uint4*>(d)[0], d1 = reinterpret_cast<const uint4*>(d)[1];
    const uint32_t low = (uint32_t)gray;
    const uint32_t bits[8] = {d0.x, d0.y, d0.z, d0.w, d1.x, d1.y, d1.z, d1.w};
    uint32_t point = 0u;
#pragma unroll
    for (uint32_t b = 0; b < 8u; ++b) point ^= bits[b] & (uint32_t)__builtin_amdgcn_sbfe((int)low, b, 1u);
    for (uint64_t rest = gray & ~0xFFull; rest != 0u; rest &= rest - 1u) point ^= d[__builtin_ctzll(rest)];
    const uint64_t packed = ((uint64_t)k.px << 32) | (uint64_t)k.py;
    const uint64_t key = mix_bits(k.seed ^ sc.dimension_keys[(uint32_t)sobol_dim]) ^ mix_bits(packed);
    const uint64_t first = key ^ (key >> 30); /* nodes have 25 bits: they never reach this shift */
    o.input = point;
    o.key_low = (uint32_t)first;
    o.product = (uint64_t)((uint32_t)(first >> 32) * 0x1CE4E5B9u) << 32;
    return true;
}

/* Sample bit of one depth: the input's bit flipped by bit 63 of mix_bits(key ^ node), node = 1 followed by
 * the input's leading bits. The last xor-shift of mix_bits leaves bit 63 alone, and of the last
 * product only the high word is formed. Returns it in bit 31. */
BF_D uint32_t owen_flip(const owen_stream& o, uint32_t depth) {
    const uint32_t v = o.key_low ^ ((o.input | 0x1000000u) >> (24u - depth));
    const uint64_t w = (uint64_t)v * 0x1CE4E5B9u + o.product;
    const uint32_t wl = (uint32_t)w, wh = (uint32_t)(w >> 32) + v * 0xBF58476Du;
    const uint32_t xl = wl ^ __builtin_amdgcn_alignbit(wh, wl, 27u), xh = wh ^ (wh >> 27);
    return __umulhi(xl, 0x133111EBu) + xl * 0x94D049BBu + xh * 0x133111EBu;
}

/* Sample bits of depths [FROM, TO) (leading bit first), in the low TO - FROM bits. Rolled loops: the
 * shade kernels are longer than the instruction cache. */
template <uint32_t FROM, uint32_t TO>
BF_D uint32_t owen_bits(const owen_stream& o) {
    uint32_t flips = 0u;
#pragma unroll 4
    for (uint32_t depth = FROM; depth < TO; ++depth) flips = (flips << 1) | (owen_flip(o, depth) >> 31);
    return ((o.input >> (24u - TO)) & ((1u << (TO - FROM)) - 1u)) ^ flips;
}

BF_D uint64_t sobol_dimension(uint64_t dim) {
    return dim == BF_DIM_RASTER_X ? 0ull : (dim == BF_DIM_RASTER_Y ? 1ull : dim + 2u);
}

/* One transport dimension -> binary32 in [0, 1): (bits >> 40) * 2^-24 (SampleStreamDevice.cuh:29-32). */
BF_D float sample_1d(const sampler_ctx& sc, const sample_key& k, uint64_t dim) {
    if (sc.kind == BF_SAMPLER_SOBOL_OWEN) {
        owen_stream o;
        return owen_open(sc, k, sobol_dimension(dim), o) ? (float)owen_bits<0u, 24u>(o) * 0x1p-24f : -1.0f;
    }
    return (float)(indexed_bits(k, dim) >> 40) * 0x1p-24f;
}

/* sample_1d of several dimensions, their scrambles in one loop. */
template <int COUNT>
BF_D void sample_each(const sampler_ctx& sc, const sample_key& k, const uint64_t* dims, float* out) {
    if (sc.kind == BF_SAMPLER_SOBOL_OWEN) {
        owen_stream o[COUNT];
        bool ok[COUNT];
        uint32_t flips[COUNT];
#pragma unroll
        for (int j = 0; j < COUNT; ++j) {
            o[j] = owen_stream{0u, 0u, 0u};
            ok[j] = owen_open(sc, k, sobol_dimension(dims[j]), o[j]);
            flips[j] = 0u;
        }
#pragma unroll 1
        for (uint32_t depth = 0; depth < 24u; ++depth)
#pragma unroll
            for (int j = 0; j < COUNT; ++j) flips[j] = (flips[j] << 1) | (owen_flip(o[j], depth) >> 31);
#pragma unroll
        for (int j = 0; j < COUNT; ++j) out[j] = ok[j] ? (float)(o[j].input ^ flips[j]) * 0x1p-24f : -1.0f;
        return;
    }
#pragma unroll
    for (int j = 0; j < COUNT; ++j) out[j] = (float)(indexed_bits(k, dims[j]) >> 40) * 0x1p-24f;
}

/* sample_1d(dim) < p, formed from as many leading bits as decide it (eight, but for one lane in
 * 256); false when the dimension has no sample. */
BF_D bool sample_below(const sampler_ctx& sc, const sample_key& k, uint64_t dim, float p, bool& below) {
    if (sc.kind == BF_SAMPLER_SOBOL_OWEN) {
        owen_stream o;
        if (!owen_open(sc, k, sobol_dimension(dim), o)) return false;
        const uint32_t head = owen_bits<0u, 8u>(o);
        below = (float)(head + 1u) * 0x1p-8f <= p;
        if (!below && (float)head * 0x1p-8f < p) below = (float)((head << 16) | owen_bits<8u, 24u>(o)) * 0x1p-24f < p;
        return true;
    }
    below = (float)(indexed_bits(k, dim) >> 40) * 0x1p-24f < p;
    return true;
}

/* The leading eight bits of sample_1d(dim), as a binary32 value: the sample rounded down to a multiple of
 * 1/256. Negative when the dimension has no sample. */
BF_D float sample_head(const sampler_ctx& sc, const sample_key& k, uint64_t dim) {
    if (sc.kind == BF_SAMPLER_SOBOL_OWEN) {
        owen_stream o;
        return owen_open(sc, k, sobol_dimension(dim), o) ? (float)owen_bits<0u, 8u>(o) * 0x1p-8f : -1.0f;
    }
    return (float)(indexed_bits(k, dim) >> 56) * 0x1p-8f;
}

/* ---- checked arithmetic: TransportDevice.cuh:196-259 --------------------------------------- */
/* The helpers of the shade stage evaluate every condition and combine the verdicts without branches:
 * a failed check is rare, a value computed past one is never used, and nested early exits cost the
 * kernels more scalar mask arithmetic than the skipped operations. */
BF_D bool checked_product(float l, float r, float& out) {
    const float p = l * r;
    out = p;
    return bf_isfinite(l) & (l >= 0.0f) & bf_isfinite(r) & (r >= 0.0f) & bf_isfinite(p) & (p >= 0.0f) &
           ((l == 0.0f) | (r == 0.0f) | (p != 0.0f));
}

template <int NN, int ND>
BF_D int checked_product_quotient(const float (&num)[NN], const float (&den)[ND], float& out) {
    bool has_zero = false, valid = true;
    float significand = 1.0f;
    int exponent = 0;
#pragma unroll
    for (int i = 0; i < NN; ++i) {
        valid = valid & (bool)bf_isfinite(num[i]) & (num[i] >= 0.0f);
        has_zero = has_zero | (num[i] == 0.0f);
        int e;
        significand *= bf_frexpf(num[i], &e);
        exponent += e;
    }
#pragma unroll
    for (int i = 0; i < ND; ++i) {
        valid = valid & (bool)bf_isfinite(den[i]) & (den[i] > 0.0f);
        int e;
        significand /= bf_frexpf(den[i], &e);
        exponent -= e;
    }
    int ne;
    const float scaled = bf_frexpf(significand, &ne);
    const float r = bf_ldexpf(scaled, exponent + ne);
    const bool representable = bf_isfinite(significand) & (significand > 0.0f) & bf_isfinite(r) & (r > 0.0f);
    out = has_zero ? 0.0f : r;
    return !valid ? BF_L_INVALID : (has_zero | representable ? BF_L_OK : BF_L_NOT_REPRESENTABLE);
}

/* TransportDevice.cuh:552-590 */
BF_D bool joint_light_pdf(float selection, float conditional, float& out) {
    const bool valid = bf_isfinite(selection) & (selection > 0.0f) & (selection <= 1.0f) & bf_isfinite(conditional) &
                       (conditional >= 0.0f);
    const float num[2] = {selection, conditional};
    const float den[1] = {1.0f};
    return valid & (checked_product_quotient(num, den, out) == BF_L_OK);
}

/* TransportDevice.cuh:592-628 */
BF_D bool ratio_at_most_one(float n, float d, bool squared, float& out) {
    int ne, de;
    const float ns = bf_frexpf(n, &ne);
    const float ds = bf_frexpf(d, &de);
    const float ratio = ns / ds;
    const float r = bf_ldexpf(squared ? ratio * ratio : ratio, squared ? 2 * (ne - de) : ne - de);
    out = r;
    return bf_isfinite(n) & (n > 0.0f) & bf_isfinite(d) & (d > 0.0f) & (n <= d) & bf_isfinite(r) & (r >= 0.0f) & (r <= 1.0f);
}

/* TransportDevice.cuh:630-689 */
BF_D bool mis_weight(uint32_t heuristic, float sampled, float competing, float& out) {
    const bool less = sampled < competing;
    float ratio;
    const bool ok = ratio_at_most_one(less ? sampled : competing, less ? competing : sampled, heuristic == 1u, ratio);
    const float w = (less ? ratio : 1.0f) / (1.0f + ratio);
    const bool alone = competing == 0.0f;
    out = alone ? 1.0f : w;
    return bf_isfinite(sampled) & (sampled > 0.0f) & bf_isfinite(competing) & (competing >= 0.0f) & (heuristic <= 1u) &
           (alone | (ok & (!less | (ratio > 0.0f)) & bf_isfinite(w) & (w > 0.0f) & (w <= 1.0f)));
}

/* Russian roulette (TransportDevice.cuh:711-782): the survival probability clamp(max(throughput) *
 * eta, minimum, maximum). */
BF_D bool roulette_probability(float4 t, float eta, float minimum, float maximum, float& p) {
    if (!bf_isfinite(eta) || !(eta > 0.0f)) return false;
    const float v[4] = {t.x, t.y, t.z, t.w};
    float m = 0.0f;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        if (!bf_isfinite(v[k]) || v[k] < 0.0f) return false;
        m = fmaxf(m, v[k]);
    }
    if (m == 0.0f) return false;
    if (m >= maximum / eta) p = maximum;
    else if (m <= minimum / eta) p = minimum;
    else {
        const float c = m * eta;
        p = c < minimum ? minimum : (maximum < c ? maximum : c);
    }
    return true;
}

/* The survivor's throughput, divided by its survival probability p. */
BF_D bool roulette_survive(float4& t, float p) {
    const float v[4] = {t.x, t.y, t.z, t.w};
    float o[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        o[k] = v[k] / p;
        if (!bf_isfinite(o[k]) || (v[k] != 0.0f && o[k] == 0.0f)) return false;
    }
    t = make_float4(o[0], o[1], o[2], o[3]);
    return true;
}

BF_D bool finite_nonnegative4(float4 t) {
    return bf_isfinite(t.x) && t.x >= 0.0f && bf_isfinite(t.y) && t.y >= 0.0f && bf_isfinite(t.z) && t.z >= 0.0f &&
           bf_isfinite(t.w) && t.w >= 0.0f;
}

/* TransportDevice.cuh:327-333 */
BF_D bool unit_vector(v3f d) {
    const float sq = fmaf(d.x, d.x, fmaf(d.y, d.y, d.z * d.z));
    return fin3(d) & bf_isfinite(sq) & (fabsf(sq - 1.0f) <= 128.0f * BF_EPS);
}

/* CudaWavefrontStages.cu:326-349 */
BF_D bool normalize3(v3f v, v3f& out) {
    const float m = fmaxf(fabsf(v.x), fmaxf(fabsf(v.y), fabsf(v.z)));
    const v3f s = mk(v.x / m, v.y / m, v.z / m);
    const float mag = sqrtf(dot3(s, s));
    const bool finite = fin3(v);
    out = mk(s.x / mag, s.y / mag, s.z / mag);
    return finite & bf_isfinite(m) & (m != 0.0f) & bf_isfinite(mag) & (mag > 0.0f) & fin3(out);
}

BF_D bool valid_surface_event(uint32_t bits) {
    const uint32_t family = bits & 0x7u;
    const uint32_t direction = bits & 0x18u;
    return (bits & ~0x3Fu) == 0u && (bits & BF_LOBE_VOLUME) == 0u && family != 0u && (family & (family - 1u)) == 0u &&
           direction != 0u && (direction & (direction - 1u)) == 0u;
}

#endif
