/*
 * Path-slot helpers shared by the kernel translation units: a slot's frame, sample key and failure
 * record, spectra, and ray cones.
 */
#ifndef BF_PATHS_H
#define BF_PATHS_H

#include "bf_device_lobes.h"
#include "bf_kernels.h"

#define BF_BLOCK 256u

static inline uint32_t blocks_for(uint32_t n, uint32_t b) { return n / b + (n % b != 0u ? 1u : 0u); } /* n + b may not fit */

/* ---- path helpers ----------------------------------------------------------------------------- */
/* The frame a slot belongs to: the kernel argument in a single-frame launch, the job table entry
 * recorded for the slot by the camera stage in a batched one. */
template <bool BATCH>
BF_D const bf_dev_job& job_at(const bf_transport_params& P, uint32_t slot) {
    if constexpr (BATCH) return P.jobs[P.paths.job[slot]];
    else return P.job0;
}

BF_D uint64_t path_of(const bf_dev_job& J, uint32_t slot) { return J.path_base + (slot - J.slot_begin); }

BF_D sample_key key_for_slot(const bf_dev_job& J, uint32_t slot) {
    const uint64_t global = path_of(J, slot);
    if (J.in_samples) {
        const bf_sample_stream_index in = J.in_samples[global];
        return sample_key{in.pixel_x, in.pixel_y, in.sample_index, in.seed};
    }
    const uint64_t s = global / J.pixels;
    const uint32_t rem = (uint32_t)(global - s * J.pixels);
    sample_key k;
    k.px = rem % J.camera.width;
    k.py = rem / J.camera.width;
    k.s = (uint64_t)J.first_sample_index + s;
    k.seed = J.seed;
    return k;
}

/* Marks a path failed; the workspace keeps the failure count and the lowest (job, path, code). */
BF_D void fail_path(const bf_transport_params& P, const bf_dev_job& J, uint32_t slot, uint32_t code) {
    P.paths.status[slot] = BF_TERM_FAILED | (code << 8);
    atomicAdd(&P.failure[0], 1u);
    atomicMin((unsigned long long*)(P.failure + 2),
              ((unsigned long long)J.index << 48) | ((unsigned long long)path_of(J, slot) << 8) | code);
}

/* Adds the number of active lanes to *counter with one atomic per wave. */
BF_D void wave_count(uint32_t* counter) {
    const uint64_t active = __ballot(1);
    if ((threadIdx.x & 63u) == (uint32_t)(__ffsll((unsigned long long)active) - 1)) atomicAdd(counter, (uint32_t)__popcll(active));
}

BF_D float spectrum_at(const bf_dev_scene& S, uint32_t id, float wavelength) {
    if (id == BF_INVALID_INDEX) return 0.0f;
    const bf_spectrum_desc sp = S.spectra[id];
    const float* v = S.spectrum_values + sp.offset;
    if (sp.count & BF_SPECTRUM_SAMPLED) {
        /* four (wavelength, value) pairs; the host admits only frames whose packet is these
         * wavelengths, so one lane always matches */
#pragma unroll
        for (int lane = 0; lane < 4; ++lane)
            if (v[lane] == wavelength) return v[4 + lane];
        return __builtin_nanf("");
    }
    if (sp.count <= 1u) return v[0];
    const float step = 470.0f / (float)(sp.count - 1u);
    const float t = (wavelength - 360.0f) / step;
    uint32_t i = t <= 0.0f ? 0u : (uint32_t)t;
    if (i > sp.count - 2u) i = sp.count - 2u;
    const float f = t - (float)i;
    return fmaf(v[i + 1] - v[i], f, v[i]);
}

/* spectrum_at of the four wavelengths of a path: the descriptor is read and the grid step formed once. */
BF_D void spectrum_lanes(const bf_dev_scene& S, uint32_t id, const float* wl, float* out) {
    out[0] = out[1] = out[2] = out[3] = 0.0f;
    if (id == BF_INVALID_INDEX) return;
    const bf_spectrum_desc sp = S.spectra[id];
    const float* v = S.spectrum_values + sp.offset;
    if (sp.count & BF_SPECTRUM_SAMPLED) {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            out[k] = __builtin_nanf("");
#pragma unroll
            for (int lane = 3; lane >= 0; --lane)
                if (v[lane] == wl[k]) out[k] = v[4 + lane];
        }
        return;
    }
    if (sp.count <= 1u) {
        out[0] = out[1] = out[2] = out[3] = v[0];
        return;
    }
    const float step = 470.0f / (float)(sp.count - 1u);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const float t = (wl[k] - 360.0f) / step;
        uint32_t i = t <= 0.0f ? 0u : (uint32_t)t;
        if (i > sp.count - 2u) i = sp.count - 2u;
        const float f = t - (float)i;
        out[k] = fmaf(v[i + 1] - v[i], f, v[i]);
    }
}

BF_D bool valid_cone(float w, float s) { return bf_isfinite(w) && w >= 0.0f && bf_isfinite(s) && s >= 0.0f; }

/* ---- ray cones (CudaWavefrontStages.cu:2816-2867, 3675-3782) ---------------------------------- */
BF_D bool cone_product(float a, float b, float& out) {
    out = a * b;
    return bf_isfinite(out) && !(a != 0.0f && b != 0.0f && out == 0.0f);
}

BF_D bool cone_ratio(float n, float d, float& out) {
    if (!bf_isfinite(n) || !(n > 0.0f) || !bf_isfinite(d) || !(d > 0.0f)) return false;
    out = n / d;
    return bf_isfinite(out) && out > 0.0f;
}

/* the cone at the hit: width + spread x the distance travelled along the (unnormalised) ray */
BF_D bool advance_cone(float2 cone, v3f d, float t, float2& out) {
    if (!valid_cone(cone.x, cone.y) || !bf_isfinite(t) || t < 0.0f) return false;
    const float scale = fmaxf(fabsf(d.x), fmaxf(fabsf(d.y), fabsf(d.z)));
    if (!bf_isfinite(scale) || !(scale > 0.0f)) return false;
    const float inv = 1.0f / scale;
    const float sx = d.x * inv, sy = d.y * inv, sz = d.z * inv;
    const float nl = sqrtf(sx * sx + sy * sy + sz * sz);
    float length, distance, growth;
    if (!bf_isfinite(nl) || !(nl > 0.0f) || !cone_product(scale, nl, length) || !(length > 0.0f)) return false;
    if (!cone_product(t, length, distance) || distance < 0.0f) return false;
    if (!cone_product(cone.y, distance, growth)) return false;
    const float width = fmaf(cone.y, distance, cone.x);
    if (!bf_isfinite(width) || width < cone.x || (growth != 0.0f && width == cone.x)) return false;
    out = make_float2(width, cone.y);
    return valid_cone(out.x, out.y);
}

/* the cone leaving a scattering event: the spread is floored by the sampled closure's roughness
 * (1 for diffuse closures); refraction scales the spread by the eta and cosine ratios and the width
 * by the inverse cosine ratio */
BF_D bool propagate_cone(float2 cone, const closure_t& c, uint32_t event, v3f wo, v3f wi, float2& out) {
    if (!valid_cone(cone.x, cone.y) || !valid_surface_event(event) || !unit_vector(wo) || !unit_vector(wi) ||
        wo.z == 0.0f || wi.z == 0.0f)
        return false;
    const bool reflection = (event & BF_LOBE_REFLECTION) != 0u, transmission = (event & BF_LOBE_TRANSMISSION) != 0u;
    const bool same = (wo.z > 0.0f) == (wi.z > 0.0f);
    if ((reflection && !same) || (transmission && same)) return false;
    float floor_spread = 0.0f, spread_scale = 1.0f, width_scale = 1.0f;
    switch (c.kind) {
    case BF_CLOSURE_LAMBERTIAN:
    case BF_CLOSURE_ROUGH_DIFFUSE:
        if (!reflection || !(event & BF_LOBE_DIFFUSE)) return false;
        floor_spread = 1.0f;
        break;
    case BF_CLOSURE_ROUGH_CONDUCTOR:
        if (!reflection || !(event & BF_LOBE_GLOSSY)) return false;
        if (!bf_isfinite(c.parameters[8]) || c.parameters[8] < 0.0f || !bf_isfinite(c.parameters[9]) ||
            c.parameters[9] < 0.0f)
            return false;
        floor_spread = fmaxf(c.parameters[8], c.parameters[9]);
        break;
    case BF_CLOSURE_ROUGH_DIELECTRIC:
        if (!(event & BF_LOBE_GLOSSY)) return false;
        if (!bf_isfinite(c.parameters[2]) || c.parameters[2] < 0.0f || !bf_isfinite(c.parameters[3]) ||
            c.parameters[3] < 0.0f)
            return false;
        floor_spread = fmaxf(c.parameters[2], c.parameters[3]);
        break;
    case BF_CLOSURE_SPECULAR_REFLECTION:
        if (!reflection || !(event & BF_LOBE_SPECULAR)) return false;
        break;
    case BF_CLOSURE_SPECULAR_TRANSMISSION:
        if (!transmission || !(event & BF_LOBE_SPECULAR)) return false;
        break;
    default:
        return false;
    }
    if (!bf_isfinite(floor_spread) || floor_spread < 0.0f) return false;
    if (transmission) {
        if (c.kind != BF_CLOSURE_ROUGH_DIELECTRIC && c.kind != BF_CLOSURE_SPECULAR_TRANSMISSION) return false;
        const float incident = wo.z > 0.0f ? c.parameters[0] : c.parameters[1];
        const float transmitted = wo.z > 0.0f ? c.parameters[1] : c.parameters[0];
        float eta_ratio, cosine_ratio, inverse_ratio, meridional;
        if (!cone_ratio(incident, transmitted, eta_ratio) || !cone_ratio(fabsf(wo.z), fabsf(wi.z), cosine_ratio) ||
            !cone_ratio(fabsf(wi.z), fabsf(wo.z), inverse_ratio))
            return false;
        if (!cone_product(eta_ratio, cosine_ratio, meridional)) return false;
        spread_scale = fmaxf(eta_ratio, meridional);
        width_scale = fmaxf(1.0f, inverse_ratio);
    }
    float width, spread;
    if (!cone_product(cone.x, width_scale, width) || !cone_product(cone.y, spread_scale, spread)) return false;
    out = make_float2(width, fmaxf(spread, floor_spread));
    return valid_cone(out.x, out.y);
}

#endif
