/*
 * The shade stage of a bounce: surface reconstruction, emission, light and closure sampling, Russian
 * roulette, and the texel gradients of the adjoint replay. Built once per mode (BF_SHADE_MODE, with
 * BF_SHADE_NAME naming its launchers).
 */
#include <hip/hip_runtime.h>

#include <algorithm>

#include "../../include/blackframe_texture.h"
#include "bf_device_adjoint.h"
#include "bf_device_maps.h"
#include "bf_paths.h"
#include "bf_shading.h"
#include "bf_traversal.h"

/* RGB basis spectra of textured reflectance, [3][BF_RGB_BASIS_SAMPLES] */
__constant__ float c_rgb_basis[3 * BF_RGB_BASIS_SAMPLES] = {
#include "data/rgb_basis.inc"
};

/* ---- shade stage: CudaWavefrontStages.cu:4107-4727 -------------------------------------------- */
struct surface_t {
    v3f position, error, ng, ns, dpdu, dpdv;
    float uv[2];
    uint32_t material;
};

/* surface_data (:1523-1665) plus the traversal's world normal (CudaSceneClosestHit.cu:826-871) */
BF_D bool surface_data(const bf_dev_scene& S, uint32_t inst, uint32_t prim, float4 hit, v3f ro, v3f rd, surface_t& out) {
    const bf_dev_instance& I = S.instances[inst];
    const bf_dev_geometry G = S.geometries[I.geometry_index];
    if (prim >= G.triangle_count) return false;
    const size_t t = (size_t)G.triangle_offset + prim;
    uint32_t idx[3] = {S.indices[3 * t], S.indices[3 * t + 1], S.indices[3 * t + 2]};
    const v3f bary = mk(hit.y, hit.z, hit.w);
    v3f lv[3], ln = mk(0.0f, 0.0f, 0.0f);
    float tc[3][2];
    for (int c = 0; c < 3; ++c) {
        if (idx[c] >= G.vertex_count) return false;
        const size_t gv = (size_t)G.vertex_offset + idx[c];
        lv[c] = mk(S.positions[3 * gv], S.positions[3 * gv + 1], S.positions[3 * gv + 2]);
        tc[c][0] = S.uvs[2 * gv];
        tc[c][1] = S.uvs[2 * gv + 1];
        const float w = c == 0 ? bary.x : (c == 1 ? bary.y : bary.z);
        const v3f vn = mk(S.normals[3 * gv], S.normals[3 * gv + 1], S.normals[3 * gv + 2]);
        if (!fin3(lv[c]) || !fin3(vn) || !bf_isfinite(tc[c][0]) || !bf_isfinite(tc[c][1])) return false;
        ln = add3(ln, mul3(vn, w));
    }
    v3f ng;
    if (!world_normal(I.local_to_world, lv[0], lv[1], lv[2], ng)) return false;
    const float* inv = I.world_to_local;
    const float* m = I.local_to_world;
    const v3f tn = mk(fmaf(inv[0], ln.x, fmaf(inv[4], ln.y, inv[8] * ln.z)), fmaf(inv[1], ln.x, fmaf(inv[5], ln.y, inv[9] * ln.z)),
                      fmaf(inv[2], ln.x, fmaf(inv[6], ln.y, inv[10] * ln.z)));
    v3f ns;
    if (!normalize3(tn, ns) || !normalize3(ng, ng)) return false;
    if (dot3(ns, ng) < 0.0f) ns = mul3(ns, -1.0f);
    if (!(dot3(ns, ng) > 0.0f)) return false;
    v3f wv[3];
    for (int c = 0; c < 3; ++c) {
        wv[c] = xform_point(m, lv[c]);
        if (!fin3(wv[c])) return false;
    }
    /* surface_derivatives (:1036-1060) */
    const v3f e1 = sub3(wv[1], wv[0]), e2 = sub3(wv[2], wv[0]);
    const float du1 = tc[1][0] - tc[0][0], dv1 = tc[1][1] - tc[0][1];
    const float du2 = tc[2][0] - tc[0][0], dv2 = tc[2][1] - tc[0][1];
    const float det = fmaf(du1, dv2, -dv1 * du2);
    v3f dpdu = mk(0.0f, 0.0f, 0.0f), dpdv = mk(0.0f, 0.0f, 0.0f);
    if (!fin3(e1) || !fin3(e2) || !bf_isfinite(det)) return false;
    if (det != 0.0f) {
        const float rcp = 1.0f / det;
        dpdu = mul3(sub3(mul3(e1, dv2), mul3(e2, dv1)), rcp);
        dpdv = mul3(sub3(mul3(e2, du1), mul3(e1, du2)), rcp);
        if (!bf_isfinite(rcp) || !fin3(dpdu) || !fin3(dpdv)) return false;
    }
    /* texture coordinates at the hit, for textured closures */
    for (int k = 0; k < 2; ++k) out.uv[k] = fmaf(tc[2][k], bary.z, fmaf(tc[1][k], bary.y, tc[0][k] * bary.x));
    positioned_t obj, world;
    const v3f traversal = mk(fmaf(hit.x, rd.x, ro.x), fmaf(hit.x, rd.y, ro.y), fmaf(hit.x, rd.z, ro.z));
    if (!interpolate_position_with_error(lv, bary, obj) || !transform_position_with_error(m, obj, traversal, world))
        return false;
    out.position = world.position;
    out.error = world.error;
    out.ng = ng;
    out.ns = ns;
    out.dpdu = dpdu;
    out.dpdv = dpdv;
    out.material = I.material_index;
    return fin3(out.position) && fin3(out.error);
}

/* Filtered texel value of a scene texture at (u, v); false when the lookup is not representable. */
BF_D bool texture_value(const bf_dev_scene& S, uint32_t slot, const float* uv, float* value, bf_texel_footprint& f) {
    const bf_dev_texture T = S.textures[slot];
    if (!bf_texture_footprint(T.width, T.height, uv[0], uv[1], &f)) return false;
    bf_texture_filter(T.data, T.channels, &f, value);
    return true;
}

/* The closure kind of a class's materials. */
template <uint32_t CLASS>
BF_D uint32_t class_kind(uint32_t kind) {
    return CLASS == BF_SHADE_LAMBERT      ? (uint32_t)BF_CLOSURE_LAMBERTIAN
           : CLASS == BF_SHADE_CONDUCTOR  ? (uint32_t)BF_CLOSURE_ROUGH_CONDUCTOR
           : CLASS == BF_SHADE_DIELECTRIC ? (uint32_t)BF_CLOSURE_ROUGH_DIELECTRIC
                                          : kind;
}

/* Closure records at the path's wavelengths; textured weights and GGX widths are looked up at the
 * hit's texture coordinates. False when a texture lookup is not representable. */
template <bool TEX, uint32_t CLASS, uint32_t N>
BF_D bool load_mixture(const bf_dev_scene& S, const bf_material_desc& M, const float* wl, const float* uv, mixture_t<N>& mix) {
    mix.active_count = N == 1u ? 1u : M.closure_count;
    for (uint32_t c = 0; c < N && c < mix.active_count; ++c) {
        const bf_closure_desc D = S.closures[M.closure_offset + c];
        closure_t& r = mix.closures[c];
        r.kind = class_kind<CLASS>(D.kind);
        r.lobes = D.lobes;
#pragma unroll
        for (int k = 0; k < 10; ++k) r.parameters[k] = D.parameters[k];
        spectrum_lanes(S, D.weight_spectrum, wl, r.weight);
        if (r.kind == BF_CLOSURE_ROUGH_CONDUCTOR) {
            spectrum_lanes(S, D.eta_spectrum, wl, r.parameters);
            spectrum_lanes(S, D.k_spectrum, wl, r.parameters + 4);
        }
        if (TEX && D.weight_texture) {
            float t[3];
            bf_texel_footprint f;
            if (!texture_value(S, D.weight_texture - 1u, uv, t, f)) return false;
            const uint32_t channels = S.textures[D.weight_texture - 1u].channels;
#pragma unroll
            for (int lane = 0; lane < 4; ++lane) r.weight[lane] *= bf_texel_reflectance(c_rgb_basis, t, channels, wl[lane]);
        }
        if (TEX && D.roughness_texture) {
            float t[3];
            bf_texel_footprint f;
            if (!texture_value(S, D.roughness_texture - 1u, uv, t, f)) return false;
            const float ay = S.textures[D.roughness_texture - 1u].channels == 2u ? t[1] : t[0];
            const int at = r.kind == BF_CLOSURE_ROUGH_CONDUCTOR ? 8 : 2;
            r.parameters[at] = t[0];
            r.parameters[at + 1] = ay;
        }
        mix.probabilities[c] = N == 1u ? 1.0f : M.probabilities[c];
    }
#pragma unroll
    for (uint32_t c = 0; c <= N; ++c) mix.cdf[c] = N == 1u ? (float)c : M.cdf[c];
    return true;
}

/* IncidentLightKind of the reference: a mesh-area sample (solid-angle pdf, MIS), a point or
 * spot light (discrete, shadow ray to the contracted point) or a directional light (discrete,
 * shadow ray to infinity). */
enum : uint32_t { BF_INCIDENT_SURFACE = 0u, BF_INCIDENT_POINT = 1u, BF_INCIDENT_INFINITE = 2u };

struct incident_t {
    float radiance[4];
    v3f direction, position, error, normal;
    float conditional, selection;
    uint32_t kind;
    bool present;
};

/* sample_punctual_light (:2240-2376): the scene checks it makes per sample are made by the host. */
BF_D bool sample_punctual(const bf_dev_scene& S, uint32_t index, const float* wl, const surface_t& surf, float sel,
                          incident_t& inc) {
    const bf_dev_punctual L = S.punctuals[index];
    float spectrum[4];
    bool black = true;
    spectrum_lanes(S, L.spectrum, wl, spectrum);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        if (!bf_isfinite(spectrum[c]) || spectrum[c] < 0.0f) return false;
        if (spectrum[c] != 0.0f) black = false;
    }
    const v3f axis = mk(L.direction[0], L.direction[1], L.direction[2]);
    if (L.kind == BF_PUNCTUAL_DIRECTIONAL) {
        if (black) return true;
#pragma unroll
        for (int c = 0; c < 4; ++c) inc.radiance[c] = spectrum[c];
        inc.direction = mul3(axis, -1.0f);
        inc.position = inc.error = inc.normal = mk(0.0f, 0.0f, 0.0f);
        inc.conditional = 1.0f;
        inc.selection = sel;
        inc.kind = BF_INCIDENT_INFINITE;
        inc.present = true;
        return true;
    }
    const v3f position = mk(L.position[0], L.position[1], L.position[2]);
    segment_t seg;
    if (!scaled_segment(sub3(position, surf.position), seg)) return false;
    const float ssd = dot3(seg.scaled, seg.scaled);
    if (!bf_isfinite(ssd) || !(ssd > 0.0f)) return false;
    float transition = 1.0f, smooth = 1.0f;
    if (L.kind == BF_PUNCTUAL_SPOT) {
        const float cone = dot3(axis, mul3(seg.direction, -1.0f));
        if (!bf_isfinite(cone)) return false;
        if (cone <= L.cosine_outer) return true;
        if (L.smooth && cone < L.cosine_inner) {
            transition = (cone - L.cosine_outer) / (L.cosine_inner - L.cosine_outer);
            smooth = 3.0f - 2.0f * transition;
            if (!bf_isfinite(transition) || !(transition > 0.0f) || !(transition < 1.0f) || !bf_isfinite(smooth) ||
                !(smooth > 0.0f))
                return false;
        }
    }
    float radiance[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const float num[4] = {spectrum[c], transition, transition, smooth};
        const float den[3] = {seg.scale, seg.scale, ssd};
        if (checked_product_quotient(num, den, radiance[c]) != BF_L_OK) return false;
    }
    if (black) return true;
#pragma unroll
    for (int c = 0; c < 4; ++c) inc.radiance[c] = radiance[c];
    inc.direction = seg.direction;
    inc.position = position;
    inc.error = mk(L.position_error[0], L.position_error[1], L.position_error[2]);
    inc.normal = mk(0.0f, 0.0f, 0.0f);
    inc.conditional = 1.0f;
    inc.selection = sel;
    inc.kind = BF_INCIDENT_POINT;
    inc.present = true;
    return true;
}

/* contract_point_endpoint (:2630-2682): the shadow ray of a point light stops short of the
 * light's position by its error bound along the direction to the light. */
BF_D bool endpoint_support(float direction, float error, float& contraction) {
    const float candidate = fmaf(fabsf(direction), error, contraction);
    if (!bf_isfinite(candidate) || candidate < contraction) return false;
    if (direction != 0.0f && error != 0.0f) {
        contraction = bf_next_up_f(candidate);
        return bf_isfinite(contraction);
    }
    contraction = candidate;
    return true;
}

BF_D bool contract_point_endpoint(v3f p, v3f err, v3f to_light, v3f& out) {
    if (!fin3(p) || !fin3(err) || err.x < 0.0f || err.y < 0.0f || err.z < 0.0f || !fin3(to_light)) return false;
    float contraction = 0.0f;
    if (!endpoint_support(to_light.x, err.x, contraction) || !endpoint_support(to_light.y, err.y, contraction) ||
        !endpoint_support(to_light.z, err.z, contraction))
        return false;
    out = p;
    if (contraction == 0.0f) return true;
    out = mk(fmaf(-to_light.x, contraction, p.x), fmaf(-to_light.y, contraction, p.y), fmaf(-to_light.z, contraction, p.z));
    if (to_light.x != 0.0f) out.x = to_light.x > 0.0f ? bf_next_down_f(out.x) : bf_next_up_f(out.x);
    if (to_light.y != 0.0f) out.y = to_light.y > 0.0f ? bf_next_down_f(out.y) : bf_next_up_f(out.y);
    if (to_light.z != 0.0f) out.z = to_light.z > 0.0f ? bf_next_down_f(out.z) : bf_next_up_f(out.z);
    return fin3(out);
}

/* sample_registered_light (:2378-2460) + sample_mesh_area_light (:2044-2201); the per-light area
 * CDF of :2085-2147 is a scene constant evaluated by the host, searched here in O(log n). */
BF_D bool sample_light(const bf_transport_params& P, const bf_dev_scene& S, const sample_key& k, uint64_t first_dim,
                       float area_sample, float triangle_sample, const float* wl, uint32_t visibility, const surface_t& surf, incident_t& inc) {
    inc.present = false;
    uint32_t li;
    float sel;
    /* a power-of-two number of lights (up to 256) is selected by the sample's leading bits alone */
    const bool head = !S.light_cdf && S.light_count <= 256u && (S.light_count & (S.light_count - 1u)) == 0u;
    const float u_sel = head ? sample_head(P.sampler, k, first_dim + 0) : sample_1d(P.sampler, k, first_dim + 0);
    if (S.light_cdf ? !cdf_light_selection(S.light_cdf, S.light_count, u_sel, li, sel)
                    : !uniform_light_selection(S.light_count, u_sel, li, sel))
        return false;
    if (li < S.punctual_count) return sample_punctual(S, li, wl, surf, sel, inc);
    const bf_dev_light L = S.lights[li - S.punctual_count];
    const bf_dev_instance& I = S.instances[L.instance];
    if ((I.visibility_mask & visibility) == 0u) return true;
    if (!(area_sample >= 0.0f) || !(area_sample < 1.0f) || !(triangle_sample >= 0.0f) || !(triangle_sample < 1.0f))
        return false;
    /* first triangle whose cumulative bound exceeds the sample (bounds strictly increase) */
    const float* next = S.light_next + L.table_offset;
    uint32_t lo = 0, hi = L.triangle_count;
    while (lo < hi) {
        const uint32_t mid = (lo + hi) >> 1;
        if (area_sample < next[mid]) hi = mid;
        else lo = mid + 1;
    }
    const uint32_t t = lo;
    if (t >= L.triangle_count) return false;
    const float prob = S.light_probabilities[L.table_offset + t];
    const float area = S.light_areas[L.table_offset + t];
    const float remapped = (area_sample - S.light_cumulative[L.table_offset + t]) / prob;
    if (!bf_isfinite(remapped) || remapped < 0.0f || !(remapped < 1.0f)) return false;
    const float root = sqrtf(remapped);
    const float b0 = 1.0f - root, b1 = root * (1.0f - triangle_sample), b2 = root * triangle_sample;
    const bf_dev_geometry G = S.geometries[L.geometry];
    const size_t tri = (size_t)G.triangle_offset + t;
    v3f lv[3], wv[3];
    for (int c = 0; c < 3; ++c) {
        const size_t gv = (size_t)G.vertex_offset + S.indices[3 * tri + c];
        lv[c] = mk(S.positions[3 * gv], S.positions[3 * gv + 1], S.positions[3 * gv + 2]);
        wv[c] = xform_point(I.local_to_world, lv[c]);
    }
    const float4 nrm = S.light_normals[L.table_offset + t];
    const v3f n = mk(nrm.x, nrm.y, nrm.z);
    const float density = prob / area;
    if (!bf_isfinite(density) || !(density > 0.0f)) return false;
    const bf_material_desc& M = S.materials[I.material_index];
    float radiance[4];
    bool black = true;
    spectrum_lanes(S, M.emission_spectrum, wl, radiance);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        if (!bf_isfinite(radiance[c]) || radiance[c] < 0.0f) return false;
        if (radiance[c] != 0.0f) black = false;
    }
    const v3f traversal = add3(add3(mul3(wv[0], b0), mul3(wv[1], b1)), mul3(wv[2], b2));
    positioned_t obj, world;
    if (!interpolate_position_with_error(lv, mk(b0, b1, b2), obj) ||
        !transform_position_with_error(I.local_to_world, obj, traversal, world))
        return false;
    if (black) return true;
    segment_t seg;
    if (!scaled_segment(sub3(world.position, surf.position), seg)) return false;
    float absolute;
    bool supported;
    if (!light_surface_alignment(n, seg.scaled, absolute, supported)) return false;
    if (!supported) return true;
    const float num[4] = {density, seg.scale, seg.scale, seg.cubed};
    const float den[1] = {absolute};
    float cond;
    if (checked_product_quotient(num, den, cond) != BF_L_OK || !(cond > 0.0f)) return false;
#pragma unroll
    for (int c = 0; c < 4; ++c) inc.radiance[c] = radiance[c];
    inc.direction = seg.direction;
    inc.position = world.position;
    inc.error = world.error;
    inc.normal = n;
    inc.conditional = cond;
    inc.selection = sel;
    inc.kind = BF_INCIDENT_SURFACE;
    inc.present = true;
    return true;
}

/* emissive_hit_mis_weight (:2513-2594) */
BF_D bool emission_weight(const bf_transport_params& P, const bf_dev_scene& S, uint32_t inst, float4 prev,
                          const surface_t& surf, float& w) {
    w = 1.0f;
    if (!(prev.w > 0.0f)) return true;
    const int32_t li = S.instances[inst].light_index;
    if (li < 0) return false;
    float sel;
    const uint32_t slot = S.punctual_count + (uint32_t)li;
    if (S.light_cdf ? !cdf_light_probability(S.light_cdf, S.light_count, slot, sel)
                    : !uniform_light_probability(S.light_count, slot, sel))
        return false;
    const float inv_area = S.lights[li].inverse_area;
    segment_t seg;
    if (!scaled_segment(sub3(surf.position, mk(prev.x, prev.y, prev.z)), seg)) return false;
    float absolute;
    bool supported;
    if (!light_surface_alignment(surf.ng, seg.scaled, absolute, supported) || !supported) return false;
    const float num[4] = {inv_area, seg.scale, seg.scale, seg.cubed};
    const float den[1] = {absolute};
    float cond, joint;
    if (checked_product_quotient(num, den, cond) != BF_L_OK) return false;
    if (!joint_light_pdf(sel, cond, joint)) return false;
    return mis_weight(P.mis, prev.w, joint, w);
}

BF_D bool zero4(const float* v) { return v[0] == 0.0f && v[1] == 0.0f && v[2] == 0.0f && v[3] == 0.0f; }

/* ---- adjoint: texel gradients of one path vertex ---------------------------------------------
 * The path's estimate is a sum of products over its vertices; with sampling, MIS weights and
 * roulette held constant, a parameter p of the closures at vertex j scales every term that passes
 * through that vertex's BSDF value. For the light sample (visible contribution N, closure value
 * f_l) and the continuation (radiance R it carried back, value f_s):
 *   dLoss/dp += sum_lanes a * (N * (df_l/dp) / f_l + R * (df_s/dp) / f_s),
 * a = dLoss/d(radiance lane) of the path's pixel. Texel gradients follow through the bilinear
 * weights and, for weights, the RGB basis spectra. */
/* Adds v to texel-channel e of texture k's gradient, through a lane-chosen replica row when the
 * texture is small. */
BF_D void gradient_add(const bf_transport_params& P, const bf_dev_job& J, uint32_t k, size_t e, float v) {
    const uint32_t offset = J.gradient_replica[k];
    if (offset != BF_INVALID_INDEX) {
        const uint32_t row = (blockIdx.x * blockDim.x + threadIdx.x) % BF_GRADIENT_REPLICAS;
        unsafeAtomicAdd(&P.gradient_replicas[(size_t)row * BF_GRADIENT_ROW + offset + e], v);
    } else {
        unsafeAtomicAdd(&J.texture_gradients[k][e], v);
    }
}

/* Texel gradients of one texture at one footprint, summed over the closures that bind it before
 * they go out as atomics: closures of a material share the hit's texture coordinate, so
 * consecutive closures bound to the same texture add into one set of texels. */
struct texel_pending {
    uint32_t slot, channels;
    bf_texel_footprint f;
    float sc[3];
};

BF_D void texel_flush(const bf_transport_params& P, const bf_dev_job& J, texel_pending& p) {
    if (p.slot == BF_INVALID_INDEX) return;
    for (int q = 0; q < 4; ++q)
        for (uint32_t ch = 0; ch < p.channels; ++ch)
            if (p.f.weight[q] != 0.0f && p.sc[ch] != 0.0f)
                gradient_add(P, J, p.slot, (size_t)p.f.index[q] * p.channels + ch, p.f.weight[q] * p.sc[ch]);
    p.slot = BF_INVALID_INDEX;
}

BF_D void texel_add(const bf_transport_params& P, const bf_dev_job& J, texel_pending& p, uint32_t slot, uint32_t channels,
                    const bf_texel_footprint& f, const float* sc) {
    if (p.slot != slot) {
        texel_flush(P, J, p);
        p.slot = slot;
        p.channels = channels;
        p.f = f;
        p.sc[0] = p.sc[1] = p.sc[2] = 0.0f;
    }
    for (uint32_t ch = 0; ch < channels; ++ch) p.sc[ch] += sc[ch];
}

template <uint32_t N_>
BF_D void texel_gradients(const bf_transport_params& P, const bf_dev_job& J, const bf_dev_scene& S, const bf_material_desc& M,
                          const mixture_t<N_>& mix, const filter_t<N_>& filtered, const float* uv, const float* wl, const float* a, bool light, v3f wo,
                          v3f wi_light, const float* f_light, const float* N, bool cont, bool cont_discrete, v3f wi_cont,
                          const float* f_cont, const float* R) {
    texel_pending weights{BF_INVALID_INDEX, 0u, {}, {0.0f, 0.0f, 0.0f}};
    texel_pending widths{BF_INVALID_INDEX, 0u, {}, {0.0f, 0.0f, 0.0f}};
    for (uint32_t i = 0; i < N_ && i < mix.active_count; ++i) {
        const bf_closure_desc D = S.closures[M.closure_offset + filtered.source_indices[i]];
        const bool wgrad = D.weight_texture && J.texture_gradients[D.weight_texture - 1u];
        const bool rgrad = D.roughness_texture && J.texture_gradients[D.roughness_texture - 1u];
        if (!wgrad && !rgrad) continue;
        const closure_t& c = mix.closures[i];
        float gl[4], gs[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            gl[k] = light && f_light[k] > 0.0f ? a[k] * N[k] / f_light[k] : 0.0f;
            gs[k] = cont && f_cont[k] > 0.0f ? a[k] * R[k] / f_cont[k] : 0.0f;
        }
        if (wgrad) {
            float dl[4] = {0.0f, 0.0f, 0.0f, 0.0f}, ds[4] = {0.0f, 0.0f, 0.0f, 0.0f};
            const bool lw = light && closure_weight_derivative(c, filtered.allowed[i], wo, wi_light, dl) == BF_L_OK;
            /* a delta continuation carries the sum of the matching delta atoms: only their weights
             * move it, and each by its unit-weight atom value */
            const bool cw = cont && (cont_discrete ? delta_weight_derivative(c, wo, wi_cont, ds)
                                                   : closure_weight_derivative(c, filtered.allowed[i], wo, wi_cont, ds) == BF_L_OK);
            const uint32_t slot = D.weight_texture - 1u;
            const uint32_t channels = S.textures[slot].channels;
            float t[3];
            bf_texel_footprint f;
            if (texture_value(S, slot, uv, t, f)) {
                float sc[3] = {0.0f, 0.0f, 0.0f};
                for (int k = 0; k < 4; ++k) {
                    const float g = (lw ? gl[k] * dl[k] : 0.0f) + (cw ? gs[k] * ds[k] : 0.0f);
                    if (g == 0.0f) continue;
                    const float w = g * spectrum_at(S, D.weight_spectrum, wl[k]);
                    if (channels == 1u) {
                        if (t[0] > 0.0f && t[0] < 1.0f) sc[0] += w;
                    } else {
                        float b[3];
                        bf_rgb_basis_at(c_rgb_basis, wl[k], b);
                        const float rho = t[0] * b[0] + t[1] * b[1] + t[2] * b[2];
                        if (!(rho > 0.0f) || !(rho < 1.0f)) continue; /* clamped: no gradient */
                        for (int ch = 0; ch < 3; ++ch) sc[ch] += w * b[ch];
                    }
                }
                texel_add(P, J, weights, slot, channels, f, sc);
            }
        }
        if (rgrad && (c.kind == BF_CLOSURE_ROUGH_CONDUCTOR || c.kind == BF_CLOSURE_ROUGH_DIELECTRIC)) {
            alpha_gradient ql{0.0f, 0.0f}, qs{0.0f, 0.0f};
            const bool use_l = light && closure_alpha_log_gradient(c, wo, wi_light, ql);
            const bool use_s = cont && !cont_discrete && closure_alpha_log_gradient(c, wo, wi_cont, qs);
            /* the closure's own value at each direction: the mixture value when it is alone */
            float fl[4], fs[4];
            for (int k = 0; k < 4; ++k) {
                fl[k] = f_light[k];
                fs[k] = f_cont[k];
            }
            if (mix.active_count > 1u) {
                if (use_l && record_eval(c, filtered.allowed[i], wo, wi_light, fl) != BF_L_OK) continue;
                if (use_s && record_eval(c, filtered.allowed[i], wo, wi_cont, fs) != BF_L_OK) continue;
            }
            float hx = 0.0f, hy = 0.0f;
            for (int k = 0; k < 4; ++k) {
                const float el = use_l ? gl[k] * fl[k] : 0.0f, es = use_s ? gs[k] * fs[k] : 0.0f;
                hx += el * ql.x + es * qs.x;
                hy += el * ql.y + es * qs.y;
            }
            const uint32_t slot = D.roughness_texture - 1u;
            const uint32_t channels = S.textures[slot].channels;
            float t[3];
            bf_texel_footprint f;
            if (texture_value(S, slot, uv, t, f)) {
                const float h[3] = {channels == 2u ? hx : hx + hy, hy, 0.0f};
                texel_add(P, J, widths, slot, channels, f, h);
            }
        }
    }
    texel_flush(P, J, weights);
    texel_flush(P, J, widths);
}

/* route codes written per queue item: 0 terminated, 1 shadow, 2 continuation. MODE is
 * BF_SHADE_PLAIN (no texture lookups compiled in), BF_SHADE_TEXTURED, BF_SHADE_MAPPED (textures and
 * normal / bump maps), or BF_SHADE_ADJOINT: the
 * adjoint replay resolves the light sample from the tape, never routes to the shadow queue and
 * accumulates texel gradients. */
template <bool BATCH, uint32_t MODE, uint32_t CLASS>
BF_D uint32_t shade_item(const bf_transport_params& P, const uint32_t* queue, uint32_t i, uint8_t* route,
                     uint32_t* sample_counts) {
    constexpr bool ADJ = MODE == BF_SHADE_ADJOINT;
    constexpr uint32_t N = CLASS == BF_SHADE_ANY ? BF_MAX_CLOSURES : 1u;
    const uint32_t slot = queue[i];
    route[i] = 0;
    const bf_dev_job& J = job_at<BATCH>(P, slot);
    const bf_dev_scene& S = J.scene;
    const sample_key key = key_for_slot(J, slot);
    const float4 ro4 = P.paths.ray_origin[slot];
    const float4 rd4 = P.paths.ray_direction[slot];
    const v3f ro = mk(ro4.x, ro4.y, ro4.z), rd = mk(rd4.x, rd4.y, rd4.z);
    const float4 hit = P.paths.hit[slot];
    const uint2 ids = P.paths.hit_ids[slot];
    const float4 wl4 = P.paths.wavelengths[slot];
    const float wl[4] = {wl4.x, wl4.y, wl4.z, wl4.w};
    float4 beta4 = P.paths.beta[slot];
    float beta[4] = {beta4.x, beta4.y, beta4.z, beta4.w};
    const float4 L4 = P.paths.radiance[slot];
    float L[4] = {L4.x, L4.y, L4.z, L4.w};
    uint4 dstate = P.paths.depth[slot];
    uint32_t diffuse = dstate.x & 0xFFu, glossy = (dstate.x >> 8) & 0xFFu, specular = (dstate.x >> 16) & 0xFFu,
             transmission = (dstate.x >> 24) & 0xFFu;
    uint32_t depth = dstate.y, delta_flags = dstate.z & 3u;
    const uint32_t vertex = depth;
    float eta_scale = __uint_as_float(dstate.w);
    const float4 prev = P.paths.previous[slot];
    const uint32_t visibility = P.paths.visibility[slot];

    surface_t surf;
    if (!surface_data(S, ids.x, ids.y, hit, ro, rd, surf)) return 10u;
    if (MODE == BF_SHADE_MAPPED && S.maps &&
        (S.maps[surf.material].normal_texture != BF_INVALID_INDEX || S.maps[surf.material].bump_texture != BF_INVALID_INDEX)) {
        /* the shade stage's surface maps (:4170-4193): the cone advanced to the hit sets the
         * footprint; 46 the cone, 47-49 the maps (invalid, numerical, texel budget) */
        float2 at_hit;
        if (!(J.in_cones || J.frame_cones) || !advance_cone(P.paths.cone[slot], rd, hit.x, at_hit))
            return 46u;
        const int st = apply_surface_maps(S, surf.material, at_hit, rd, surf.uv[0], surf.uv[1], surf.ng, surf.dpdu,
                                          surf.dpdv, surf.ns);
        if (st != BF_MAP_OK) return 46u + (uint32_t)st;
    }
    v3f wo;
    if (!normalize3(mk(-rd.x, -rd.y, -rd.z), wo)) return 11u;
    bool front = false;
    if (!one_sided_emission_support(surf.ng, wo, front)) return 12u;
    const bf_material_desc& M = S.materials[surf.material];
    float emitted[4];
    spectrum_lanes(S, M.emission_spectrum, wl, emitted);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        if (!bf_isfinite(emitted[c]) || emitted[c] < 0.0f) return 13u;
    }
    mixture_t<N> mix;
    if (!load_mixture<MODE != BF_SHADE_PLAIN, CLASS>(S, M, wl, surf.uv, mix)) return 42u;
    frame3 frame, unrotated;
    const bool created = M.frame_mode == 0u ? make_local_frame(surf.ns, unrotated) : frame_from_tangent(surf.ns, surf.dpdu, unrotated);
    if (!created || !rotate_frame(unrotated, M.tangent_rotation, frame)) return 14u;
    if (front && !zero4(emitted)) {
        float weight;
        if (!emission_weight(P, S, ids.x, prev, surf, weight)) return 15u;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            if (beta[c] == 0.0f || emitted[c] == 0.0f || weight == 0.0f) continue;
            const float num[3] = {beta[c], emitted[c], weight};
            const float den[1] = {1.0f};
            float contribution;
            if (checked_product_quotient(num, den, contribution) != BF_L_OK) return 16u;
            L[c] += contribution;
            if (!bf_isfinite(L[c])) return 16u;
        }
        P.paths.radiance[slot] = make_float4(L[0], L[1], L[2], L[3]);
    }
    if (zero4(beta)) {
        P.paths.status[slot] = BF_TERM_ZERO_THROUGHPUT;
        return 0u;
    }
    const uint32_t limits[5] = {P.limits[0], P.limits[1], P.limits[2], P.limits[3], P.limits[4]};
    const uint32_t counters[5] = {diffuse, glossy, specular, transmission, 0u};
    if (diffuse > limits[0] || glossy > limits[1] || specular > limits[2] || transmission > limits[3])
        return 17u;
    filter_t<N> filtered;
    filter_by_depth(mix, limits, counters, depth, filtered);
    if (filtered.status != BF_L_OK) return 18u;
    if (mix.active_count == 0 && filtered.source_count != 0) {
        /* the depth categories that blocked the path ride above the termination byte */
        P.paths.status[slot] = BF_TERM_DEPTH_LIMIT | (filtered.blocked << 8);
        return 0u;
    }
    if (N == 1u) mix.active_count = 1u;
    const v3f wo_local = to_local(frame, wo);
    const uint64_t first_dim = 4ull + (uint64_t)depth * 10ull;
    /* light area and triangle, closure u and v, closure selection: one Lambert or conductor closure has
     * nothing to select (where that dimension has no sample the next one has none either, and that
     * fails the path the same way) */
    constexpr bool SELECTS = CLASS != BF_SHADE_LAMBERT && CLASS != BF_SHADE_CONDUCTOR;
    const uint64_t dims[5] = {first_dim + 1, first_dim + 2, first_dim + 4, first_dim + 5, first_dim + 3};
    float samples[5] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    sample_each<SELECTS ? 5 : 4>(P.sampler, key, dims, samples);
    const float bsdf_u = samples[2], bsdf_v = samples[3], bsdf_component = samples[4];
    wave_count(&sample_counts[0]);
    mixture_sample_t bs;
    sample_mixture(mix, filtered, wo_local, bsdf_component, bsdf_u, bsdf_v, bs);
    const bool has_continuation = bs.status == BF_L_OK;
    if (!has_continuation && bs.status != BF_L_OUTSIDE) return 19u;
    if (has_continuation) {
        const bool delta = valid_surface_event(bs.lobes) && (bs.lobes & BF_LOBE_SPECULAR);
        if (!valid_surface_event(bs.lobes) || (bs.discrete != 0u) != delta || !bf_isfinite(bs.pdf) || !(bs.pdf > 0.0f) ||
            (delta && bs.pdf > 1.0f))
            return 20u;
    }
    incident_t inc;
    inc.present = false;
    if (S.light_count != 0u && mixture_nonblack(mix)) {
        wave_count(&sample_counts[1]);
        if (!sample_light(P, S, key, first_dim, samples[0], samples[1], wl, visibility, surf, inc)) return 21u;
    }
    bool has_shadow = false;
    float4 shadow_o = make_float4(0.0f, 0.0f, 0.0f, 0.0f), shadow_d = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    float contribution[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    float nee_f[4] = {0.0f, 0.0f, 0.0f, 0.0f}; /* closure value toward the light (adjoint) */
    v3f nee_wi = mk(0.0f, 0.0f, 0.0f);
    if (inc.present) {
        const v3f wi_local = to_local(frame, inc.direction);
        nee_wi = wi_local;
        if (wo_local.z != 0.0f && wi_local.z != 0.0f) {
            const bool singleton_lambert = mix.active_count == 1 && mix.closures[0].kind == BF_CLOSURE_LAMBERTIAN;
            float bsdf[4] = {0.0f, 0.0f, 0.0f, 0.0f};
            if (singleton_lambert) {
                if (wo_local.z > 0.0f && wi_local.z > 0.0f)
                    for (int c = 0; c < 4; ++c) bsdf[c] = mix.closures[0].weight[c];
            } else if (mixture_eval(mix, filtered, wo_local, wi_local, bsdf) != BF_L_OK) {
                return 22u;
            }
            for (int c = 0; c < 4; ++c) nee_f[c] = singleton_lambert ? bsdf[c] * BF_INV_PI : bsdf[c];
            if (!zero4(bsdf)) {
                float corr;
                if (!shading_correction(surf.ng, surf.ns, wo, inc.direction, corr)) return 23u;
                if (corr > 0.0f) {
                    float w = 1.0f; /* punctual lights are discrete: no MIS (:4437-4470) */
                    if (inc.kind == BF_INCIDENT_SURFACE) {
                        float joint, bsdf_pdf;
                        if (!joint_light_pdf(inc.selection, inc.conditional, joint)) return 24u;
                        if (mixture_pdf(mix, filtered, wo_local, wi_local, bsdf_pdf) != BF_L_OK) return 24u;
                        if (!mis_weight(P.mis, joint, bsdf_pdf, w)) return 24u;
                    }
                    /* the visible-shadow contribution of process_shadow_kernel (:4772-4908),
                     * evaluated now from the same frozen factors */
                    const float coefficient = singleton_lambert ? BF_INV_PI : 1.0f;
                    const float cosine = fabsf(wi_local.z);
                    for (int c = 0; c < 4; ++c) {
                        const float den[2] = {inc.selection, inc.conditional};
                        int st;
                        if (w == 1.0f) {
                            const float num[6] = {beta[c], bsdf[c], coefficient, inc.radiance[c], cosine, corr};
                            st = checked_product_quotient(num, den, contribution[c]);
                        } else {
                            const float num[7] = {beta[c], bsdf[c], coefficient, inc.radiance[c], cosine, corr, w};
                            st = checked_product_quotient(num, den, contribution[c]);
                        }
                        if (st != BF_L_OK) return 41u;
                    }
                    /* prepare_shadow_ray (:4042-4105) */
                    v3f src, endpoint;
                    if (!offset_point(surf.position, surf.error, surf.ng, inc.direction, src)) return 25u;
                    if (inc.kind == BF_INCIDENT_INFINITE) {
                        shadow_o = make_float4(src.x, src.y, src.z, BF_INFINITY_F);
                        shadow_d = make_float4(inc.direction.x, inc.direction.y, inc.direction.z, 0.0f);
                    } else {
                        segment_t seg;
                        const bool ends = inc.kind == BF_INCIDENT_POINT
                                              ? contract_point_endpoint(inc.position, inc.error, inc.direction, endpoint)
                                              : offset_point(inc.position, inc.error, inc.normal, mul3(inc.direction, -1.0f), endpoint);
                        if (!ends || !scaled_segment(sub3(endpoint, src), seg) || !(dot3(seg.direction, inc.direction) > 0.0f))
                            return 25u;
                        const float tmax = bf_next_toward_zero_f(seg.length);
                        if (!(tmax > 0.0f)) return 25u;
                        shadow_o = make_float4(src.x, src.y, src.z, tmax);
                        shadow_d = make_float4(seg.direction.x, seg.direction.y, seg.direction.z, 0.0f);
                    }
                    has_shadow = true;
                }
            }
        }
    }
    v3f wi = mk(0.0f, 0.0f, 0.0f);
    bool continuation = has_continuation;
    float corr = 0.0f;
    if (continuation) {
        if (!to_world(frame, bs.incoming, wi)) return 26u;
        bool geo = false;
        if (!shading_correction(surf.ng, surf.ns, wo, wi, corr) || !geometric_event_support(surf.ng, wo, wi, bs.lobes, geo))
            return 27u;
        continuation = corr > 0.0f && geo;
    }
    uint32_t pending_term = BF_TERM_OUTSIDE_SUPPORT;
    bool cont_pending = false;
    if (continuation) {
        /* update_closure_throughput (:3894-3938) */
        float nb[4];
        const float cosine = fabsf(bs.incoming.z);
        if (!bf_isfinite(cosine) || !(cosine > 0.0f)) return 28u;
        if (mix.active_count == 1 && mix.closures[0].kind == BF_CLOSURE_LAMBERTIAN && corr == 1.0f) {
            for (int c = 0; c < 4; ++c)
                if (!checked_product(beta[c], mix.closures[0].weight[c], nb[c])) return 28u;
        } else {
            for (int c = 0; c < 4; ++c) {
                const float num[4] = {beta[c], bs.value[c], cosine, corr};
                const float den[1] = {bs.pdf};
                if (checked_product_quotient(num, den, nb[c]) != BF_L_OK) return 28u;
            }
        }
        const float next_eta = eta_scale * bs.eta_scale;
        if (!bf_isfinite(bs.eta_scale) || !(bs.eta_scale > 0.0f) || !bf_isfinite(next_eta) || !(next_eta > 0.0f))
            return 29u;
        v3f origin;
        if (!offset_point(surf.position, surf.error, surf.ng, wi, origin)) return 30u;
        const bool delta_event = (bs.lobes & BF_LOBE_SPECULAR) != 0u;
        delta_flags = ((delta_flags & 2u) ? 2u : 0u) | (delta_event ? 1u : 2u);
        /* advance_depth_event (:3851-3880) */
        if (bs.lobes & BF_LOBE_DIFFUSE) ++diffuse;
        else if (bs.lobes & BF_LOBE_GLOSSY) ++glossy;
        else ++specular;
        if (bs.lobes & BF_LOBE_TRANSMISSION) ++transmission;
        ++depth;
        eta_scale = next_eta;
        beta4 = make_float4(nb[0], nb[1], nb[2], nb[3]);
        P.paths.previous[slot] = delta_event ? make_float4(0.0f, 0.0f, 0.0f, 0.0f)
                                             : make_float4(surf.position.x, surf.position.y, surf.position.z, bs.pdf);
        if (J.in_cones || J.frame_cones) {
            /* the sampled closure's compact index, then the cone advanced to the hit and scattered */
            uint32_t compact = mix.active_count, matches = 0u;
            for (uint32_t k = 0; k < N && k < mix.active_count; ++k)
                if (filtered.source_indices[k] == bs.selected) {
                    compact = k;
                    ++matches;
                }
            float2 advanced, next;
            if (matches != 1u || compact >= mix.active_count) return 43u;
            if (!advance_cone(P.paths.cone[slot], rd, hit.x, advanced)) return 44u;
            if (!propagate_cone(advanced, mix.closures[N == 1u ? 0u : compact], bs.lobes, wo_local, bs.incoming, next))
                return 45u;
            P.paths.cone[slot] = next;
        }
        P.paths.ray_origin[slot] = make_float4(origin.x, origin.y, origin.z, ro4.w);
        P.paths.ray_direction[slot] = make_float4(wi.x, wi.y, wi.z, 0.0f);
        cont_pending = true;
        pending_term = BF_TERM_NONE;
        if (nb[0] == 0.0f && nb[1] == 0.0f && nb[2] == 0.0f && nb[3] == 0.0f) {
            cont_pending = false;
            pending_term = BF_TERM_ZERO_THROUGHPUT;
        } else if (P.rr_enabled && depth >= P.rr_first) {
            float* frozen = J.tape_survival ? J.tape_survival + path_of(J, slot) * J.survival_stride + vertex : nullptr;
            const bool replay = frozen && J.survival_mode == BF_SURVIVAL_REPLAY;
            float p = 1.0f;
            bool survived = false;
            if (replay) {
                p = *frozen;
                if (!finite_nonnegative4(beta4) || !bf_isfinite(p) || !(p > 0.0f) || p > 1.0f) return 32u;
            } else if (!roulette_probability(beta4, eta_scale, P.rr_min, P.rr_max, p)) {
                return 32u;
            }
            if (!sample_below(P.sampler, key, first_dim + 9, p, survived) || (survived && !roulette_survive(beta4, p)))
                return 32u;
            if (frozen && !replay && !ADJ) *frozen = p;
            if (!survived) {
                cont_pending = false;
                pending_term = BF_TERM_RUSSIAN_ROULETTE;
            }
        }
        P.paths.beta[slot] = beta4;
        P.paths.depth[slot] = make_uint4(diffuse | (glossy << 8) | (specular << 16) | (transmission << 24), depth,
                                         delta_flags, __float_as_uint(eta_scale));
    }
    if constexpr (ADJ) {
        /* the light sample's visibility from the tape, then this vertex's gradients */
        const float4 vis4 = P.paths.shadow_direction[slot];
        const unsigned long long vis =
            (unsigned long long)__float_as_uint(vis4.x) | ((unsigned long long)__float_as_uint(vis4.y) << 32);
        const bool visible = has_shadow && vertex < 64u && ((vis >> vertex) & 1ull) != 0ull;
        if (visible) {
            for (int c = 0; c < 4; ++c) {
                L[c] += contribution[c];
                if (!bf_isfinite(L[c]) || L[c] < 0.0f) return 41u;
            }
            P.paths.radiance[slot] = make_float4(L[0], L[1], L[2], L[3]);
        }
        if (S.has_textures && J.film_gradient) {
            const float4 total = P.paths.shadow_origin[slot];
            const float4 a4 = P.paths.shadow_contribution[slot];
            const float a[4] = {a4.x, a4.y, a4.z, a4.w};
            const float R[4] = {total.x - L[0], total.y - L[1], total.z - L[2], total.w - L[3]};
            texel_gradients(P, J, S, M, mix, filtered, surf.uv, wl, a, visible, wo_local, nee_wi, nee_f, contribution,
                            cont_pending, bs.discrete != 0u, bs.incoming, bs.value, R);
        }
        if (!cont_pending) {
            P.paths.status[slot] = pending_term;
            return 0u;
        }
        route[i] = 2;
        return 0u;
    }
    if (has_shadow) {
        shadow_d.w = __uint_as_float((cont_pending ? 1u : 0u) | (pending_term << 8) | (vertex << 16));
        P.paths.shadow_origin[slot] = shadow_o;
        P.paths.shadow_direction[slot] = shadow_d;
        P.paths.shadow_contribution[slot] = make_float4(contribution[0], contribution[1], contribution[2], contribution[3]);
        route[i] = 1;
        return 0u;
    }
    if (!cont_pending) {
        P.paths.status[slot] = pending_term;
        return 0u;
    }
    route[i] = 2;
    return 0u;
}

/* One kernel's items: the whole queue, or its buckets' range of the order. An item of a single closure
 * keeps it in registers and runs that kind's code alone; the general path indexes up to
 * BF_MAX_CLOSURES of any kind in scratch (1.2 KB a lane). One kernel for every kind of single closure
 * leaves no kernel waiting for the longest wave of the one before: 1.3 ms of shading in a 333x187x1
 * frame, against 2.3 with a kernel per kind and 1.5 with the general kernel alone. The Lambertian
 * kernel needs neither the order nor the other kinds' registers. */
template <bool BATCH, uint32_t MODE, uint32_t KERNEL>
__global__ __launch_bounds__(BF_SHADE_BLOCK, KERNEL == BF_SHADE_ANY ? BF_SHADE_WAVES_PER_SIMD(MODE) : BF_SHADE_SINGLE_WAVES) void k_shade(
    bf_transport_params P, const uint32_t* queue, const uint32_t* count_ptr, const uint32_t* order, uint8_t* route,
    uint32_t* sample_counts) {
    const uint32_t begin = KERNEL == BF_SHADE_ANY || !order ? 0u : P.bucket_ranges[BF_BUCKET_LAMBERT];
    const uint32_t end = !order ? *count_ptr : P.bucket_ranges[KERNEL == BF_SHADE_ANY ? BF_BUCKET_LAMBERT : BF_BUCKET_DIELECTRIC + 1u];
    /* without an order the queue holds one kind */
    const uint32_t lambert_end = order ? P.bucket_ranges[BF_BUCKET_CONDUCTOR] : 0u;
    const uint32_t conductor_end =
        order ? P.bucket_ranges[BF_BUCKET_DIELECTRIC] : (P.shade_buckets >> BF_BUCKET_CONDUCTOR & 1u) != 0u ? end : 0u;
    for (uint32_t i = begin + blockIdx.x * blockDim.x + threadIdx.x; i < end; i += gridDim.x * blockDim.x) {
        /* a single closure's items from the end: the longest, the dielectrics, first */
        const uint32_t at = KERNEL == BF_SHADE_SINGLE ? end - 1u - (i - begin) : i;
        const uint32_t item = order ? order[at] : at;
        uint32_t code;
        if constexpr (KERNEL != BF_SHADE_SINGLE) {
            code = shade_item<BATCH, MODE, KERNEL>(P, queue, item, route, sample_counts);
        } else if (at < lambert_end) {
            code = shade_item<BATCH, MODE, BF_SHADE_LAMBERT>(P, queue, item, route, sample_counts);
        } else if (at < conductor_end) {
            code = shade_item<BATCH, MODE, BF_SHADE_CONDUCTOR>(P, queue, item, route, sample_counts);
        } else {
            code = shade_item<BATCH, MODE, BF_SHADE_DIELECTRIC>(P, queue, item, route, sample_counts);
        }
        if (code != 0u) {
            const uint32_t slot = queue[item];
            fail_path(P, job_at<BATCH>(P, slot), slot, code);
        }
    }
}

#define BF_JOIN2(a, b) a##b
#define BF_JOIN(a, b) BF_JOIN2(a, b)

template <uint32_t KERNEL>
static void launch_kernel(const bf_transport_params* P, const uint32_t* queue, const uint32_t* count_ptr, uint32_t max_count,
                         const uint32_t* order, uint8_t* route, uint32_t* sample_counts, bool batch, hipStream_t s) {
    const uint32_t grid = std::min(blocks_for(max_count, BF_SHADE_BLOCK), P->shade_blocks[BF_SHADE_MODE * BF_SHADE_KERNELS + KERNEL]);
    if (batch)
        hipLaunchKernelGGL((k_shade<true, BF_SHADE_MODE, KERNEL>), dim3(grid), dim3(BF_SHADE_BLOCK), 0, s, *P, queue, count_ptr,
                           order, route, sample_counts);
    else
        hipLaunchKernelGGL((k_shade<false, BF_SHADE_MODE, KERNEL>), dim3(grid), dim3(BF_SHADE_BLOCK), 0, s, *P, queue, count_ptr,
                           order, route, sample_counts);
}

template <uint32_t KERNEL>
static uint32_t kernel_blocks(int device) {
    const void* plain = (const void*)k_shade<false, BF_SHADE_MODE, KERNEL>;
    const void* batch = (const void*)k_shade<true, BF_SHADE_MODE, KERNEL>;
    return (uint32_t)std::min(bfk_max_resident(&plain, 1, BF_SHADE_BLOCK, device), bfk_max_resident(&batch, 1, BF_SHADE_BLOCK, device));
}

extern "C" {

bool BF_JOIN(bfk_shade_blocks_, BF_SHADE_NAME)(int device, uint32_t* blocks) {
    blocks[BF_SHADE_ANY] = kernel_blocks<BF_SHADE_ANY>(device);
    blocks[BF_SHADE_LAMBERT] = kernel_blocks<BF_SHADE_LAMBERT>(device);
    blocks[BF_SHADE_SINGLE] = kernel_blocks<BF_SHADE_SINGLE>(device);
    return blocks[0] != 0u && blocks[1] != 0u && blocks[2] != 0u;
}

void BF_JOIN(bfk_shade_, BF_SHADE_NAME)(const bf_transport_params* P, uint32_t kernel, const uint32_t* queue,
                                        const uint32_t* count_ptr, uint32_t max_count, const uint32_t* order, uint8_t* route,
                                        uint32_t* sample_counts, bool batch, hipStream_t s) {
    const auto launch = kernel == BF_SHADE_LAMBERT  ? launch_kernel<BF_SHADE_LAMBERT>
                        : kernel == BF_SHADE_SINGLE ? launch_kernel<BF_SHADE_SINGLE>
                                                    : launch_kernel<BF_SHADE_ANY>;
    launch(P, queue, count_ptr, max_count, order, route, sample_counts, batch, s);
}

} /* extern "C" */
