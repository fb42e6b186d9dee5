/*
 * HIP kernels of the MI355X wavefront path-tracing backend (gfx950, wave64).
 *
 * One bounce of the path loop is: trace_closest (BVH2 closest hit; misses resolved in place) ->
 * stable compaction into the hit queue -> shade (emission + MIS, NEE light sample, BSDF sample,
 * Russian roulette) -> stable compaction into shadow / continuation queues -> trace_shadow
 * (any-hit; visible contributions accumulated) -> stable append of shadow continuations.
 * Stage semantics follow Blackframe/XPU/CUDA/Source/CudaWavefrontStages.cu; queue routing follows
 * Blackframe/Backends/GPU/CUDA/Source/WavefrontTransport.cpp:2222-2649.
 */
#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>

#include "../../include/blackframe_camera_cone.h"
#include "bf_paths.h"
#include "bf_scene_soa.h"

/* PinholeCamera.hpp:140-301 with PixelJitter.hpp:37-63 */
BF_D bool robust_unit(v3f d, v3f& out) {
    if (!fin3(d)) return false;
    const float m = fmaxf(fabsf(d.x), fmaxf(fabsf(d.y), fabsf(d.z)));
    if (m == 0.0f) return false;
    const v3f s = mk(d.x / m, d.y / m, d.z / m);
    const float mag = sqrtf(s.x * s.x + s.y * s.y + s.z * s.z);
    out = mk(s.x / mag, s.y / mag, s.z / mag);
    return fin3(out);
}

/* `cone` (optional) receives the primary ray's cone (width, spread) from its one-pixel
 * differentials, for frames whose materials carry normal or bump maps */
BF_D bool camera_ray(const bf_camera_desc& cam, const sampler_ctx& sc, const sample_key& k, v3f& origin, v3f& dir,
                     float2* cone = nullptr) {
    float ox = 0.5f, oy = 0.5f;
    if (cam.jitter_mode == BF_JITTER_UNIFORM) {
        ox = sample_1d(sc, k, BF_DIM_RASTER_X);
        oy = sample_1d(sc, k, BF_DIM_RASTER_Y);
    }
    if (k.px >= cam.width || k.py >= cam.height || !(ox >= 0.0f) || !(ox < 1.0f) || !(oy >= 0.0f) || !(oy < 1.0f))
        return false;
    const float w = (float)cam.width, h = (float)cam.height;
    const float tx = 2.0f * (float)k.px;
    const float ty = 2.0f * (float)k.py;
    const float nx = (tx + 2.0f * ox) / w - 1.0f;
    const float ny = 1.0f - (ty + 2.0f * oy) / h;
    v3f unit;
    if (!robust_unit(mk(nx * cam.half_width, ny * cam.half_height, -1.0f), unit)) return false;
    const v3f wd = mk(cam.tangent[0] * unit.x + cam.bitangent[0] * unit.y + cam.normal[0] * unit.z,
                      cam.tangent[1] * unit.x + cam.bitangent[1] * unit.y + cam.normal[1] * unit.z,
                      cam.tangent[2] * unit.x + cam.bitangent[2] * unit.y + cam.normal[2] * unit.z);
    if (!robust_unit(wd, dir)) return false;
    origin = mk(cam.origin[0], cam.origin[1], cam.origin[2]);
    if (cone) {
        const float unit_dir[3] = {dir.x, dir.y, dir.z};
        float width, spread;
        if (!bf_camera_cone(&cam, (float)k.px + ox, (float)k.py + oy, unit_dir, &width, &spread)) return false;
        *cone = make_float2(width, spread);
    }
    return true;
}

/* ---- camera stage: device-side primary rays, wavelengths and initial state ------------------- */
__constant__ double c_cie_table_rows[471][3] = {
#include "data/cie1931_cmf.inc"
};

/* color_matching_functions (Cie1931Sensor.cpp:69-93) */
BF_D void cie_cmf(float wavelength, float* response) {
    const float coordinate = wavelength - 360.0f;
    const uint32_t lower_index = (uint32_t)coordinate;
    if (lower_index + 1u >= 471u) {
        for (int c = 0; c < 3; ++c) response[c] = (float)c_cie_table_rows[470][c];
    } else {
        const float fraction = coordinate - (float)lower_index;
        for (int c = 0; c < 3; ++c) {
            const float lower = (float)c_cie_table_rows[lower_index][c];
            const float upper = (float)c_cie_table_rows[lower_index + 1][c];
            response[c] = fmaf(upper - lower, fraction, lower);
        }
    }
}

/* d(film RGB)/d(radiance lane) for the path's pixel, contracted with dLoss/d(film RGB): the film
 * adds rgb = M * sum_lanes L cmf(lambda) normalization / pdf per path (cie_xyz below). */
BF_D float4 film_adjoint(const bf_transport_params& P, const bf_dev_job& J, const sample_key& k, const float* wl) {
    const size_t pixel = (size_t)k.py * J.camera.width + k.px;
    const float d[3] = {J.film_gradient[3 * pixel], J.film_gradient[3 * pixel + 1], J.film_gradient[3 * pixel + 2]};
    const float dx = 3.2404542f * d[0] - 0.9692660f * d[1] + 0.0556434f * d[2];
    const float dy = -1.5371385f * d[0] + 1.8760108f * d[1] - 0.2040259f * d[2];
    const float dz = -0.4985314f * d[0] + 0.0415560f * d[1] + 1.0572252f * d[2];
    const float scale = P.film_normalization / P.film_pdf;
    float a[4];
#pragma unroll
    for (int lane = 0; lane < 4; ++lane) {
        float r[3];
        cie_cmf(wl[lane], r);
        a[lane] = (dx * r[0] + dy * r[1] + dz * r[2]) * scale;
    }
    return make_float4(a[0], a[1], a[2], a[3]);
}

/* camera_stage_kernel's path-input form (CudaWavefrontStages.cu:1347-1405, validity checks
 * :528-575): the slot takes its path's ray, ray cone and path state. Depth counters above 255 (kept
 * in bytes here) and participating media fail the path. */
BF_D bool valid_input_ray(const bf_transport_ray& r) {
    const float d2 = r.direction_x * r.direction_x + r.direction_y * r.direction_y + r.direction_z * r.direction_z;
    return bf_isfinite(r.origin_x) && bf_isfinite(r.origin_y) && bf_isfinite(r.origin_z) && bf_isfinite(r.t_min) &&
           r.t_min >= 0.0f && !isnan(r.t_max) && r.t_max >= r.t_min && bf_isfinite(r.time) && r.time >= 0.0f &&
           r.time <= 1.0f && bf_isfinite(r.direction_x) && bf_isfinite(r.direction_y) && bf_isfinite(r.direction_z) &&
           d2 > 0.0f && r.reserved == 0u;
}

BF_D bool valid_input_state(const bf_path_state_lane& s) {
#pragma unroll
    for (int k = 0; k < 4; ++k)
        if (!bf_isfinite(s.beta.values[k]) || s.beta.values[k] < 0.0f || !bf_isfinite(s.accumulated_radiance.values[k]) ||
            s.accumulated_radiance.values[k] < 0.0f)
            return false;
    if (!bf_isfinite(s.eta_scale) || !(s.eta_scale > 0.0f)) return false;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const float w = s.wavelength_nanometers.values[k], pdf = s.wavelength_pdf_values.values[k];
        if (!bf_isfinite(w) || w < 360.0f || w > 830.0f || !bf_isfinite(pdf) || !(pdf > 0.0f) || s.wavelength_pdf_measures[k] != 5u)
            return false;
    }
#pragma unroll
    for (int k = 0; k < 6; ++k)
        if (s.reserved[k] != 0u) return false;
    const uint64_t total = (uint64_t)s.diffuse_depth + s.glossy_depth + s.specular_depth + s.volume_depth;
    const uint64_t surface = (uint64_t)s.diffuse_depth + s.glossy_depth + s.specular_depth;
    return total == s.depth && s.transmission_depth <= surface && (s.delta_flags & ~3u) == 0u;
}

BF_D bool input_lane(const bf_transport_params& P, const bf_dev_job& J, uint32_t slot) {
    const uint64_t path = path_of(J, slot);
    const bf_transport_ray r = J.in_rays[path];
    const bf_ray_cone c = J.in_cones[path];
    const bf_path_state_lane& s = J.in_states[path];
    P.paths.status[slot] = BF_TERM_NONE;
    P.paths.previous[slot] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    uint32_t code = 0u;
    if (!valid_input_ray(r)) code = 3u;
    else if (!valid_cone(c.width, c.spread) || !valid_input_state(s) || r.current_medium != s.current_medium) code = 4u;
    else if (s.current_medium != 0u || s.volume_depth != 0u) code = 5u;
    else if (s.diffuse_depth > 255u || s.glossy_depth > 255u || s.specular_depth > 255u || s.transmission_depth > 255u)
        code = 6u;
    if (code != 0u) {
        fail_path(P, J, slot, code);
        return false;
    }
    P.paths.beta[slot] = make_float4(s.beta.values[0], s.beta.values[1], s.beta.values[2], s.beta.values[3]);
    P.paths.radiance[slot] = make_float4(s.accumulated_radiance.values[0], s.accumulated_radiance.values[1],
                                         s.accumulated_radiance.values[2], s.accumulated_radiance.values[3]);
    P.paths.wavelengths[slot] = make_float4(s.wavelength_nanometers.values[0], s.wavelength_nanometers.values[1],
                                            s.wavelength_nanometers.values[2], s.wavelength_nanometers.values[3]);
    P.paths.depth[slot] = make_uint4(s.diffuse_depth | (s.glossy_depth << 8) | (s.specular_depth << 16) |
                                         (s.transmission_depth << 24),
                                     s.depth, s.delta_flags | BF_FIRST_RAY, __float_as_uint(s.eta_scale));
    P.paths.visibility[slot] = r.visibility_mask;
    P.paths.cone[slot] = make_float2(c.width, c.spread);
    P.paths.ray_origin[slot] = make_float4(r.origin_x, r.origin_y, r.origin_z, r.time);
    P.paths.ray_direction[slot] = make_float4(r.direction_x, r.direction_y, r.direction_z, r.t_min);
    return true;
}

template <bool BATCH, bool ADJ>
__global__ __launch_bounds__(BF_BLOCK) void k_camera(bf_transport_params P, uint32_t count, uint32_t* ray_queue,
                                                     uint8_t* route) {
    const uint32_t slot = blockIdx.x * blockDim.x + threadIdx.x;
    if (slot >= count) return;
    uint32_t j = 0;
    if constexpr (BATCH) {
        /* jobs are ordered by slot_begin: the last one starting at or before this slot */
        uint32_t lo = 0, hi = P.job_count;
        while (hi - lo > 1u) {
            const uint32_t mid = (lo + hi) >> 1;
            if (P.jobs[mid].slot_begin <= slot) lo = mid;
            else hi = mid;
        }
        j = lo;
        P.paths.job[slot] = (uint16_t)j;
    }
    const bf_dev_job& J = BATCH ? P.jobs[j] : P.job0;
    if (J.in_rays) {
        /* the ray queue is compacted from these routes: paths whose inputs failed never trace */
        ray_queue[slot] = slot;
        route[slot] = input_lane(P, J, slot) ? 1u : 0u;
        return;
    }
    const sample_key k = key_for_slot(J, slot);
    v3f o, d;
    ray_queue[slot] = slot;
    P.paths.status[slot] = BF_TERM_NONE;
    P.paths.beta[slot] = make_float4(1.0f, 1.0f, 1.0f, 1.0f);
    P.paths.radiance[slot] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    P.paths.depth[slot] = make_uint4(0u, 0u, BF_FIRST_RAY, __float_as_uint(1.0f));
    P.paths.previous[slot] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    P.paths.visibility[slot] = J.camera.visibility_mask;
    float wl[4];
    if (P.wavelength_mode == BF_WAVELENGTHS_PER_PATH) {
        const float u = sample_1d(P.sampler, k, 3ull);
        if (!(u >= 0.0f) || !(u < 1.0f)) {
            fail_path(P, J, slot, 2);
            return;
        }
        /* WavelengthSampling.hpp:62-84 */
#pragma unroll
        for (int lane = 0; lane < 4; ++lane) {
            const float offset = (float)lane / 4.0f;
            const float wrap = 1.0f - offset;
            const float shifted = lane != 0 && u >= wrap ? u - wrap : u + offset;
            wl[lane] = fmaf(470.0f, shifted, 360.0f);
        }
    } else {
#pragma unroll
        for (int lane = 0; lane < 4; ++lane) wl[lane] = P.packet[lane];
    }
    P.paths.wavelengths[slot] = make_float4(wl[0], wl[1], wl[2], wl[3]);
    if (J.tape_visibility) {
        const uint64_t path = path_of(J, slot);
        if constexpr (ADJ) {
            /* adjoint lanes keep the tape in the shadow columns, which the replay never traces */
            const unsigned long long vis = J.tape_visibility[path];
            P.paths.shadow_origin[slot] = J.tape_radiance[path];
            P.paths.shadow_direction[slot] =
                make_float4(__uint_as_float((uint32_t)vis), __uint_as_float((uint32_t)(vis >> 32)), 0.0f, 0.0f);
            P.paths.shadow_contribution[slot] = film_adjoint(P, J, k, wl);
        } else {
            J.tape_visibility[path] = 0ull;
        }
    }
    float2 cone;
    if (!camera_ray(J.camera, P.sampler, k, o, d, J.frame_cones ? &cone : nullptr)) {
        fail_path(P, J, slot, 1);
        return;
    }
    if (J.frame_cones) P.paths.cone[slot] = cone;
    P.paths.ray_origin[slot] = make_float4(o.x, o.y, o.z, J.camera.time);
    P.paths.ray_direction[slot] = make_float4(d.x, d.y, d.z, J.camera.t_min);
}

/* ---- stable partition of a queue ---------------------------------------------------------------
 * A launch has one workgroup per chunk of consecutive items. The first kernel counts each chunk's
 * items per destination; in the second every workgroup adds up the chunks before its own (a few
 * thousand words that all of them read from L2) and writes its items behind them, so no kernel of one
 * workgroup stands between the two: the scan of 256-item tiles that did took 5.6 us where everything
 * else fits in 4, and 9.6 ms of a 1920x1080x64 frame. The item count is read on the device, so
 * launches can be issued (and captured) before it is known.
 *
 * Within a chunk a workgroup takes BF_PART_TILE items at a time, each wave a run of 128 in rounds of
 * 64 whose loads are in flight together, with one barrier for the tile. Two rounds: 8 leave a small
 * launch too few workgroups (a 64x64x16 frame 1573 us, 4 1508, 2 1442), 1 gains nothing more there and
 * loses in large ones. */
#define BF_PART_ROUNDS 2u
#define BF_PART_TILE (BF_PART_ROUNDS * BF_BLOCK)

struct chunk_t {
    uint32_t begin, end;
    uint32_t used; /* chunks that hold items, at least one */
};

/* n < 2^31 (a workspace's capacity) and at most 2^12 chunks, so no product leaves 32 bits */
BF_D chunk_t own_chunk(uint32_t n) {
    const uint32_t tiles = (n + BF_PART_TILE - 1u) / BF_PART_TILE;
    const uint32_t per = tiles > gridDim.x ? (tiles + gridDim.x - 1u) / gridDim.x : 1u;
    const uint32_t items = per * BF_PART_TILE;
    const uint32_t begin = blockIdx.x * items;
    chunk_t c;
    c.begin = begin < n ? begin : n;
    c.end = begin + items < n ? begin + items : n;
    c.used = tiles > 1u ? (per > 1u ? (tiles + per - 1u) / per : tiles) : 1u;
    return c;
}

/* chunk_counts[N * blockIdx.x + b] = items of the chunk with key b */
template <uint32_t N, typename KEY>
BF_D void count_chunk(uint32_t n, uint32_t* chunk_counts, KEY&& key_at) {
    __shared__ uint32_t wave_counts[N][BF_BLOCK / 64];
    const chunk_t c = own_chunk(n);
    if (blockIdx.x >= c.used) return;
    uint32_t own[N] = {};
    for (uint32_t base = c.begin; base < c.end; base += BF_PART_TILE) {
        uint32_t keys[BF_PART_ROUNDS];
#pragma unroll
        for (uint32_t r = 0; r < BF_PART_ROUNDS; ++r) {
            const uint32_t offset = r * BF_BLOCK + threadIdx.x;
            keys[r] = offset < c.end - base ? key_at(base + offset) : N;
        }
#pragma unroll
        for (uint32_t r = 0; r < BF_PART_ROUNDS; ++r)
#pragma unroll
            for (uint32_t b = 0; b < N; ++b) own[b] += (uint32_t)__popcll(__ballot(keys[r] == b));
    }
    if ((threadIdx.x & 63u) == 0u)
#pragma unroll
        for (uint32_t b = 0; b < N; ++b) wave_counts[b][threadIdx.x >> 6] = own[b];
    __syncthreads();
    if (threadIdx.x < N) {
        uint32_t total = 0;
        for (uint32_t w = 0; w < BF_BLOCK / 64; ++w) total += wave_counts[threadIdx.x][w];
        chunk_counts[N * blockIdx.x + threadIdx.x] = total;
    }
}

/* before[b], all[b]: items with key b in the chunks before this one, and in all of them */
template <uint32_t N>
BF_D void chunk_prefix(const chunk_t& c, const uint32_t* chunk_counts, uint32_t (&before)[N], uint32_t (&all)[N]) {
    __shared__ uint32_t partial[2][N][BF_BLOCK / 64];
    uint32_t lower[N] = {}, every[N] = {};
    for (uint32_t k = threadIdx.x; k < c.used; k += BF_BLOCK)
#pragma unroll
        for (uint32_t b = 0; b < N; ++b) {
            const uint32_t v = chunk_counts[N * k + b];
            every[b] += v;
            lower[b] += k < blockIdx.x ? v : 0u;
        }
#pragma unroll
    for (uint32_t b = 0; b < N; ++b)
#pragma unroll
        for (uint32_t step = 32u; step != 0u; step >>= 1) {
            every[b] += __shfl_xor(every[b], (int)step, 64);
            lower[b] += __shfl_xor(lower[b], (int)step, 64);
        }
    if ((threadIdx.x & 63u) == 0u)
#pragma unroll
        for (uint32_t b = 0; b < N; ++b) {
            partial[0][b][threadIdx.x >> 6] = lower[b];
            partial[1][b][threadIdx.x >> 6] = every[b];
        }
    __syncthreads();
#pragma unroll
    for (uint32_t b = 0; b < N; ++b) {
        before[b] = 0u;
        all[b] = 0u;
#pragma unroll
        for (uint32_t w = 0; w < BF_BLOCK / 64; ++w) {
            before[b] += partial[0][b][w];
            all[b] += partial[1][b][w];
        }
    }
}

/* put(i, b, p) for every item i of the chunk with key b < N: p counts from run[b] up, in queue order */
template <uint32_t N, typename KEY, typename PUT>
BF_D void scatter_chunk(const chunk_t& c, uint32_t (&run)[N], KEY&& key_at, PUT&& put) {
    __shared__ uint32_t wave_counts[2][N][BF_BLOCK / 64];
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = threadIdx.x >> 6;
    const uint64_t below = lane == 0u ? 0ull : (~0ull >> (64u - lane));
    uint32_t parity = 0;
    for (uint32_t base = c.begin; base < c.end; base += BF_PART_TILE, parity ^= 1u) {
        uint32_t keys[BF_PART_ROUNDS], own[N] = {};
#pragma unroll
        for (uint32_t r = 0; r < BF_PART_ROUNDS; ++r) {
            const uint32_t offset = (wave * BF_PART_ROUNDS + r) * 64u + lane;
            keys[r] = offset < c.end - base ? key_at(base + offset) : N;
        }
#pragma unroll
        for (uint32_t r = 0; r < BF_PART_ROUNDS; ++r)
#pragma unroll
            for (uint32_t b = 0; b < N; ++b) own[b] += (uint32_t)__popcll(__ballot(keys[r] == b));
        if (lane == 0u)
#pragma unroll
            for (uint32_t b = 0; b < N; ++b) wave_counts[parity][b][wave] = own[b];
        /* the other parity's counts are read by waves of the tile before, the same parity's by none:
         * a wave gets here again only past the barrier of the tile between */
        __syncthreads();
        uint32_t at[N];
#pragma unroll
        for (uint32_t b = 0; b < N; ++b) {
            at[b] = run[b];
#pragma unroll
            for (uint32_t w = 0; w < BF_BLOCK / 64; ++w) {
                const uint32_t v = wave_counts[parity][b][w];
                at[b] += w < wave ? v : 0u;
                run[b] += v;
            }
        }
#pragma unroll
        for (uint32_t r = 0; r < BF_PART_ROUNDS; ++r) {
            uint32_t position = 0;
#pragma unroll
            for (uint32_t b = 0; b < N; ++b) {
                const uint64_t m = __ballot(keys[r] == b);
                if (keys[r] == b) position = at[b] + (uint32_t)__popcll(m & below);
                at[b] += (uint32_t)__popcll(m);
            }
            if (keys[r] < N) put(base + (wave * BF_PART_ROUNDS + r) * 64u + lane, keys[r], position);
        }
    }
}

/* Compaction. For route values r = 1, 2: dst_r[base_r + exclusive_prefix(route == r)] = src[i], which is
 * the stable exclusive-scan append of CudaWavefrontQueueCompaction.cu:55-315; base_r is the size of
 * the destination where it is appended to. */
__global__ __launch_bounds__(BF_BLOCK) void k_compact_count(const uint8_t* route, const uint32_t* count_ptr,
                                                            uint32_t* chunk_counts, uint32_t* bases, const uint32_t* size1,
                                                            const uint32_t* size2, uint32_t append1, uint32_t append2) {
    if (blockIdx.x == 0u && threadIdx.x == 0u) { /* the next kernel overwrites the sizes */
        bases[0] = append1 ? *size1 : 0u;
        bases[1] = append2 ? *size2 : 0u;
    }
    count_chunk<2u>(*count_ptr, chunk_counts, [&](uint32_t i) { return (uint32_t)route[i] - 1u; });
}

__global__ __launch_bounds__(BF_BLOCK) void k_compact_scatter(const uint8_t* route, const uint32_t* count_ptr,
                                                              const uint32_t* src, const uint32_t* chunk_counts,
                                                              const uint32_t* bases, uint32_t* dst1, uint32_t* dst2,
                                                              uint32_t* size1, uint32_t* size2) {
    const chunk_t c = own_chunk(*count_ptr);
    if (blockIdx.x >= c.used) return;
    uint32_t run[2], all[2];
    chunk_prefix<2u>(c, chunk_counts, run, all);
    const uint32_t base1 = bases[0], base2 = bases[1];
    if (blockIdx.x == 0u && threadIdx.x == 0u) {
        *size1 = base1 + all[0];
        *size2 = base2 + all[1];
    }
    run[0] += base1;
    run[1] += base2;
    scatter_chunk<2u>(
        c, run, [&](uint32_t i) { return (uint32_t)route[i] - 1u; },
        [&](uint32_t i, uint32_t b, uint32_t p) { (b == 0u ? dst1 : dst2)[p] = src[i]; });
}

/* ---- shade order: hit-queue items grouped by the closure kind of their material ---------------
 * Shading a wave of mixed closure kinds issues every kind's code under a partial mask, and a kernel
 * that can shade every kind needs registers for the widest of them. The shade stage therefore
 * visits the hit queue through a permutation that groups items by bucket (stable within one); each item still writes its route at its own queue position, so the
 * compactions that follow see the queue order unchanged. */
template <bool BATCH>
BF_D uint32_t shade_bucket(const bf_transport_params& P, const uint32_t* queue, uint32_t i) {
    const uint32_t slot = queue[i];
    const bf_dev_scene& S = job_at<BATCH>(P, slot).scene;
    return S.material_buckets[S.instances[P.paths.hit_ids[slot].x].material_index];
}

/* Traversal order: rays grouped by direction octant, so that a wave's rays tend to take the same
 * near/far child order. */
BF_D uint32_t octant(float4 d) { return (d.x < 0.0f ? 1u : 0u) | (d.y < 0.0f ? 2u : 0u) | (d.z < 0.0f ? 4u : 0u); }

template <bool BATCH, uint32_t KEY>
BF_D uint32_t bucket_key(const bf_transport_params& P, const uint32_t* queue, uint32_t i) {
    if constexpr (KEY == BF_KEY_SHADE) return shade_bucket<BATCH>(P, queue, i);
    else if constexpr (KEY == BF_KEY_RAY) return octant(P.paths.ray_direction[queue[i]]);
    else return octant(P.paths.shadow_direction[queue[i]]);
}

template <bool BATCH, uint32_t KEY>
__global__ __launch_bounds__(BF_BLOCK) void k_bucket_count(bf_transport_params P, const uint32_t* queue,
                                                           const uint32_t* count_ptr, uint8_t* keys, uint32_t* chunk_counts) {
    count_chunk<BF_SHADE_BUCKETS>(*count_ptr, chunk_counts, [&](uint32_t i) {
        const uint32_t key = bucket_key<BATCH, KEY>(P, queue, i);
        keys[i] = (uint8_t)key;
        return key;
    });
}

/* Bucket b starts behind the items of the lower ones: at ranges[b]. */
__global__ __launch_bounds__(BF_BLOCK) void k_bucket_scatter(const uint8_t* keys, const uint32_t* count_ptr,
                                                             const uint32_t* chunk_counts, uint32_t* ranges, uint32_t* order) {
    const chunk_t c = own_chunk(*count_ptr);
    if (blockIdx.x >= c.used) return;
    uint32_t run[BF_SHADE_BUCKETS], all[BF_SHADE_BUCKETS];
    chunk_prefix<BF_SHADE_BUCKETS>(c, chunk_counts, run, all);
    uint32_t start = 0;
#pragma unroll
    for (uint32_t b = 0; b < BF_SHADE_BUCKETS; ++b) {
        run[b] += start;
        if (blockIdx.x == 0u && threadIdx.x == 0u) ranges[b] = start;
        start += all[b];
    }
    if (blockIdx.x == 0u && threadIdx.x == 0u) ranges[BF_SHADE_BUCKETS] = start;
    scatter_chunk<BF_SHADE_BUCKETS>(
        c, run, [&](uint32_t i) { return (uint32_t)keys[i]; },
        [&](uint32_t i, uint32_t, uint32_t p) { order[p] = i; });
}

/* End of a bounce: record the queue sizes of the bounce, make the continuation queue the next ray
 * queue, clear the scratch sizes, and advance the bounce counter (one thread). */
__global__ void k_bounce_end(uint32_t* sizes, uint32_t* history, uint32_t history_bounces) {
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    const uint32_t b = sizes[7];
    if (b < history_bounces) {
        history[4 * b + 0] = sizes[0];
        history[4 * b + 1] = sizes[1];
        history[4 * b + 2] = sizes[2];
        history[4 * b + 3] = sizes[3];
    }
    sizes[0] = sizes[3];
    sizes[1] = 0u;
    sizes[2] = 0u;
    sizes[3] = 0u;
    sizes[4] = 0u;
    sizes[5] = 0u;
    sizes[7] = b + 1u;
}

/* ---- film: per-pixel accumulation in sample order (Film.hpp:150-248, Cie1931Sensor.cpp) ----- */
BF_D void cie_xyz(const float* radiance, const float* wavelengths, float pdf, float normalization, float* xyz) {
    float sum[3] = {0.0f, 0.0f, 0.0f};
    for (int lane = 0; lane < 4; ++lane) {
        float response[3];
        cie_cmf(wavelengths[lane], response);
        for (int c = 0; c < 3; ++c) {
            /* scaled_sensor_term (Cie1931Sensor.cpp:104-124) */
            float term = 0.0f;
            if (radiance[lane] != 0.0f && response[c] != 0.0f) {
                int ce, re, ne, pe;
                const float cm = bf_frexpf(radiance[lane], &ce);
                const float rm = bf_frexpf(response[c], &re);
                const float nm = bf_frexpf(normalization, &ne);
                const float pm = bf_frexpf(pdf, &pe);
                const float mantissa = cm * rm * nm / pm;
                term = bf_ldexpf(mantissa, ce + re + ne - pe);
            }
            sum[c] += term;
        }
    }
    xyz[0] = sum[0];
    xyz[1] = sum[1];
    xyz[2] = sum[2];
}

__global__ __launch_bounds__(BF_BLOCK) void k_film(bf_dev_paths paths, bf_dev_job J, float pdf, float normalization) {
    const uint32_t pixels = J.pixels;
    const uint32_t passes = J.slot_count / pixels;
    float* film = J.film;
    double* film_compensated = J.film_compensated;
    uint32_t* film_counts = J.film_counts;
    const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= pixels) return;
    float f[3] = {film[3 * (size_t)p], film[3 * (size_t)p + 1], film[3 * (size_t)p + 2]};
    double s[3], cmp[3];
    for (int c = 0; c < 3; ++c) {
        s[c] = film_compensated[6 * (size_t)p + 2 * c];
        cmp[c] = film_compensated[6 * (size_t)p + 2 * c + 1];
    }
    uint32_t count = film_counts[p];
    for (uint32_t pass = 0; pass < passes; ++pass) {
        const size_t slot = (size_t)J.slot_begin + (size_t)pass * pixels + p;
        const float4 L4 = paths.radiance[slot];
        if (J.tape_radiance) J.tape_radiance[path_of(J, (uint32_t)slot)] = L4;
        const float4 W4 = paths.wavelengths[slot];
        const float L[4] = {L4.x, L4.y, L4.z, L4.w};
        const float W[4] = {W4.x, W4.y, W4.z, W4.w};
        float xyz[3];
        cie_xyz(L, W, pdf, normalization, xyz);
        /* Color.hpp:77-87 */
        const float rgb[3] = {3.2404542f * xyz[0] - 1.5371385f * xyz[1] - 0.4985314f * xyz[2],
                              -0.9692660f * xyz[0] + 1.8760108f * xyz[1] + 0.0415560f * xyz[2],
                              0.0556434f * xyz[0] - 0.2040259f * xyz[1] + 1.0572252f * xyz[2]};
        for (int c = 0; c < 3; ++c) {
            f[c] += rgb[c] * 1.0f;
            const double value = (double)rgb[c] * 1.0;
            const double updated = s[c] + value;
            if (fabs(s[c]) >= fabs(value)) cmp[c] += (s[c] - updated) + value;
            else cmp[c] += (value - updated) + s[c];
            s[c] = updated;
        }
        ++count;
    }
    for (int c = 0; c < 3; ++c) {
        film[3 * (size_t)p + c] = f[c];
        film_compensated[6 * (size_t)p + 2 * c] = s[c];
        film_compensated[6 * (size_t)p + 2 * c + 1] = cmp[c];
    }
    film_counts[p] = count;
}

/* FNV-1a-64 of a queue's slot bytes (diagnostic; one thread) */
__global__ void k_queue_hash(const uint32_t* queue, const uint32_t* count_ptr, unsigned long long* out) {
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    uint64_t h = 14695981039346656037ull;
    const uint32_t n = *count_ptr;
    for (uint32_t i = 0; i < n; ++i) {
        const uint32_t v = queue[i];
        for (int b = 0; b < 4; ++b) {
            h ^= (v >> (8 * b)) & 0xFFu;
            h *= 1099511628211ull;
        }
    }
    out[0] = h;
    out[1] = n;
}

/* ---- sampler probe (SampleStreamKernel.hpp:170-176 counterpart) ------------------------------ */
__global__ void k_sample_dump(sampler_ctx sc, const bf_sample_stream_index* indices, const uint64_t* dims, uint32_t count,
                              float* out) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count) return;
    sample_key k;
    k.px = indices[i].pixel_x;
    k.py = indices[i].pixel_y;
    k.s = indices[i].sample_index;
    k.seed = indices[i].seed;
    out[i] = sample_1d(sc, k, dims[i]);
}

/* The reference's dimension map (SampleDimensionMap.cpp:13-69, SampleStreamKernel.hpp:60-91):
 * bounce b uses dimensions 4 + 10 b + {light selection, light u/v, bsdf component/u/v, medium x3,
 * roulette} for b <= 2^32 - 1. */
__global__ void k_sample_stream_dump(const bf_sample_dump_request* requests, uint32_t count,
                                     bf_sample_dimension_manifest* manifest, bf_sample_dump_result* results) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i == 0u) {
        bf_sample_dimension_manifest m;
        m.schema_version = BF_SAMPLE_DIMENSION_SCHEMA;
        m.reserved = 0u;
        m.primary_dimensions = bf_sample_primary_dimensions{BF_DIM_RASTER_X, BF_DIM_RASTER_Y, 0u, 1u, 2u, 3u};
        m.first_bounce_dimension = BF_SAMPLE_FIRST_BOUNCE_DIMENSION;
        m.dimensions_per_bounce = BF_SAMPLE_DIMENSIONS_PER_BOUNCE;
        m.maximum_bounce_index = BF_SAMPLE_MAXIMUM_BOUNCE;
        m.bounce_offsets = bf_sample_bounce_dimensions{0u, 1u, 2u, 3u, 4u, 5u, 6u, 7u, 8u, 9u};
        *manifest = m;
    }
    if (i >= count) return;
    const bf_sample_dump_request r = requests[i];
    sample_key k;
    k.px = r.sample_stream.pixel_x;
    k.py = r.sample_stream.pixel_y;
    k.s = r.sample_stream.sample_index;
    k.seed = r.sample_stream.seed;
    bf_sample_dump_result out;
    out.reserved = 0u;
    out.reserved_tail = 0u;
    out.indexed_bits = indexed_bits(k, r.dimension);
    out.sample = (float)(out.indexed_bits >> 40) * 0x1p-24f;
    uint64_t d[10];
    if (r.bounce_index > BF_SAMPLE_MAXIMUM_BOUNCE) {
        out.status = BF_SAMPLE_DUMP_BOUNCE_OUT_OF_RANGE;
        for (int k2 = 0; k2 < 10; ++k2) d[k2] = 0u;
    } else {
        out.status = BF_SAMPLE_DUMP_SUCCESS;
        const uint64_t first = BF_SAMPLE_FIRST_BOUNCE_DIMENSION + r.bounce_index * BF_SAMPLE_DIMENSIONS_PER_BOUNCE;
        for (int k2 = 0; k2 < 10; ++k2) d[k2] = first + (uint64_t)k2;
    }
    out.bounce_dimensions = bf_sample_bounce_dimensions{d[0], d[1], d[2], d[3], d[4], d[5], d[6], d[7], d[8], d[9]};
    results[i] = out;
}

/* ---- small utility kernels (used instead of hipMemsetAsync so the sequence stays capturable) - */
/* one thread per gradient element: the replica rows in row order, then one add to the caller's buffer */
__global__ __launch_bounds__(BF_BLOCK) void k_reduce_replicas(const float* replicas, uint32_t offset, uint32_t count,
                                                              float* dst) {
    const uint32_t e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= count) return;
    float sum = 0.0f;
    for (uint32_t row = 0; row < BF_GRADIENT_REPLICAS; ++row) sum += replicas[(size_t)row * BF_GRADIENT_ROW + offset + e];
    dst[e] += sum;
}

/* ---- texture fitting: L2 film loss and Adam ------------------------------------------------- */

__device__ inline void adam_element(float& p, float g, float& m, float& v, const bfk_adam_coefficients& c) {
    m = c.beta1 * m + c.one_minus_beta1 * g;
    v = c.beta2 * v + c.one_minus_beta2 * (g * g);
    const float den = sqrtf(v) / c.bias2_sqrt + c.epsilon;
    p = p - c.step_size * (m / den);
    p = fminf(fmaxf(p, c.lower), c.upper);
}

/* VEC: the four arrays are 16-byte aligned and the body runs on float4 (the tail of count % 4
 * elements is done by the first threads of the grid). */
template <bool VEC>
__global__ __launch_bounds__(BF_BLOCK) void k_adam(float* value, const float* gradient, float* first, float* second,
                                                   uint64_t count, bfk_adam_coefficients c, const float2* schedule,
                                                   const uint32_t* step) {
    if (schedule) {
        /* a replayed step: the bias-corrected step size and sqrt(bias2) of the current step number,
         * computed on the host in the same binary64 arithmetic as a direct call */
        const float2 row = schedule[*step];
        c.step_size = row.x;
        c.bias2_sqrt = row.y;
    }
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    uint64_t scalar_begin = 0;
    if (VEC) {
        const uint64_t quads = count / 4u;
        for (uint64_t i = t; i < quads; i += stride) {
            float4 p = reinterpret_cast<float4*>(value)[i];
            const float4 g = reinterpret_cast<const float4*>(gradient)[i];
            float4 m = reinterpret_cast<float4*>(first)[i];
            float4 v = reinterpret_cast<float4*>(second)[i];
            adam_element(p.x, g.x, m.x, v.x, c);
            adam_element(p.y, g.y, m.y, v.y, c);
            adam_element(p.z, g.z, m.z, v.z, c);
            adam_element(p.w, g.w, m.w, v.w, c);
            reinterpret_cast<float4*>(value)[i] = p;
            reinterpret_cast<float4*>(first)[i] = m;
            reinterpret_cast<float4*>(second)[i] = v;
        }
        scalar_begin = quads * 4u;
    }
    for (uint64_t i = scalar_begin + t; i < count; i += stride) {
        float p = value[i], m = first[i], v = second[i];
        adam_element(p, gradient[i], m, v, c);
        value[i] = p;
        first[i] = m;
        second[i] = v;
    }
}

__global__ __launch_bounds__(BF_BLOCK) void k_film_l2(const float* film, const uint32_t* counts, const float* target,
                                                      float* gradient, uint32_t pixels, float two_scale, double scale,
                                                      double* loss) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    double sum = 0.0;
    if (i < pixels) {
        const float c = (float)(counts[i] > 1u ? counts[i] : 1u);
        for (uint32_t ch = 0; ch < 3u; ++ch) {
            const float d = film[(size_t)i * 3u + ch] / c - target[(size_t)i * 3u + ch];
            gradient[(size_t)i * 3u + ch] = (two_scale * d) / c;
            sum += (double)d * (double)d;
        }
    }
    for (int o = 32; o > 0; o >>= 1) sum += __shfl_down(sum, o, 64);
    __shared__ double partial[BF_BLOCK / 64];
    if ((threadIdx.x & 63u) == 0) partial[threadIdx.x >> 6] = sum;
    __syncthreads();
    if (threadIdx.x == 0) {
        double block = 0.0;
        for (uint32_t w = 0; w < BF_BLOCK / 64; ++w) block += partial[w];
        atomicAdd(loss, scale * block);
    }
}

__global__ void k_zero_doubles(double* dst, uint32_t count) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) dst[i] = 0.0;
}

/* ---- scene blob hash: FNV-1a-64 with the content-hash field read as zero ---------------------- */
/* The byte chain is sequential by definition, so one lane walks it; it reads 16-byte words where
 * the blob is 16-byte aligned and single bytes otherwise. */
/* validate_scene_soa_header on the device copy of a blob (the check every reference stage makes
 * of the uploaded header, CudaWavefrontStages.cu:818-880), one thread; plus the byte count. */
/* validate_scene_soa_header (SceneSoaAbi.hpp:283-341), then the stage check's further conditions
 * (CudaWavefrontStages.cu:818-862): the header's total size equals the device byte count, every
 * record count fits 32 bits, and the mesh-area lights fit the uniform light registry (2^24). */
__global__ void k_scene_soa_validate(const bf_scene_soa_header* header, uint64_t byte_count, uint32_t* status) {
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    const bf_scene_soa_header& h = *header;
    uint32_t st = bf_soa::validate_header(h);
    if (st == BF_SCENE_SOA_VALID && h.total_size_bytes > byte_count) st = BF_SCENE_SOA_TRUNCATED;
    if (st == BF_SCENE_SOA_VALID && h.total_size_bytes != byte_count) st = BF_SCENE_SOA_SIZE_MISMATCH;
    const uint64_t counts[12] = {h.object_count, h.geometry_count, h.vertex_count, h.triangle_count,
                                 h.material_count, h.closure_count, h.instance_count, h.mesh_area_light_count,
                                 h.punctual_light_count, h.texture_count, h.image_texture_count, h.image_mip_count};
    for (int k = 0; k < 12 && st == BF_SCENE_SOA_VALID; ++k)
        if (counts[k] > 0xFFFFFFFFull) st = BF_SCENE_SOA_COUNT_OVERFLOW;
    if (st == BF_SCENE_SOA_VALID && h.mesh_area_light_count > (1ull << 24)) st = BF_SCENE_SOA_TOO_MANY_MESH_LIGHTS;
    *status = st;
}

__global__ void k_scene_hash(const uint8_t* bytes, size_t count, uint64_t* out) {
    if (blockIdx.x != 0u || threadIdx.x != 0u) return;
    uint64_t h = BF_FNV1A64_OFFSET_BASIS;
    const auto step = [&](size_t index, uint32_t byte) {
        const uint32_t v = index >= BF_SCENE_SOA_HASH_OFFSET && index < BF_SCENE_SOA_HASH_OFFSET + 8u ? 0u : byte;
        h ^= v;
        h *= BF_FNV1A64_PRIME;
    };
    size_t i = 0;
    if ((reinterpret_cast<uintptr_t>(bytes) & 15u) == 0u) {
        for (; i + 16u <= count; i += 16u) {
            const uint4 w = *reinterpret_cast<const uint4*>(bytes + i);
            const uint32_t words[4] = {w.x, w.y, w.z, w.w};
            for (int k = 0; k < 4; ++k)
                for (int b = 0; b < 4; ++b) step(i + 4u * k + b, (words[k] >> (8 * b)) & 0xFFu);
        }
    }
    for (; i < count; ++i) step(i, bytes[i]);
    *out = h;
}

/* ---- transport record layout, as device code sees it (CudaTransportAbiProbe.cu:33-160) ------- */
__global__ void k_layout_manifest(bf_layout_manifest* out) {
    if (blockIdx.x != 0u || threadIdx.x != 0u) return;
    bf_layout_manifest m;
    memset(&m, 0, sizeof m);
    m.abi_major = BF_QUEUE_ABI_MAJOR;
    m.abi_minor = BF_QUEUE_ABI_MINOR;
    m.device_cxx_standard = (uint32_t)__cplusplus;
    m.value_count = BF_LAYOUT_VALUE_COUNT;
    uint32_t k = 0;
    const auto put = [&](size_t v) { m.values[k++] = (uint32_t)v; };
    /* the reference's LayoutValue order */
    put(sizeof(bf_transport_spectrum)); put(alignof(bf_transport_spectrum)); put(offsetof(bf_transport_spectrum, values));
    put(sizeof(bf_transport_ray)); put(alignof(bf_transport_ray));
    put(offsetof(bf_transport_ray, origin_x)); put(offsetof(bf_transport_ray, origin_y));
    put(offsetof(bf_transport_ray, origin_z)); put(offsetof(bf_transport_ray, t_min));
    put(offsetof(bf_transport_ray, direction_x)); put(offsetof(bf_transport_ray, direction_y));
    put(offsetof(bf_transport_ray, direction_z)); put(offsetof(bf_transport_ray, t_max));
    put(offsetof(bf_transport_ray, time)); put(offsetof(bf_transport_ray, visibility_mask));
    put(offsetof(bf_transport_ray, current_medium)); put(offsetof(bf_transport_ray, reserved));
    put(sizeof(bf_sample_stream_index)); put(alignof(bf_sample_stream_index));
    put(offsetof(bf_sample_stream_index, pixel_x)); put(offsetof(bf_sample_stream_index, pixel_y));
    put(offsetof(bf_sample_stream_index, sample_index)); put(offsetof(bf_sample_stream_index, seed));
    put(sizeof(bf_path_slot)); put(alignof(bf_path_slot)); put(offsetof(bf_path_slot, value));
    put(sizeof(bf_queue_header)); put(alignof(bf_queue_header));
    put(offsetof(bf_queue_header, abi_major)); put(offsetof(bf_queue_header, abi_minor));
    put(offsetof(bf_queue_header, struct_size)); put(offsetof(bf_queue_header, queue_kind));
    put(offsetof(bf_queue_header, capacity)); put(offsetof(bf_queue_header, size));
    put(offsetof(bf_queue_header, overflow_count)); put(offsetof(bf_queue_header, rejected_count));
    put(offsetof(bf_queue_header, reserved));
    put(sizeof(bf_surface_identifiers)); put(alignof(bf_surface_identifiers));
    put(offsetof(bf_surface_identifiers, object)); put(offsetof(bf_surface_identifiers, instance));
    put(offsetof(bf_surface_identifiers, geometry)); put(offsetof(bf_surface_identifiers, primitive));
    put(offsetof(bf_surface_identifiers, material)); put(offsetof(bf_surface_identifiers, reserved));
    put(sizeof(bf_closest_hit)); put(alignof(bf_closest_hit));
    put(offsetof(bf_closest_hit, parameter)); put(offsetof(bf_closest_hit, barycentric0));
    put(offsetof(bf_closest_hit, barycentric1)); put(offsetof(bf_closest_hit, barycentric2));
    put(offsetof(bf_closest_hit, normal_x)); put(offsetof(bf_closest_hit, normal_y));
    put(offsetof(bf_closest_hit, normal_z)); put(offsetof(bf_closest_hit, reserved)); put(offsetof(bf_closest_hit, ids));
    put(sizeof(bf_path_state_lane)); put(alignof(bf_path_state_lane));
    put(offsetof(bf_path_state_lane, beta)); put(offsetof(bf_path_state_lane, accumulated_radiance));
    put(offsetof(bf_path_state_lane, wavelength_nanometers)); put(offsetof(bf_path_state_lane, wavelength_pdf_values));
    put(offsetof(bf_path_state_lane, diffuse_depth)); put(offsetof(bf_path_state_lane, glossy_depth));
    put(offsetof(bf_path_state_lane, specular_depth)); put(offsetof(bf_path_state_lane, transmission_depth));
    put(offsetof(bf_path_state_lane, volume_depth)); put(offsetof(bf_path_state_lane, depth));
    put(offsetof(bf_path_state_lane, eta_scale)); put(offsetof(bf_path_state_lane, current_medium));
    put(offsetof(bf_path_state_lane, delta_flags)); put(offsetof(bf_path_state_lane, wavelength_pdf_measures));
    put(offsetof(bf_path_state_lane, reserved));
    *out = m;
}

/* ---- queue compaction: CudaWavefrontQueueCompaction.cu:55-250 -------------------------------- */
/* A selected outcome succeeded and names the route; the selected slots keep their outcome order
 * (a stable partition), the append is all or nothing, and a header is used only while its
 * immutable fields and counters satisfy the queue contract (WavefrontQueueDevice.cuh:77-85). */
BF_D bool qc_header_ok(const bf_queue_header& h, uint32_t kind, uint32_t stride) {
    return h.abi_major == BF_QUEUE_ABI_MAJOR && h.abi_minor == BF_QUEUE_ABI_MINOR &&
           h.struct_size == (uint32_t)sizeof(bf_queue_header) && h.queue_kind == kind && h.capacity == stride &&
           h.reserved == 0u;
}

BF_D bool qc_selected(const bf_stage_outcome& o, uint32_t route) { return o.status == 0u && o.route == route; }

BF_D void qc_saturating_add(uint32_t* counter, uint32_t value) {
    uint32_t observed = *counter;
    for (;;) {
        const uint32_t next = value > 0xFFFFFFFFu - observed ? 0xFFFFFFFFu : observed + value;
        const uint32_t previous = atomicCAS(counter, observed, next);
        if (previous == observed) return;
        observed = previous;
    }
}

/* Queue pushes (WavefrontQueueDevice.cuh:118-197): the requests of one wave that name one queue
 * kind reserve a contiguous run with one compare-and-swap on its size, leader lane first; the
 * lanes past the room that was left are rejected and counted. */
__global__ __launch_bounds__(BF_BLOCK) void k_queue_push(bf_queue_soa q, const bf_queue_push* requests, uint32_t n,
                                                         uint32_t* outcomes) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t lane = threadIdx.x & 63u;
    const bool live = i < n;
    bf_queue_push r{0xFFFFFFFFu, 0u};
    if (live) r = requests[i];
    uint32_t status = BF_PUSH_INVALID_CONTRACT;
    const bool grouped = live && r.queue_kind < BF_QUEUE_COUNT && qc_header_ok(q.headers[r.queue_kind], r.queue_kind, q.slot_stride);
    uint64_t pending = __ballot(grouped);
    while (pending != 0ull) {
        const uint32_t leader = (uint32_t)__ffsll((long long)pending) - 1u;
        const uint32_t kind = __shfl(r.queue_kind, (int)leader, 64);
        const uint64_t group = __ballot(grouped && r.queue_kind == kind) & pending;
        pending &= ~group;
        const uint32_t size = (uint32_t)__popcll(group);
        uint32_t base = 0u, accepted = 0u, valid = 1u;
        if (lane == leader) {
            bf_queue_header& h = q.headers[kind];
            uint32_t observed = __hip_atomic_load(&h.size, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            for (;;) {
                if (observed > h.capacity) {
                    valid = 0u;
                    break;
                }
                const uint32_t remaining = h.capacity - observed;
                accepted = remaining < size ? remaining : size;
                base = observed;
                if (accepted == 0u) break;
                const uint32_t previous = atomicCAS(&h.size, observed, observed + accepted);
                if (previous == observed) break;
                observed = previous;
            }
            if (valid) {
                qc_saturating_add(&h.overflow_count, size - accepted);
                qc_saturating_add(&h.rejected_count, size - accepted);
            }
        }
        base = __shfl(base, (int)leader, 64);
        accepted = __shfl(accepted, (int)leader, 64);
        valid = __shfl(valid, (int)leader, 64);
        if ((group >> lane) & 1ull) {
            const uint32_t rank = (uint32_t)__popcll(group & ((1ull << lane) - 1ull));
            if (!valid) {
                status = BF_PUSH_INVALID_CONTRACT;
            } else if (rank >= accepted) {
                status = BF_PUSH_CAPACITY_EXHAUSTED;
            } else {
                q.path_slots[(size_t)kind * q.slot_stride + base + rank] = r.slot;
                status = BF_PUSH_PUSHED;
            }
        }
    }
    if (live) outcomes[i] = status;
}

__global__ void k_qc_init(bf_queue_soa q, uint32_t route, uint32_t n, bf_compaction_result* result) {
    if (blockIdx.x != 0u || threadIdx.x != 0u) return;
    bf_compaction_result r;
    memset(&r, 0, sizeof r);
    r.status = BF_COMPACTION_SUCCESS;
    r.queue_kind = route;
    r.route = route;
    r.input_count = n;
    const bf_queue_header h = q.headers[route];
    r.initial_size = h.size;
    if (!qc_header_ok(h, route, q.slot_stride) || h.size > h.capacity || h.overflow_count != 0u || h.rejected_count != 0u)
        r.status = BF_COMPACTION_INVALID_CONTRACT;
    *result = r;
}

__global__ void k_qc_validate(const bf_stage_outcome* outcomes, uint32_t n, uint32_t route, uint32_t capacity,
                              bf_compaction_result* result) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const bf_stage_outcome o = outcomes[i];
    if (qc_selected(o, route) && o.path_slot >= capacity)
        atomicCAS(&result->status, (uint32_t)BF_COMPACTION_SUCCESS, (uint32_t)BF_COMPACTION_INVALID_CONTRACT);
}

/* selected outcomes per BF_BLOCK-item tile, from wave ballots */
__global__ __launch_bounds__(BF_BLOCK) void k_qc_count(const bf_stage_outcome* outcomes, uint32_t n, uint32_t route,
                                                       uint32_t* tile_counts) {
    __shared__ uint32_t waves[BF_BLOCK / 64u];
    const uint32_t tiles = (n + BF_BLOCK - 1u) / BF_BLOCK;
    for (uint32_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
        const uint32_t i = tile * BF_BLOCK + threadIdx.x;
        const bool sel = i < n && qc_selected(outcomes[i], route);
        const uint32_t c = (uint32_t)__popcll(__ballot(sel));
        if ((threadIdx.x & 63u) == 0u) waves[threadIdx.x >> 6] = c;
        __syncthreads();
        if (threadIdx.x == 0u) {
            uint32_t sum = 0u;
            for (uint32_t w = 0; w < BF_BLOCK / 64u; ++w) sum += waves[w];
            tile_counts[tile] = sum;
        }
        __syncthreads();
    }
}

/* one workgroup: exclusive scan of the tile counts, and their total */
__global__ __launch_bounds__(1024) void k_qc_scan(const uint32_t* tile_counts, uint32_t tiles, uint32_t* tile_offsets,
                                                  uint32_t* total) {
    __shared__ uint32_t partial[1024];
    const uint32_t t = threadIdx.x;
    const uint32_t per = (tiles + 1023u) / 1024u;
    const uint32_t begin = t * per < tiles ? t * per : tiles;
    const uint32_t end = begin + per < tiles ? begin + per : tiles;
    uint32_t own = 0u;
    for (uint32_t k = begin; k < end; ++k) own += tile_counts[k];
    partial[t] = own;
    __syncthreads();
    for (uint32_t off = 1u; off < 1024u; off <<= 1) {
        const uint32_t add = t >= off ? partial[t - off] : 0u;
        __syncthreads();
        partial[t] += add;
        __syncthreads();
    }
    uint32_t run = partial[t] - own;
    for (uint32_t k = begin; k < end; ++k) {
        tile_offsets[k] = run;
        run += tile_counts[k];
    }
    if (t == 1023u) *total = partial[1023];
}

/* the transactional capacity decision (CudaWavefrontQueueCompaction.cu:155-192) */
__global__ void k_qc_decide(bf_queue_soa q, const uint32_t* total, bf_compaction_result* result) {
    if (blockIdx.x != 0u || threadIdx.x != 0u) return;
    const uint32_t selected = *total;
    result->selected_count = selected;
    if (result->status != BF_COMPACTION_SUCCESS) return;
    bf_queue_header& h = q.headers[result->queue_kind];
    if (!qc_header_ok(h, result->queue_kind, q.slot_stride) || h.size != result->initial_size || h.overflow_count != 0u ||
        h.rejected_count != 0u) {
        result->status = BF_COMPACTION_INVALID_CONTRACT;
        return;
    }
    if (selected > h.capacity - h.size) {
        qc_saturating_add(&h.overflow_count, selected);
        qc_saturating_add(&h.rejected_count, selected);
        result->status = BF_COMPACTION_CAPACITY_EXHAUSTED;
        result->rejected_count = selected;
    }
}

/* stable scatter: rank = tile offset + earlier waves of the tile + earlier lanes of the wave */
__global__ __launch_bounds__(BF_BLOCK) void k_qc_scatter(bf_queue_soa q, const bf_stage_outcome* outcomes, uint32_t n,
                                                         uint32_t route, const uint32_t* tile_offsets,
                                                         const bf_compaction_result* result) {
    __shared__ uint32_t waves[BF_BLOCK / 64u];
    if (result->status != BF_COMPACTION_SUCCESS) return;
    const uint32_t tiles = (n + BF_BLOCK - 1u) / BF_BLOCK;
    const uint32_t lane = threadIdx.x & 63u;
    const size_t base = (size_t)result->queue_kind * q.slot_stride + result->initial_size;
    for (uint32_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
        const uint32_t i = tile * BF_BLOCK + threadIdx.x;
        bf_stage_outcome o{0u, 0u, 0u, 0u};
        if (i < n) o = outcomes[i];
        const bool sel = i < n && qc_selected(o, route);
        const uint64_t mask = __ballot(sel);
        if (lane == 0u) waves[threadIdx.x >> 6] = (uint32_t)__popcll(mask);
        __syncthreads();
        uint32_t rank = tile_offsets[tile];
        for (uint32_t w = 0; w < (threadIdx.x >> 6); ++w) rank += waves[w];
        rank += (uint32_t)__popcll(mask & ((1ull << lane) - 1ull));
        if (sel) q.path_slots[base + rank] = o.path_slot;
        __syncthreads();
    }
}

__global__ void k_qc_publish(bf_queue_soa q, bf_compaction_result* result) {
    if (blockIdx.x != 0u || threadIdx.x != 0u || result->status != BF_COMPACTION_SUCCESS) return;
    bf_queue_header& h = q.headers[result->queue_kind];
    if (!qc_header_ok(h, result->queue_kind, q.slot_stride) || h.size != result->initial_size || h.overflow_count != 0u ||
        h.rejected_count != 0u || result->selected_count > h.capacity - h.size) {
        result->status = BF_COMPACTION_INVALID_CONTRACT;
        return;
    }
    h.size += result->selected_count;
    result->published_count = result->selected_count;
}

__global__ void k_set_words(uint32_t* dst, uint32_t count, uint32_t value) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) dst[i] = value;
}

__global__ void k_copy_word(const uint32_t* src, uint32_t* dst) {
    if (threadIdx.x == 0 && blockIdx.x == 0) dst[0] = src[0];
}

__global__ void k_copy_words(const uint32_t* src, uint32_t* dst, uint32_t count) {
    for (uint32_t i = threadIdx.x; i < count; i += blockDim.x) dst[i] = src[i];
}

/* advances a replayed step counter (after the kernels that read it) */
__global__ void k_tick(uint32_t* counter) {
    if (threadIdx.x == 0 && blockIdx.x == 0) counter[0] += 1u;
}

/* Adds one launch's per-bounce queue sizes (rows of [ray, hit, shadow, continuation], ended by the
 * first empty ray queue) to totals [closest-hit queries, shade lanes, shadow queries, largest bounce
 * count]: the report of a launch whose host never reads its history. */
__global__ void k_history_totals(const uint32_t* history, uint32_t rows, unsigned long long* totals) {
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    unsigned long long ray = 0, hit = 0, shadow = 0;
    uint32_t active = 0;
    for (uint32_t b = 0; b < rows; ++b) {
        const uint32_t* h = history + 4 * b;
        if (h[0] == 0u) break;
        ray += h[0];
        hit += h[1];
        shadow += h[2];
        active = b + 1u;
    }
    totals[0] += ray;
    totals[1] += hit;
    totals[2] += shadow;
    if (active > totals[3]) totals[3] = active;
}

__global__ __launch_bounds__(BF_BLOCK) void k_export_paths(bf_dev_paths paths, bf_dev_job J) {
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= J.slot_count) return;
    const uint32_t i = J.slot_begin + k;
    bf_path_result* out = J.paths + J.path_base;
    bf_path_result r;
    const float4 L = paths.radiance[i], B = paths.beta[i], W = paths.wavelengths[i];
    const uint4 D = paths.depth[i];
    r.radiance[0] = L.x;
    r.radiance[1] = L.y;
    r.radiance[2] = L.z;
    r.radiance[3] = L.w;
    r.beta[0] = B.x;
    r.beta[1] = B.y;
    r.beta[2] = B.z;
    r.beta[3] = B.w;
    r.wavelengths[0] = W.x;
    r.wavelengths[1] = W.y;
    r.wavelengths[2] = W.z;
    r.wavelengths[3] = W.w;
    r.depth = D.y;
    r.termination = paths.status[i] & 0xFFu; /* the failure code stays in the workspace report */
    r.depth_counters = D.x;
    r.eta_scale = __uint_as_float(D.w);
    out[k] = r;
}

/* The terminal records of the path-input mode (WavefrontTransport.cpp:2753-2786): the path state
 * from the slot's columns (wavelength pdfs and measures pass through from the input), the ray the
 * path ended on (its first ray keeps the input's t_max, every later one runs to infinity), the ray
 * cone and a terminated lane control. A failed path returns zero records and termination NONE; its
 * failure is in the report. */
__global__ __launch_bounds__(BF_BLOCK) void k_export_path_records(bf_dev_paths paths, bf_dev_job J) {
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= J.slot_count) return;
    const uint32_t i = J.slot_begin + k;
    const uint64_t path = J.path_base + k;
    const uint32_t status = paths.status[i];
    const uint32_t termination = status & 0xFFu;
    bf_path_state_lane st;
    bf_transport_ray ray;
    float2 cone = make_float2(0.0f, 0.0f);
    memset(&st, 0, sizeof st);
    memset(&ray, 0, sizeof ray);
    bf_lane_control ctl;
    ctl.phase = BF_PHASE_TERMINATED;
    ctl.termination = 0u;
    ctl.flags = 0u;
    ctl.blocked_depth_limits = 0u;
    if (termination != BF_TERM_FAILED) {
        const bf_path_state_lane& in = J.in_states[path];
        const float4 B = paths.beta[i], L = paths.radiance[i], W = paths.wavelengths[i];
        const uint4 D = paths.depth[i];
        st.beta.values[0] = B.x;
        st.beta.values[1] = B.y;
        st.beta.values[2] = B.z;
        st.beta.values[3] = B.w;
        st.accumulated_radiance.values[0] = L.x;
        st.accumulated_radiance.values[1] = L.y;
        st.accumulated_radiance.values[2] = L.z;
        st.accumulated_radiance.values[3] = L.w;
        st.wavelength_nanometers.values[0] = W.x;
        st.wavelength_nanometers.values[1] = W.y;
        st.wavelength_nanometers.values[2] = W.z;
        st.wavelength_nanometers.values[3] = W.w;
        st.wavelength_pdf_values = in.wavelength_pdf_values;
#pragma unroll
        for (int w = 0; w < 4; ++w) st.wavelength_pdf_measures[w] = in.wavelength_pdf_measures[w];
        st.diffuse_depth = D.x & 0xFFu;
        st.glossy_depth = (D.x >> 8) & 0xFFu;
        st.specular_depth = (D.x >> 16) & 0xFFu;
        st.transmission_depth = D.x >> 24;
        st.depth = D.y;
        st.eta_scale = __uint_as_float(D.w);
        st.delta_flags = D.z & 3u;
        const float4 o = paths.ray_origin[i], d = paths.ray_direction[i];
        ray.origin_x = o.x;
        ray.origin_y = o.y;
        ray.origin_z = o.z;
        ray.t_min = d.w;
        ray.direction_x = d.x;
        ray.direction_y = d.y;
        ray.direction_z = d.z;
        ray.t_max = (D.z & BF_FIRST_RAY) != 0u ? J.in_rays[path].t_max : BF_INFINITY_F;
        ray.time = o.w;
        ray.visibility_mask = paths.visibility[i];
        cone = paths.cone[i];
        ctl.termination = termination;
        ctl.blocked_depth_limits = termination == BF_TERM_DEPTH_LIMIT ? status >> 8 : 0u;
    }
    J.out_states[path] = st;
    J.out_rays[path] = ray;
    J.out_cones[path] = bf_ray_cone{cone.x, cone.y};
    J.out_controls[path] = ctl;
}

/* ---- stage audit (CudaWavefrontStages.cu:4945-5033) -------------------------------------------
 * Each workgroup reduces its outcomes with wave ballots and shuffles into one partial (smallest
 * failing index, closure and light sample counts), written to the audit's reserved words through
 * atomics; a second one-wave launch on the same stream closes the audit (inspected count, first
 * failing outcome) and clears the words it used. */
BF_D bool outcome_failed(const bf_stage_outcome& o, uint32_t allowed_route_mask, uint32_t path_capacity) {
    if (o.status != BF_STAGE_SUCCESS || o.route > BF_ROUTE_TERMINATED) return true;
    return (allowed_route_mask & (1u << o.route)) == 0u || o.path_slot >= path_capacity;
}

__global__ void k_audit_init(uint32_t work_count, uint32_t stage_kind, bf_stage_audit* audit) {
    if (threadIdx.x != 0u) return;
    bf_stage_audit a;
    memset(&a, 0, sizeof a);
    a.abi_major = BF_STAGE_AUDIT_ABI_MAJOR;
    a.abi_minor = BF_STAGE_AUDIT_ABI_MINOR;
    a.struct_size = sizeof(bf_stage_audit);
    a.stage_kind = stage_kind;
    a.expected_work_count = work_count;
    a.first_failure_work_index = 0xFFFFFFFFu;
    *audit = a;
}

__global__ __launch_bounds__(BF_BLOCK) void k_audit_reduce(const bf_stage_outcome* outcomes, uint32_t work_count,
                                                           uint32_t allowed_route_mask, uint32_t path_capacity,
                                                           uint32_t shade, bf_stage_audit* audit) {
    __shared__ uint32_t wave_first[BF_BLOCK / 64], wave_closure[BF_BLOCK / 64], wave_light[BF_BLOCK / 64];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    uint32_t first = 0xFFFFFFFFu, closure = 0u, light = 0u;
    for (uint32_t i = blockIdx.x * BF_BLOCK + threadIdx.x; i < work_count; i += gridDim.x * BF_BLOCK) {
        const bf_stage_outcome o = outcomes[i];
        if (outcome_failed(o, allowed_route_mask, path_capacity)) first = min(first, i);
        if (shade) {
            closure += (o.detail & BF_SHADE_DETAIL_CLOSURE_SAMPLED) ? 1u : 0u;
            light += (o.detail & BF_SHADE_DETAIL_LIGHT_SAMPLED) ? 1u : 0u;
        }
    }
    for (int off = 32; off > 0; off >>= 1) {
        first = min(first, (uint32_t)__shfl_xor((int)first, off, 64));
        closure += (uint32_t)__shfl_xor((int)closure, off, 64);
        light += (uint32_t)__shfl_xor((int)light, off, 64);
    }
    if (lane == 0u) {
        wave_first[wave] = first;
        wave_closure[wave] = closure;
        wave_light[wave] = light;
    }
    __syncthreads();
    if (threadIdx.x == 0u) {
        for (uint32_t w = 1; w < BF_BLOCK / 64; ++w) {
            first = min(first, wave_first[w]);
            closure += wave_closure[w];
            light += wave_light[w];
        }
        if (first != 0xFFFFFFFFu) atomicMin(&audit->first_failure_work_index, first);
        if (closure) atomicAdd(&audit->closure_samples, closure);
        if (light) atomicAdd(&audit->light_samples, light);
    }
}

__global__ void k_audit_close(const bf_stage_outcome* outcomes, uint32_t work_count, bf_stage_audit* audit) {
    if (threadIdx.x != 0u) return;
    audit->inspected_work_count = work_count;
    const uint32_t f = audit->first_failure_work_index;
    if (f < work_count) {
        const bf_stage_outcome o = outcomes[f];
        audit->first_failure[0] = o.status;
        audit->first_failure[1] = o.route;
        audit->first_failure[2] = o.path_slot;
        audit->first_failure[3] = o.detail;
    }
}

/* ---- host-side launch helpers (stream-ordered, never synchronising) -------------------------- */
extern "C" {

hipError_t bfk_camera(const bf_transport_params* P, uint32_t count, uint32_t* ray_queue, uint8_t* route, bool batch,
                      bool adjoint, hipStream_t s) {
    if (count == 0) return hipSuccess;
    const dim3 grid(blocks_for(count, BF_BLOCK)), block(BF_BLOCK);
    if (batch && adjoint) hipLaunchKernelGGL((k_camera<true, true>), grid, block, 0, s, *P, count, ray_queue, route);
    else if (batch) hipLaunchKernelGGL((k_camera<true, false>), grid, block, 0, s, *P, count, ray_queue, route);
    else if (adjoint) hipLaunchKernelGGL((k_camera<false, true>), grid, block, 0, s, *P, count, ray_queue, route);
    else hipLaunchKernelGGL((k_camera<false, false>), grid, block, 0, s, *P, count, ray_queue, route);
    return hipGetLastError();
}

} /* extern "C" */

/* Workgroups of a partition: one tile each, until the counts that each of them adds up (`keys` words a
 * workgroup) would outweigh its items. */
static uint32_t partition_blocks(uint32_t max_count, uint32_t keys) {
    return std::min(blocks_for(max_count ? max_count : 1u, BF_PART_TILE), BF_PART_COUNTS / keys);
}

template <bool BATCH, uint32_t KEY>
static void launch_work_order(const bf_transport_params* P, const uint32_t* queue, const uint32_t* count_ptr,
                               uint32_t max_count, uint8_t* keys, uint32_t* order, hipStream_t s) {
    const dim3 grid(partition_blocks(max_count, BF_SHADE_BUCKETS));
    hipLaunchKernelGGL((k_bucket_count<BATCH, KEY>), grid, dim3(BF_BLOCK), 0, s, *P, queue, count_ptr, keys, P->bucket_counts);
    hipLaunchKernelGGL(k_bucket_scatter, grid, dim3(BF_BLOCK), 0, s, keys, count_ptr, P->bucket_counts, P->bucket_ranges, order);
}

/* max_count items' permutation grouped by `key` into `order`; `keys` holds one byte per item. */
extern "C" {

void bfk_work_order(const bf_transport_params* P, uint32_t key, const uint32_t* queue, const uint32_t* count_ptr,
                    uint32_t max_count, uint8_t* keys, uint32_t* order, bool batch, hipStream_t s) {
    const auto launch = [&](auto kernel) { kernel(P, queue, count_ptr, max_count, keys, order, s); };
    if (key == BF_KEY_SHADE) launch(batch ? launch_work_order<true, BF_KEY_SHADE> : launch_work_order<false, BF_KEY_SHADE>);
    else if (key == BF_KEY_RAY) launch(batch ? launch_work_order<true, BF_KEY_RAY> : launch_work_order<false, BF_KEY_RAY>);
    else launch(batch ? launch_work_order<true, BF_KEY_SHADOW> : launch_work_order<false, BF_KEY_SHADOW>);
}

bool bfk_shade_resident_blocks(int device, uint32_t* blocks) {
    return bfk_shade_blocks_plain(device, blocks + BF_SHADE_PLAIN * BF_SHADE_KERNELS) &&
           bfk_shade_blocks_textured(device, blocks + BF_SHADE_TEXTURED * BF_SHADE_KERNELS) &&
           bfk_shade_blocks_adjoint(device, blocks + BF_SHADE_ADJOINT * BF_SHADE_KERNELS) &&
           bfk_shade_blocks_mapped(device, blocks + BF_SHADE_MAPPED * BF_SHADE_KERNELS);
}

/* The kernels that the frames' materials need, in one order of the hit queue when it holds more than
 * one kind of item. */
uint32_t bfk_shade_plan(const bf_transport_params* P, bool* ordered) {
    const uint32_t mask = P->shade_buckets;
    const uint32_t single = mask >> BF_BUCKET_LAMBERT;
    uint32_t kernels = (mask & 0xFu) != 0u ? 1u << BF_SHADE_ANY : 0u;
    if (single != 0u) kernels |= single == 1u ? 1u << BF_SHADE_LAMBERT : 1u << BF_SHADE_SINGLE;
    const bool one_kind = (single & (single - 1u)) == 0u && ((mask & 0xFu) == 0u || single == 0u);
    *ordered = !one_kind || (P->shade_grouped != 0u && (mask & (mask - 1u)) != 0u);
    return kernels;
}

hipError_t bfk_shade(const bf_transport_params* P, const uint32_t* queue, const uint32_t* count_ptr, uint32_t max_count,
                     uint8_t* route, uint32_t* sample_counts, bool batch, uint32_t mode, hipStream_t s) {
    if (max_count == 0) return hipSuccess;
    bool ordered = false;
    const uint32_t kernels = bfk_shade_plan(P, &ordered);
    const uint32_t* order = nullptr;
    if (ordered) {
        /* the route bytes of the hit queue are free until shade writes them: they hold the keys */
        bfk_work_order(P, BF_KEY_SHADE, queue, count_ptr, max_count, route, P->shade_order, batch, s);
        order = P->shade_order;
    }
    const auto launch = mode == BF_SHADE_ADJOINT    ? bfk_shade_adjoint
                        : mode == BF_SHADE_TEXTURED ? bfk_shade_textured
                        : mode == BF_SHADE_MAPPED   ? bfk_shade_mapped
                                                    : bfk_shade_plain;
    for (uint32_t k = 0; k < BF_SHADE_KERNELS; ++k)
        if (kernels >> k & 1u) launch(P, k, queue, count_ptr, max_count, order, route, sample_counts, batch, s);
    return hipGetLastError();
}

int bfk_max_resident(const void* const* kernels, int count, uint32_t block, int device) {
    int cus = 0, per_cu = 0, m = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess || cus <= 0) return 0;
    for (int k = 0; k < count; ++k) {
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernels[k], (int)block, 0) != hipSuccess) return 0;
        if (per_cu > m) m = per_cu;
    }
    return cus * m;
}

hipError_t bfk_compact(const uint8_t* route, const uint32_t* count_ptr, uint32_t max_count, const uint32_t* src,
                       uint32_t* counts, uint32_t* dst1, uint32_t* size1, uint32_t append1, uint32_t* dst2, uint32_t* size2,
                       uint32_t append2, hipStream_t s) {
    const dim3 grid(partition_blocks(max_count, 2u));
    uint32_t* bases = counts + BF_PART_COUNTS;
    hipLaunchKernelGGL(k_compact_count, grid, dim3(BF_BLOCK), 0, s, route, count_ptr, counts, bases, size1, size2, append1,
                       append2);
    hipLaunchKernelGGL(k_compact_scatter, grid, dim3(BF_BLOCK), 0, s, route, count_ptr, src, counts, bases, dst1, dst2, size1,
                       size2);
    return hipGetLastError();
}

hipError_t bfk_bounce_end(uint32_t* sizes, uint32_t* history, uint32_t history_bounces, hipStream_t s) {
    hipLaunchKernelGGL(k_bounce_end, dim3(1), dim3(64), 0, s, sizes, history, history_bounces);
    return hipGetLastError();
}

hipError_t bfk_film(const bf_dev_paths* paths, const bf_dev_job* job, float pdf, float normalization, hipStream_t s) {
    hipLaunchKernelGGL(k_film, dim3(blocks_for(job->pixels, BF_BLOCK)), dim3(BF_BLOCK), 0, s, *paths, *job, pdf,
                       normalization);
    return hipGetLastError();
}

hipError_t bfk_queue_hash(const uint32_t* queue, const uint32_t* count_ptr, unsigned long long* out, hipStream_t s) {
    hipLaunchKernelGGL(k_queue_hash, dim3(1), dim3(64), 0, s, queue, count_ptr, out);
    return hipGetLastError();
}

hipError_t bfk_sample_dump(const sampler_ctx* sampler, const bf_sample_stream_index* indices,
                           const uint64_t* dimensions, uint32_t count, float* out, hipStream_t s) {
    if (count == 0) return hipSuccess;
    hipLaunchKernelGGL(k_sample_dump, dim3(blocks_for(count, BF_BLOCK)), dim3(BF_BLOCK), 0, s, *sampler, indices, dimensions, count,
                       out);
    return hipGetLastError();
}

hipError_t bfk_sample_stream_dump(const bf_sample_dump_request* requests, uint32_t count,
                                  bf_sample_dimension_manifest* manifest, bf_sample_dump_result* results) {
    hipLaunchKernelGGL(k_sample_stream_dump, dim3(blocks_for(count, BF_BLOCK)), dim3(BF_BLOCK), 0, nullptr, requests, count,
                       manifest, results);
    return hipGetLastError();
}

hipError_t bfk_reduce_replicas(const float* replicas, uint32_t offset, uint32_t count, float* dst, hipStream_t s) {
    if (count == 0) return hipSuccess;
    hipLaunchKernelGGL(k_reduce_replicas, dim3(blocks_for(count, BF_BLOCK)), dim3(BF_BLOCK), 0, s, replicas, offset, count, dst);
    return hipGetLastError();
}

hipError_t bfk_adam(float* value, const float* gradient, float* first, float* second, uint64_t count,
                    const bfk_adam_coefficients* c, const float2* schedule, const uint32_t* step, hipStream_t s) {
    if (count == 0) return hipSuccess;
    const bool vec = ((reinterpret_cast<uintptr_t>(value) | reinterpret_cast<uintptr_t>(gradient) |
                       reinterpret_cast<uintptr_t>(first) | reinterpret_cast<uintptr_t>(second)) & 15u) == 0;
    const uint64_t work = vec ? (count + 3u) / 4u : count;
    const uint32_t blocks = (uint32_t)std::min<uint64_t>((work + BF_BLOCK - 1u) / BF_BLOCK, 16384u);
    if (vec)
        hipLaunchKernelGGL(k_adam<true>, dim3(blocks), dim3(BF_BLOCK), 0, s, value, gradient, first, second, count, *c,
                           schedule, step);
    else
        hipLaunchKernelGGL(k_adam<false>, dim3(blocks), dim3(BF_BLOCK), 0, s, value, gradient, first, second, count, *c,
                           schedule, step);
    return hipGetLastError();
}

hipError_t bfk_film_l2(const float* film, const uint32_t* counts, const float* target, float* gradient, uint32_t pixels,
                       float two_scale, double scale, double* loss, hipStream_t s) {
    if (pixels == 0) return hipSuccess;
    hipLaunchKernelGGL(k_film_l2, dim3(blocks_for(pixels, BF_BLOCK)), dim3(BF_BLOCK), 0, s, film, counts, target, gradient,
                       pixels, two_scale, scale, loss);
    return hipGetLastError();
}

hipError_t bfk_zero_doubles(double* dst, uint32_t count, hipStream_t s) {
    if (count == 0) return hipSuccess;
    hipLaunchKernelGGL(k_zero_doubles, dim3(blocks_for(count, BF_BLOCK)), dim3(BF_BLOCK), 0, s, dst, count);
    return hipGetLastError();
}

hipError_t bfk_scene_soa_validate(const uint8_t* bytes, size_t count, uint32_t* status, hipStream_t s) {
    hipLaunchKernelGGL(k_scene_soa_validate, dim3(1), dim3(64), 0, s, (const bf_scene_soa_header*)bytes, (uint64_t)count, status);
    return hipGetLastError();
}

hipError_t bfk_scene_hash(const uint8_t* bytes, size_t count, uint64_t* out, hipStream_t s) {
    hipLaunchKernelGGL(k_scene_hash, dim3(1), dim3(64), 0, s, bytes, count, out);
    return hipGetLastError();
}

hipError_t bfk_queue_pushes(const bf_queue_soa* queues, const bf_queue_push* requests, uint32_t n, uint32_t* outcomes,
                            hipStream_t s) {
    if (n == 0u) return hipSuccess;
    hipLaunchKernelGGL(k_queue_push, dim3(blocks_for(n, BF_BLOCK)), dim3(BF_BLOCK), 0, s, *queues, requests, n, outcomes);
    return hipGetLastError();
}

hipError_t bfk_layout_manifest(bf_layout_manifest* out, hipStream_t s) {
    hipLaunchKernelGGL(k_layout_manifest, dim3(1), dim3(64), 0, s, out);
    return hipGetLastError();
}

static size_t align_scratch(size_t bytes) {
    return (bytes + BF_COMPACTION_SCRATCH_ALIGNMENT - 1u) / BF_COMPACTION_SCRATCH_ALIGNMENT * BF_COMPACTION_SCRATCH_ALIGNMENT;
}

size_t bfk_queue_compaction_scratch(uint32_t n) {
    if (n == 0u) return 0u;
    const size_t tiles = (n + BF_BLOCK - 1u) / BF_BLOCK;
    return 2u * align_scratch(tiles * sizeof(uint32_t)) + BF_COMPACTION_SCRATCH_ALIGNMENT;
}

hipError_t bfk_queue_compaction(const bf_queue_soa* queues, const bf_stage_outcome* outcomes, uint32_t n, uint32_t route,
                                void* scratch, bf_compaction_result* result, hipStream_t s) {
    const bf_queue_soa q = *queues;
    hipLaunchKernelGGL(k_qc_init, dim3(1), dim3(64), 0, s, q, route, n, result);
    if (n == 0u) return hipGetLastError();
    const uint32_t tiles = (n + BF_BLOCK - 1u) / BF_BLOCK;
    const size_t part = align_scratch((size_t)tiles * sizeof(uint32_t));
    uint8_t* base = static_cast<uint8_t*>(scratch);
    uint32_t* tile_counts = reinterpret_cast<uint32_t*>(base);
    uint32_t* tile_offsets = reinterpret_cast<uint32_t*>(base + part);
    uint32_t* total = reinterpret_cast<uint32_t*>(base + 2u * part);
    const dim3 grid(tiles < 4096u ? tiles : 4096u);
    hipLaunchKernelGGL(k_qc_validate, dim3(blocks_for(n, BF_BLOCK)), dim3(BF_BLOCK), 0, s, outcomes, n, route, q.slot_stride,
                       result);
    hipLaunchKernelGGL(k_qc_count, grid, dim3(BF_BLOCK), 0, s, outcomes, n, route, tile_counts);
    hipLaunchKernelGGL(k_qc_scan, dim3(1), dim3(1024), 0, s, tile_counts, tiles, tile_offsets, total);
    hipLaunchKernelGGL(k_qc_decide, dim3(1), dim3(64), 0, s, q, total, result);
    hipLaunchKernelGGL(k_qc_scatter, grid, dim3(BF_BLOCK), 0, s, q, outcomes, n, route, tile_offsets, result);
    hipLaunchKernelGGL(k_qc_publish, dim3(1), dim3(64), 0, s, q, result);
    return hipGetLastError();
}

/*
 * Library-owned compaction scratch for callers that cannot allocate: one copy per device, held
 * until the process ends. Its size serves BF_STATIC_COMPACTION_MAX_INPUT outcomes. In host code
 * `scratch` names a host-side stand-in, never the device array: every host use goes through the
 * address hipGetSymbolAddress returned for the current device. Nothing in it must start at zero
 * (the count kernel writes every tile it uses, the scan writes the total), and every call on a
 * device shares it, so calls that overlap on one device race.
 */
#define BF_STATIC_COMPACTION_SCRATCH_BYTES                                                                  \
    (2u * (((BF_STATIC_COMPACTION_MAX_INPUT / BF_BLOCK) * 4u + BF_COMPACTION_SCRATCH_ALIGNMENT - 1u) /     \
           BF_COMPACTION_SCRATCH_ALIGNMENT * BF_COMPACTION_SCRATCH_ALIGNMENT) +                             \
     BF_COMPACTION_SCRATCH_ALIGNMENT)
static __device__ __align__(256) uint8_t scratch[BF_STATIC_COMPACTION_SCRATCH_BYTES];

namespace {
constexpr int kStaticScratchDevices = 64;
std::mutex g_static_scratch_lock;
void* g_static_scratch[kStaticScratchDevices] = {};
} // namespace

hipError_t bfk_static_compaction_scratch(void** out) {
    *out = nullptr;
    int device = 0;
    hipError_t e = hipGetDevice(&device);
    if (e != hipSuccess) return e;
    if (device < 0 || device >= kStaticScratchDevices) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> guard(g_static_scratch_lock);
    if (g_static_scratch[device] == nullptr) {
        void* ptr = nullptr;
        e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        g_static_scratch[device] = ptr;
    }
    *out = g_static_scratch[device];
    return hipSuccess;
}

static_assert(BF_STATIC_COMPACTION_MAX_INPUT % BF_BLOCK == 0u, "the static scratch covers whole tiles");

hipError_t bfk_set_words(uint32_t* dst, uint32_t count, uint32_t value, hipStream_t s) {
    if (count == 0) return hipSuccess;
    hipLaunchKernelGGL(k_set_words, dim3(blocks_for(count, BF_BLOCK)), dim3(BF_BLOCK), 0, s, dst, count, value);
    return hipGetLastError();
}

hipError_t bfk_copy_words(const uint32_t* src, uint32_t* dst, uint32_t count, hipStream_t s) {
    hipLaunchKernelGGL(k_copy_words, dim3(1), dim3(64), 0, s, src, dst, count);
    return hipGetLastError();
}

hipError_t bfk_tick(uint32_t* counter, hipStream_t s) {
    hipLaunchKernelGGL(k_tick, dim3(1), dim3(64), 0, s, counter);
    return hipGetLastError();
}

hipError_t bfk_history_totals(const uint32_t* history, uint32_t rows, unsigned long long* totals, hipStream_t s) {
    hipLaunchKernelGGL(k_history_totals, dim3(1), dim3(64), 0, s, history, rows, totals);
    return hipGetLastError();
}

hipError_t bfk_copy_word(const uint32_t* src, uint32_t* dst, hipStream_t s) {
    hipLaunchKernelGGL(k_copy_word, dim3(1), dim3(64), 0, s, src, dst);
    return hipGetLastError();
}

hipError_t bfk_export_paths(const bf_dev_paths* paths, const bf_dev_job* job, hipStream_t s) {
    if (job->slot_count == 0 || !job->paths) return hipSuccess;
    hipLaunchKernelGGL(k_export_paths, dim3(blocks_for(job->slot_count, BF_BLOCK)), dim3(BF_BLOCK), 0, s, *paths, *job);
    return hipGetLastError();
}

hipError_t bfk_audit_stage(const bf_stage_outcome* outcomes, uint32_t work_count, uint32_t allowed_route_mask,
                           uint32_t path_capacity, uint32_t stage_kind, bf_stage_audit* audit, hipStream_t s) {
    hipLaunchKernelGGL(k_audit_init, dim3(1), dim3(64), 0, s, work_count, stage_kind, audit);
    if (work_count == 0u) return hipGetLastError();
    const uint32_t blocks = std::min<uint32_t>(blocks_for(work_count, BF_BLOCK), 2048u);
    hipLaunchKernelGGL(k_audit_reduce, dim3(blocks), dim3(BF_BLOCK), 0, s, outcomes, work_count, allowed_route_mask,
                       path_capacity, stage_kind == BF_STAGE_KIND_SHADE ? 1u : 0u, audit);
    hipLaunchKernelGGL(k_audit_close, dim3(1), dim3(64), 0, s, outcomes, work_count, audit);
    return hipGetLastError();
}

hipError_t bfk_export_path_records(const bf_dev_paths* paths, const bf_dev_job* job, hipStream_t s) {
    if (job->slot_count == 0 || !job->out_states) return hipSuccess;
    hipLaunchKernelGGL(k_export_path_records, dim3(blocks_for(job->slot_count, BF_BLOCK)), dim3(BF_BLOCK), 0, s, *paths,
                       *job);
    return hipGetLastError();
}

} /* extern "C" */
