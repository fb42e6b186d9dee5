/*
 * Traversal kernels: the closest-hit and shadow stages of a bounce, and the stand-alone ray queries
 * over prepared scenes and over the reference's device blobs.
 */
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "bf_paths.h"
#include "bf_scene_soa.h"
#include "bf_traversal.h"

/* ---- closest-hit stage: gather + traversal + classify + miss ---------------------------------- */
/* The traversal kernels are persistent: a grid sized to the device's resident capacity, whose waves claim
 * queue items until none is left (shared_claim), so that the per-lane stack spill area is bounded by the
 * grid and empty tail workgroups cost nothing. */

/* One lane's ray of a counting launch between traversal steps. */
struct lane_ray {
    uint32_t item, slot, status;
    trav_state ts;
    trav_hit best;
    bool occluded;
};

/* One lane's ray of any other launch. */
struct bound_ray {
    uint32_t item, slot, status;
    const bf_dev_scene* scene; /* batched launches: the ray's own scene */
    bound_state ts;
    bool occluded;
};

template <bool BATCH>
BF_D const bf_dev_scene& scene_of(const bf_transport_params& P, const bound_ray& L) {
    if constexpr (BATCH) return *L.scene;
    else return P.job0.scene;
}

/* A closest-hit ray's parameter range and visibility mask. */
BF_D void closest_range(const bf_transport_params& P, const bf_dev_job& J, uint32_t slot, float t_min, trav_ray& ray) {
    ray.t_min = t_min;
    ray.t_max = (P.paths.depth[slot].z & BF_FIRST_RAY) == 0u
                    ? BF_INFINITY_F
                    : (J.in_rays ? J.in_rays[path_of(J, slot)].t_max : J.camera.t_max);
    ray.mask = P.paths.visibility[slot];
}

/* World-space ray of a slot, re-read from the path columns (closest-hit rays): the step-exact walk
 * asks for (o, d) when it leaves a BLAS, the bound one for (d, mask) when it enters an instance. */
struct closest_world {
    const bf_dev_paths* paths;
    uint32_t slot;
    BF_D void operator()(v3f& o, v3f& d) const {
        const float4 a = paths->ray_origin[slot];
        const float4 b = paths->ray_direction[slot];
        o = mk(a.x, a.y, a.z);
        d = mk(b.x, b.y, b.z);
    }
    BF_D void operator()(v3f& d, uint32_t& mask) const {
        const float4 b = paths->ray_direction[slot];
        d = mk(b.x, b.y, b.z);
        mask = paths->visibility[slot];
    }
};

/* World-space shadow ray of a slot, from the pending-shadow columns. */
struct shadow_world {
    const bf_dev_paths* paths;
    uint32_t slot;
    BF_D void operator()(v3f& o, v3f& d) const {
        const float4 a = paths->shadow_origin[slot];
        const float4 b = paths->shadow_direction[slot];
        o = mk(a.x, a.y, a.z);
        d = mk(b.x, b.y, b.z);
    }
    BF_D void operator()(v3f& d, uint32_t& mask) const {
        const float4 b = paths->shadow_direction[slot];
        d = mk(b.x, b.y, b.z);
        mask = paths->visibility[slot];
    }
};

/* Reads queue item i's ray. */
template <bool ANY, bool BATCH>
BF_D const bf_dev_job& load_ray(const bf_transport_params& P, uint32_t slot, trav_ray& ray) {
    const bf_dev_job& J = job_at<BATCH>(P, slot);
    const float4 o = ANY ? P.paths.shadow_origin[slot] : P.paths.ray_origin[slot];
    const float4 d = ANY ? P.paths.shadow_direction[slot] : P.paths.ray_direction[slot];
    ray.o = mk(o.x, o.y, o.z);
    ray.d = mk(d.x, d.y, d.z);
    if (ANY) {
        ray.t_min = 0.0f;
        ray.t_max = o.w;
        ray.mask = P.paths.visibility[slot];
    } else {
        closest_range(P, J, slot, d.w, ray);
    }
    return J;
}

/* Classifies a finished closest-hit query: hit (route 1, barycentrics re-derived for the winner),
 * miss (environment radiance, path escapes) or traversal failure. */
template <bool BATCH>
BF_D void closest_finish(const bf_transport_params& P, uint8_t* route, uint32_t item, uint32_t slot, uint32_t st,
                         trav_hit& best) {
    const bf_dev_job& J = job_at<BATCH>(P, slot);
    if (st == BF_HIT_MISS && best.present) {
        const float4 o = P.paths.ray_origin[slot], d = P.paths.ray_direction[slot];
        trav_ray ray;
        closest_range(P, J, slot, d.w, ray);
        st = closest_hit_barycentrics(J.scene, mk(o.x, o.y, o.z), mk(d.x, d.y, d.z), ray.t_min, ray.t_max, best);
    }
    uint8_t r = 0;
    if (st != BF_HIT_MISS) {
        fail_path(P, J, slot, 60u + st);
    } else if (best.present) {
        P.paths.hit[slot] = make_float4(best.t, best.b0, best.b1, best.b2);
        P.paths.hit_ids[slot] = make_uint2(best.scene_instance, best.primitive);
        r = 1;
    } else {
        /* miss stage: CudaWavefrontStages.cu:3962-4040 */
        if (J.scene.has_environment) {
            const float4 wl = P.paths.wavelengths[slot];
            const float4 beta = P.paths.beta[slot];
            float4 Lr = P.paths.radiance[slot];
            const float w4[4] = {wl.x, wl.y, wl.z, wl.w};
            const float b4[4] = {beta.x, beta.y, beta.z, beta.w};
            float l4[4] = {Lr.x, Lr.y, Lr.z, Lr.w};
            bool ok = true;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                float product;
                const float radiance = spectrum_at(J.scene, J.scene.environment_spectrum, w4[k]);
                if (!checked_product(b4[k], radiance, product)) ok = false;
                else {
                    l4[k] += product;
                    if (!bf_isfinite(l4[k]) || l4[k] < 0.0f) ok = false;
                }
            }
            if (!ok) {
                fail_path(P, J, slot, 50);
            } else {
                P.paths.radiance[slot] = make_float4(l4[0], l4[1], l4[2], l4[3]);
                P.paths.status[slot] = BF_TERM_ESCAPED;
            }
        } else {
            P.paths.status[slot] = BF_TERM_ESCAPED;
        }
    }
    route[item] = r;
}

/*
 * The persistent lane loop shared by the traversal kernels. Every lane holds one ray; a lane whose
 * ray is done waits until REFILL lanes of its wave do (or none is left running). Then the waiting
 * rays are finished together and the wave claims as many queue items as it has idle lanes. A wave
 * therefore keeps working while any ray of the queue is unclaimed, and the finishing code
 * (barycentrics, environment lookup, shadow contribution) runs under wide masks: one lane at a
 * time it was about a third of a launch's vector instructions.
 *
 * Within a wave an iteration steps either the lanes whose next entry is an interior node or those
 * whose next entry is a leaf (once they are a LEAF-th of the running ones, or all of them), so one
 * kind of step code is issued at a time. Every ray's traversal is the same sequence of steps in
 * any schedule, so results do not depend on it.
 *
 * A launch with fewer items than its resident waves have lanes gives each wave an equal share
 * (`quota` lanes) instead of filling the first waves: the chip's other SIMDs would be idle, and
 * rays that share a wave wait for each other's steps.
 */
template <uint32_t REFILL, uint32_t LEAF, typename Claim, typename Start, typename Step, typename Finish>
BF_D void lane_loop(uint32_t n, Claim claim, Start start, Step step, Finish finish) {
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t quota = claim.quota, refill = (quota * REFILL + 63u) / 64u;
    bool active = false, done = false, exhausted = false;
    for (;;) {
        const uint64_t running = __ballot(active);
        const uint32_t count = (uint32_t)__popcll(running);
        if (count == 0u || (!exhausted && count + refill <= quota)) {
            if (done) {
                finish();
                done = false;
            }
            if (exhausted) break;
            const uint32_t want = quota - count;
            uint32_t end;
            const uint32_t base = claim(n, want, end, exhausted);
            if (!active) {
                const uint32_t rank = (uint32_t)__popcll(~running & ((1ull << lane) - 1ull));
                if (base < end && rank < end - base) {
                    active = start(base + rank);
                    done = !active;
                }
            }
            continue;
        }
        const bool leaf = active && step.leaf_next();
        const uint64_t leaves = __ballot(leaf);
        const bool leaf_phase = (uint32_t)__popcll(leaves) * LEAF >= count;
        if (leaf_phase) {
            if (leaf) step.leaf();
        } else if (active && !leaf) {
            step.node();
        }
        if (active && leaf == leaf_phase) {
            active = step.next();
            done = !active;
        }
    }
}

/*
 * How the waves of a launch claim its items. The queue is cut into BF_CLAIM_SEGMENTS contiguous
 * segments, and workgroup b starts in segment b mod BF_CLAIM_SEGMENTS: workgroups go to the eight
 * XCDs in turn, so each XCD works through its own part of the queue, whose neighbouring rays meet
 * neighbouring nodes, and its 4 MB L2 holds one part's nodes instead of every part's. A wave first
 * takes a fixed share of its segment's head, then draws from the segment's counter (one atomic per
 * refill), then from the other segments in turn. When the shares cover the queue nothing is drawn:
 * `quota` lanes of each wave hold the whole queue at once.
 */
struct shared_claim {
    uint32_t* fetch; /* the segments' counters */
    uint32_t per;    /* items of a segment (the last may have fewer) */
    uint32_t segment, segments;
    uint32_t wave, share_waves; /* the wave's number in its segment; waves of a full segment's share */
    uint32_t quota;
    uint32_t tried;
    bool opened, covered;
    BF_D uint32_t heads(uint32_t s) const {
        /* items of segment s given out as fixed shares */
        const uint32_t blocks = (gridDim.x - s + segments - 1u) / segments;
        return blocks * (blockDim.x / 64u) * quota;
    }
    /* items [result, end) are the wave's; at most `want` */
    BF_D uint32_t operator()(uint32_t n, uint32_t want, uint32_t& end, bool& exhausted) {
        if (!opened) {
            opened = true;
            exhausted = covered;
            const uint32_t base = segment * per + wave * quota;
            end = min(min(n, segment * per + per), base + want);
            return base;
        }
        for (; tried < segments; ++tried) {
            uint32_t drawn = 0u;
            if ((threadIdx.x & 63u) == 0u) drawn = atomicAdd(fetch + segment * BF_CLAIM_STRIDE, want);
            drawn = heads(segment) + __shfl(drawn, 0, 64);
            const uint32_t base = segment * per + drawn, stop = min(n, segment * per + per);
            if (drawn < per && base < stop) {
                end = min(stop, base + want);
                return base;
            }
            segment = segment + 1u == segments ? 0u : segment + 1u;
        }
        exhausted = true;
        end = 0u;
        return 0u;
    }
};

template <uint32_t BLOCK>
BF_D shared_claim wave_claim(uint32_t* fetch, uint32_t n) {
    shared_claim c;
    c.fetch = fetch;
    c.segments = gridDim.x < BF_CLAIM_SEGMENTS ? 1u : BF_CLAIM_SEGMENTS;
    c.per = (n + c.segments - 1u) / c.segments;
    c.segment = blockIdx.x % c.segments;
    c.wave = __builtin_amdgcn_readfirstlane(blockIdx.x / c.segments * (BLOCK / 64u) + (threadIdx.x >> 6));
    c.share_waves = gridDim.x / c.segments * (BLOCK / 64u);
    const uint32_t share = (c.per + c.share_waves - 1u) / c.share_waves;
    c.covered = share <= 64u;
    c.quota = share < 1u ? 1u : (share < 64u ? share : 64u);
    c.tried = 0u;
    c.opened = false;
    return c;
}

BF_D void reduce_counters(const trav_counters& c, unsigned long long* counters) {
    trav_counters ctr = c;
    for (int off = 32; off > 0; off >>= 1) {
        ctr.nodes += __shfl_down(ctr.nodes, off, 64);
        ctr.triangles += __shfl_down(ctr.triangles, off, 64);
        ctr.instances += __shfl_down(ctr.instances, off, 64);
    }
    if ((threadIdx.x & 63u) == 0u) {
        atomicAdd(&counters[0], (unsigned long long)ctr.nodes);
        atomicAdd(&counters[1], (unsigned long long)ctr.triangles);
        atomicAdd(&counters[2], (unsigned long long)ctr.instances);
    }
}

/* process_shadow (:4772-4908): the frozen contribution is added when the light is visible (and the
 * vertex's tape bit set), then the path continues or ends with its pending termination. */
template <bool BATCH>
BF_D void shadow_finish(const bf_transport_params& P, uint8_t* route, uint32_t item, uint32_t slot, uint32_t st,
                        bool occluded) {
    const bf_dev_job& J = job_at<BATCH>(P, slot);
    const uint32_t packed = __float_as_uint(P.paths.shadow_direction[slot].w);
    uint8_t r = 0;
    if (st != BF_HIT_MISS) {
        fail_path(P, J, slot, 40);
    } else {
        bool ok = true;
        if (!occluded) {
            if (J.tape_visibility) J.tape_visibility[path_of(J, slot)] |= 1ull << ((packed >> 16) & 63u);
            const float4 c = P.paths.shadow_contribution[slot];
            float4 Lr = P.paths.radiance[slot];
            Lr.x += c.x;
            Lr.y += c.y;
            Lr.z += c.z;
            Lr.w += c.w;
            if (!bf_isfinite(Lr.x) || !bf_isfinite(Lr.y) || !bf_isfinite(Lr.z) || !bf_isfinite(Lr.w) || Lr.x < 0.0f ||
                Lr.y < 0.0f || Lr.z < 0.0f || Lr.w < 0.0f) {
                ok = false;
                fail_path(P, J, slot, 41);
            } else {
                P.paths.radiance[slot] = Lr;
            }
        }
        if (ok) {
            if (packed & 1u) r = 2;
            else P.paths.status[slot] = (packed >> 8) & 0xFFu;
        }
    }
    route[item] = r;
}

/* ---- closest-hit and shadow stages: gather + traversal + finish ------------------------------
 * The step-exact, counting launch: every launch that counts its steps, and every one outside the bound
 * engine's range. Nodes and leaves step in separate iterations, and a lane's world-space reciprocals
 * wait in LDS for the end of each BLAS. Counted, 1024 instances at 1920x1080x4: 38.4 ms a frame; with
 * both kinds in one step, three binary64 divisions at each BLAS end and 208 bytes of spilled
 * registers a lane (6 waves per SIMD) 68.3. At 64 samples the closest hits take 216 ms and the shadow
 * rays 108 ms of a counted frame, 586 and 166 like that. Finishing each ray as it ends spares
 * registers, but loses more to the thin masks of the finishing code (236 and 102 ms at best). */
template <bool ANY, bool BATCH, uint32_t BLOCK>
__global__ __launch_bounds__(BLOCK, BF_COUNT_WAVES_PER_SIMD) void k_trace_counting(bf_transport_params P, const uint32_t* queue,
                                                                       const uint32_t* count_ptr, const uint32_t* order,
                                                                       uint8_t* route, unsigned long long* counters) {
    __shared__ uint2 s_stack[BF_SHORT_STACK * BLOCK];
    __shared__ double s_inv[3 * BLOCK];
    const uint32_t n = *count_ptr;
    using stack_t = trav_stack<BF_SHORT_STACK, BLOCK>;
    stack_t stack{
        s_stack + threadIdx.x, {P.spill + blockIdx.x * BLOCK + threadIdx.x, P.spill_stride}, 0u, 0u, BF_STACK_DEPTH};
    trav_counters ctr{0u, 0u, 0u};
    lane_ray L;
    using world_t = std::conditional_t<ANY, shadow_world, closest_world>;
    double* inv = s_inv + threadIdx.x;
    struct stepper {
        const bf_transport_params* P;
        stack_t* stack;
        lane_ray* L;
        trav_counters* ctr;
        const double* inv;
        BF_D bool leaf_next() const { return leaf_on_top(*stack); }
        BF_D const bf_dev_scene& scene() const { return job_at<BATCH>(*P, L->slot).scene; }
        BF_D bool pop(uint32_t& ref) const {
            return traverse_pop<ANY>(
                scene(),
                [&](trav_space& s) {
                    world_t{&P->paths, L->slot}(s.o, s.d);
                    for (uint32_t a = 0; a < 3u; ++a) s.inv[a] = inv[a * BLOCK];
                    finish_space(s);
                },
                *stack, L->ts, L->best, *ctr, ref);
        }
        BF_D void leaf() const {
            uint32_t ref;
            if (pop(ref)) L->status = traverse_leaf<ANY>(scene(), ref, *stack, L->ts, L->best, L->occluded, *ctr);
        }
        BF_D void node() const {
            uint32_t ref;
            if (pop(ref)) L->status = traverse_node<ANY>(scene(), ref, *stack, L->ts, L->best);
        }
        BF_D bool next() const {
            stack_refill(*stack);
            return L->status == BF_HIT_MISS && stack_depth(*stack) != 0u;
        }
    };
    lane_loop<BF_COUNT_REFILL, BF_COUNT_LEAF_PHASE>(
        n, wave_claim<BLOCK>(P.fetch + (ANY ? BF_CLAIM_SEGMENTS * BF_CLAIM_STRIDE : 0u), n),
        [&](uint32_t i) {
            L.item = order ? order[i] : i;
            L.slot = queue[L.item];
            trav_ray ray;
            const bf_dev_job& J = load_ray<ANY, BATCH>(P, L.slot, ray);
            L.status = traverse_begin(J.scene, ray, stack, L.ts, L.best, L.occluded, ctr);
            for (uint32_t a = 0; a < 3u; ++a) inv[a * BLOCK] = L.ts.space.inv[a];
            return L.status == BF_HIT_MISS && stack_depth(stack) != 0u;
        },
        stepper{&P, &stack, &L, &ctr, inv},
        [&] {
            if constexpr (ANY) shadow_finish<BATCH>(P, route, L.item, L.slot, L.status, L.occluded);
            else closest_finish<BATCH>(P, route, L.item, L.slot, L.status, L.best);
        });
    reduce_counters(ctr, counters + (ANY ? 3 : 0));
}

/* The launch every render takes: the walk on binary32 bounds. Bound by vector issue under
 * divergence. */
template <bool ANY, bool BATCH, uint32_t BLOCK>
__global__ __launch_bounds__(BLOCK, ANY ? BF_SHADOW_WAVES_PER_SIMD : BF_TRACE_WAVES_PER_SIMD) void k_trace(
    bf_transport_params P, const uint32_t* queue, const uint32_t* count_ptr, const uint32_t* order, uint8_t* route) {
    using entry_t = std::conditional_t<ANY, uint32_t, uint2>;
    __shared__ entry_t s_stack[(ANY ? BF_SHADOW_STACK : BF_SHORT_STACK) * BLOCK];
    __shared__ float s_world[6 * BLOCK];
    const uint32_t n = *count_ptr;
    using stack_t = ring_stack<entry_t, ANY ? BF_SHADOW_STACK : BF_SHORT_STACK, BLOCK, column_spill>;
    stack_t stack{reinterpret_cast<uint8_t*>(s_stack), threadIdx.x * (uint32_t)sizeof(entry_t),
                  {P.spill + blockIdx.x * BLOCK + threadIdx.x, P.spill_stride}, 0u, 0u};
    bound_ray L;
    using world_t = std::conditional_t<ANY, shadow_world, closest_world>;
    struct stepper {
        const bf_transport_params* P;
        stack_t* stack;
        bound_ray* L;
        const float* cache;
        BF_D bool leaf_next() const { return (L->ts.cur & BF_WIDE_LEAF) != 0u; }
        BF_D void node() const { bound_node(world_t{&P->paths, L->slot}, *stack, L->ts); }
        BF_D void leaf() const {
            L->status = bound_leaf<ANY>(scene_of<BATCH>(*P, *L), world_t{&P->paths, L->slot}, *stack, L->ts, L->occluded);
            if (L->status != BF_HIT_MISS) L->ts.cur = BF_TRAV_DONE;
        }
        BF_D bool next() const {
            bound_pop<ANY>(scene_of<BATCH>(*P, *L), *stack, L->ts, cache, BLOCK);
            return L->ts.cur != BF_TRAV_DONE;
        }
    };
    float* cache = s_world + threadIdx.x;
    lane_loop<ANY ? BF_SHADOW_REFILL : BF_TRACE_REFILL, ANY ? BF_SHADOW_LEAF_PHASE : BF_LEAF_PHASE>(
        n, wave_claim<BLOCK>(P.fetch + (ANY ? BF_CLAIM_SEGMENTS * BF_CLAIM_STRIDE : 0u), n),
        [&](uint32_t i) {
            L.item = order ? order[i] : i;
            L.slot = queue[L.item];
            L.status = BF_HIT_MISS;
            L.occluded = false;
            trav_ray ray;
            const bf_dev_job& J = load_ray<ANY, BATCH>(P, L.slot, ray);
            L.scene = &J.scene;
            bound_begin<ANY>(J.scene, ray.o, ray.d, ray.t_min, ray.t_max, stack, L.ts, cache, BLOCK);
            return L.ts.cur != BF_TRAV_DONE;
        },
        stepper{&P, &stack, &L, cache},
        [&] {
            if constexpr (ANY) {
                shadow_finish<BATCH>(P, route, L.item, L.slot, L.status, L.occluded);
            } else {
                trav_hit best;
                bound_result(scene_of<BATCH>(P, L), L.ts, best);
                closest_finish<BATCH>(P, route, L.item, L.slot, L.status, best);
            }
        });
}

/* ---- stand-alone traversal (blackframe_hip_launch_scene_closest_hit / _occlusion) ----------- */
/* A closest-hit record from the traversal's result. */
BF_D void closest_record(const bf_dev_scene& S, const trav_ray& ray, uint32_t st, trav_hit& best, bf_closest_hit_result& out) {
    memset(&out, 0, sizeof out);
    if (st == BF_HIT_MISS && best.present) st = closest_hit_barycentrics(S, ray.o, ray.d, ray.t_min, ray.t_max, best);
    if (st != BF_HIT_MISS) {
        out.status = st;
        return;
    }
    if (!best.present) return;
    const bf_dev_instance& I = S.instances[best.scene_instance];
    const float4 q0 = S.leaf_triangles[3 * (size_t)best.leaf + 0];
    const float4 q1 = S.leaf_triangles[3 * (size_t)best.leaf + 1];
    const float4 q2 = S.leaf_triangles[3 * (size_t)best.leaf + 2];
    v3f n;
    if (!world_normal(I.local_to_world, mk(q0.x, q0.y, q0.z), mk(q1.x, q1.y, q1.z), mk(q2.x, q2.y, q2.z), n)) {
        out.status = BF_HIT_NUMERICAL_FAILURE;
        return;
    }
    out.status = BF_HIT_HIT;
    out.hit.parameter = best.t;
    out.hit.barycentric0 = best.b0;
    out.hit.barycentric1 = best.b1;
    out.hit.barycentric2 = best.b2;
    out.hit.normal_x = n.x;
    out.hit.normal_y = n.y;
    out.hit.normal_z = n.z;
    out.hit.ids.object = I.object_id;
    out.hit.ids.instance = I.id;
    out.hit.ids.geometry = S.geometries[I.geometry_index].id;
    out.hit.ids.primitive = best.primitive;
    out.hit.ids.material = S.materials[I.material_index].id;
}

BF_D trav_ray api_ray(const bf_transport_ray& r) {
    trav_ray ray;
    ray.o = mk(r.origin_x, r.origin_y, r.origin_z);
    ray.d = mk(r.direction_x, r.direction_y, r.direction_z);
    ray.t_min = r.t_min;
    ray.t_max = r.t_max;
    ray.mask = r.visibility_mask;
    return ray;
}

/* World-space ray of a stand-alone query (see closest_world). */
struct api_world {
    const bf_transport_ray* ray;
    BF_D void operator()(v3f& d, uint32_t& mask) const {
        d = mk(ray->direction_x, ray->direction_y, ray->direction_z);
        mask = ray->visibility_mask;
    }
};

/* The step-exact walk, for queries that count their steps and scenes outside the bound engine's
 * range: one ray per lane with a 64-entry LDS stack and no spill area. A lane whose TLAS and BLAS
 * entries together exceed 64 reports stack overflow (the reference allows 64 per structure; a
 * median-split BVH never holds more than its depth + 1 entries per structure). */
template <bool ANY>
__global__ __launch_bounds__(BF_API_BLOCK) void k_scene_counting(bf_dev_scene S, const bf_transport_ray* rays, uint32_t count,
                                                                 void* results, uint32_t* counters) {
    __shared__ uint2 s_stack[BF_API_STACK * BF_API_BLOCK];
    trav_stack<BF_API_STACK, BF_API_BLOCK> stack{s_stack + threadIdx.x, {nullptr, 0u}, 0u, 0u, BF_API_STACK};
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count) return;
    const bf_transport_ray r = rays[i];
    trav_counters ctr{0u, 0u, 0u};
    trav_hit best;
    best.present = false;
    bool occluded = false;
    uint32_t st = BF_HIT_INVALID_RAY;
    const trav_ray ray = api_ray(r);
    const auto leave = [&](trav_space& s) {
        const trav_ray w = api_ray(rays[i]);
        make_space(w.o, w.d, s);
    };
    if (valid_traversal_ray(r)) st = traverse<ANY>(S, ray, leave, stack, best, occluded, ctr);
    if constexpr (ANY) {
        bf_occlusion_result out;
        memset(&out, 0, sizeof out);
        out.status = st != BF_HIT_MISS ? st : (occluded ? BF_OCCLUDED : BF_VISIBLE);
        ((bf_occlusion_result*)results)[i] = out;
    } else {
        bf_closest_hit_result out;
        closest_record(S, ray, st, best, out);
        ((bf_closest_hit_result*)results)[i] = out;
    }
    if (counters) {
        counters[3 * (size_t)i] = ctr.nodes;
        counters[3 * (size_t)i + 1] = ctr.triangles;
        counters[3 * (size_t)i + 2] = ctr.instances;
    }
}

/* Items of one wave's own chunk of the rays, claimed without atomics. */
struct chunk_claim {
    uint32_t next, quota;
    BF_D uint32_t operator()(uint32_t n, uint32_t want, uint32_t& end, bool& exhausted) {
        const uint32_t base = next;
        next += want;
        exhausted = base >= n || n - base <= want;
        end = exhausted ? n : base + want;
        return base;
    }
};

/* The bound walk over the caller's rays: one wave per workgroup, each with a chunk of consecutive
 * rays that it takes through lane_loop, so that a lane whose ray is done takes the chunk's next
 * ones. BF_SHORT_STACK entries of the stack are in LDS, the rest (deep walks only) in the lane's
 * scratch: a full 64-entry LDS stack holds the CU to 5 waves, and this walk is bound by vector
 * issue and latency under divergence. */
template <bool ANY>
__global__ __launch_bounds__(BF_API_BLOCK, BF_TRACE_WAVES_PER_SIMD) void k_scene_trace(
    bf_dev_scene S, const bf_transport_ray* rays, uint32_t count, uint32_t chunk, void* results) {
    using entry_t = std::conditional_t<ANY, uint32_t, uint2>;
    __shared__ entry_t s_stack[(ANY ? BF_SHADOW_STACK : BF_SHORT_STACK) * BF_API_BLOCK];
    __shared__ float s_world[6 * BF_API_BLOCK];
    using stack_t = ring_stack<entry_t, ANY ? BF_SHADOW_STACK : BF_SHORT_STACK, BF_API_BLOCK, scratch_spill>;
    uint32_t spilled[ANY ? 1 : 2][BF_STACK_DEPTH];
    stack_t stack{reinterpret_cast<uint8_t*>(s_stack), threadIdx.x * (uint32_t)sizeof(entry_t),
                  {spilled[0], spilled[ANY ? 0 : 1]}, 0u, 0u};
    bound_state ts;
    uint32_t item = 0u, status = BF_HIT_MISS;
    bool occluded = false;
    float* cache = s_world + threadIdx.x;
    struct stepper {
        const bf_dev_scene* S;
        const bf_transport_ray* rays;
        stack_t* stack;
        bound_state* ts;
        uint32_t *item, *status;
        bool* occluded;
        const float* cache;
        BF_D bool leaf_next() const { return (ts->cur & BF_WIDE_LEAF) != 0u; }
        BF_D void node() const { bound_node(api_world{rays + *item}, *stack, *ts); }
        BF_D void leaf() const {
            *status = bound_leaf<ANY>(*S, api_world{rays + *item}, *stack, *ts, *occluded);
            if (*status != BF_HIT_MISS) ts->cur = BF_TRAV_DONE;
        }
        BF_D bool next() const {
            bound_pop<ANY>(*S, *stack, *ts, cache, BF_API_BLOCK);
            return ts->cur != BF_TRAV_DONE;
        }
    };
    const uint32_t begin = blockIdx.x * chunk;
    const uint32_t end = count - begin < chunk ? count : begin + chunk;
    lane_loop<ANY ? BF_SHADOW_REFILL : BF_TRACE_REFILL, ANY ? BF_SHADOW_LEAF_PHASE : BF_LEAF_PHASE>(
        end, chunk_claim{begin, chunk < 64u ? chunk : 64u},
        [&](uint32_t i) {
            item = i;
            status = BF_HIT_INVALID_RAY;
            occluded = false;
            ts.hit_leaf = BF_INVALID_INDEX;
            const bf_transport_ray r = rays[i];
            if (!valid_traversal_ray(r)) return false;
            status = BF_HIT_MISS;
            const trav_ray ray = api_ray(r);
            bound_begin<ANY>(S, ray.o, ray.d, ray.t_min, ray.t_max, stack, ts, cache, BF_API_BLOCK);
            return ts.cur != BF_TRAV_DONE;
        },
        stepper{&S, rays, &stack, &ts, &item, &status, &occluded, cache},
        [&] {
            if constexpr (ANY) {
                bf_occlusion_result out;
                memset(&out, 0, sizeof out);
                out.status = status != BF_HIT_MISS ? status : (occluded ? BF_OCCLUDED : BF_VISIBLE);
                ((bf_occlusion_result*)results)[item] = out;
            } else {
                trav_hit best;
                bound_result(S, ts, best);
                bf_closest_hit_result out;
                closest_record(S, api_ray(rays[item]), status, best, out);
                ((bf_closest_hit_result*)results)[item] = out;
            }
        });
}

/* ---- stand-alone traversal over the reference's device blobs ----------------------------------
 * blackframe_hip_launch_scene_closest_hit_blob / _occlusion_blob take the reference launcher's
 * arguments (SceneClosestHit.hpp, CudaSceneClosestHit.cu:188-1330): "BLKFSOA4" scene bytes and a
 * "BLKFBVH1" BVH in device memory. The first lane of every workgroup validates both layouts
 * (validate_scene_layout / validate_bvh_layout, :199-358) and a bad one answers every ray of the
 * workgroup with invalid_scene / invalid_bvh. Each lane then traverses one ray over the canonical
 * 48-byte nodes in the reference's order: pop, re-test the node's own box against the current
 * t_max, push both intersecting children far then near (ties to the first), enter an instance leaf
 * in object space after checking it against the scene's columns, and test a BLAS leaf's triangle
 * from the scene's index and position columns. The box and triangle decisions are this library's
 * binary64 slab and watertight test, so the results equal those of
 * blackframe_hip_launch_scene_closest_hit on the scene the blobs describe. The TLAS and each BLAS
 * get their own 64-entry LDS stack, as in the reference. */
struct blob_view {
    const uint8_t* scene;
    const bf_scene_soa_header* sh;
    const uint8_t* bvh;
    const bf_bvh_header* bh;
};

template <typename T>
BF_D const T* soa_col(const blob_view& b, uint32_t column) {
    return (const T*)(b.scene + b.sh->columns[column].offset_bytes);
}

template <typename T>
BF_D const T* bvh_arr(const blob_view& b, uint32_t array) {
    return (const T*)(b.bvh + b.bh->arrays[array].offset_bytes);
}

BF_D uint64_t blob_align(uint64_t v, uint64_t a) { return (v + a - 1u) / a * a; }

/* validate_scene_layout (:199-250) */
BF_D uint32_t blob_scene_layout(const uint8_t* bytes, size_t n) {
    if (n < sizeof(bf_scene_soa_header)) return BF_HIT_INVALID_SCENE;
    const bf_scene_soa_header& h = *(const bf_scene_soa_header*)bytes;
    if (h.magic != BF_SCENE_SOA_MAGIC || h.abi_major != BF_SCENE_SOA_ABI_MAJOR || h.abi_minor != BF_SCENE_SOA_ABI_MINOR ||
        h.header_size != sizeof(bf_scene_soa_header) || h.column_count != BF_SCENE_SOA_COLUMN_COUNT ||
        h.hash_algorithm != BF_SCENE_SOA_HASH_FNV1A64 || h.environment_count > 1u || h.total_size_bytes != n ||
        h.total_size_bytes < sizeof(bf_scene_soa_header) || h.texture_count > 0xFFFFFFFFull ||
        h.image_texture_count > 0xFFFFFFFFull || h.image_mip_count > 0xFFFFFFFFull)
        return BF_HIT_INVALID_SCENE;
    for (int k = 0; k < 5; ++k)
        if (h.reserved[k] != 0u) return BF_HIT_INVALID_SCENE;
    const uint64_t max = ~0ull;
    uint64_t cursor = blob_align(sizeof(bf_scene_soa_header), BF_SCENE_SOA_COLUMN_ALIGNMENT);
    for (uint32_t c = 0; c < BF_SCENE_SOA_COLUMN_COUNT; ++c) {
        const bf_scene_soa_column& d = h.columns[c];
        const uint64_t count = bf_soa::column_count(h, c);
        const uint64_t size = bf_soa::column_element_size(c);
        if (d.element_count != count || d.element_size != size || d.reserved != 0u) return BF_HIT_INVALID_SCENE;
        if (count == 0u) {
            if (d.offset_bytes != 0u) return BF_HIT_INVALID_SCENE;
            continue;
        }
        if (cursor > max - (BF_SCENE_SOA_COLUMN_ALIGNMENT - 1u)) return BF_HIT_INVALID_SCENE;
        cursor = blob_align(cursor, BF_SCENE_SOA_COLUMN_ALIGNMENT);
        if (d.offset_bytes != cursor || count > max / size) return BF_HIT_INVALID_SCENE;
        const uint64_t bytes_in_column = count * size;
        if (cursor > max - bytes_in_column) return BF_HIT_INVALID_SCENE;
        cursor += bytes_in_column;
    }
    return cursor == h.total_size_bytes ? BF_HIT_MISS : BF_HIT_INVALID_SCENE;
}

/* validate_bvh_layout (:291-358) */
BF_D uint32_t blob_bvh_layout(const uint8_t* bytes, size_t n, const bf_scene_soa_header& scene) {
    if (n < sizeof(bf_bvh_header)) return BF_HIT_INVALID_BVH;
    const bf_bvh_header& h = *(const bf_bvh_header*)bytes;
    const uint64_t invalid = BF_INVALID_INDEX;
    if (h.magic != BF_BVH_MAGIC || h.abi_major != BF_BVH_ABI_MAJOR || h.abi_minor != BF_BVH_ABI_MINOR ||
        h.header_size != sizeof(bf_bvh_header) || h.array_count != BF_BVH_ARRAY_COUNT ||
        h.hash_algorithm != BF_BVH_HASH_FNV1A64 || h.leaf_capacity != BF_BVH_LEAF_CAPACITY || h.total_size_bytes != n ||
        h.total_size_bytes < sizeof(bf_bvh_header) || h.source_scene_hash != scene.content_hash ||
        h.blas_count != scene.geometry_count || h.primitive_reference_count != scene.triangle_count ||
        h.instance_reference_count != scene.instance_count || h.blas_count > invalid || h.blas_node_count > invalid ||
        h.primitive_reference_count > invalid || h.tlas_node_count > invalid || h.instance_reference_count > invalid)
        return BF_HIT_INVALID_BVH;
    if ((h.blas_count == 0u && (h.blas_node_count != 0u || h.primitive_reference_count != 0u)) ||
        (h.blas_count != 0u && (h.primitive_reference_count < h.blas_count ||
                                h.blas_node_count != h.primitive_reference_count * 2u - h.blas_count)) ||
        (h.instance_reference_count == 0u && h.tlas_node_count != 0u) ||
        (h.instance_reference_count != 0u && h.tlas_node_count != h.instance_reference_count * 2u - 1u) ||
        (h.tlas_node_count == 0u && h.tlas_root_node != BF_INVALID_INDEX) ||
        (h.tlas_node_count != 0u && h.tlas_root_node != 0u))
        return BF_HIT_INVALID_BVH;
    for (int k = 0; k < 5; ++k)
        if (h.reserved[k] != 0u) return BF_HIT_INVALID_BVH;
    const uint64_t counts[BF_BVH_ARRAY_COUNT] = {h.blas_count, h.blas_node_count, h.primitive_reference_count,
                                                 h.tlas_node_count, h.instance_reference_count};
    const uint64_t sizes[BF_BVH_ARRAY_COUNT] = {sizeof(bf_bvh_blas), sizeof(bf_bvh_node), sizeof(uint32_t),
                                                sizeof(bf_bvh_node), sizeof(bf_bvh_instance_ref)};
    const uint64_t max = ~0ull;
    uint64_t cursor = blob_align(sizeof(bf_bvh_header), BF_BVH_ARRAY_ALIGNMENT);
    for (uint32_t a = 0; a < BF_BVH_ARRAY_COUNT; ++a) {
        const bf_bvh_array_descriptor& d = h.arrays[a];
        if (d.element_count != counts[a] || d.element_size != sizes[a] || d.reserved != 0u) return BF_HIT_INVALID_BVH;
        if (counts[a] == 0u) {
            if (d.offset_bytes != 0u) return BF_HIT_INVALID_BVH;
            continue;
        }
        if (cursor > max - (BF_BVH_ARRAY_ALIGNMENT - 1u)) return BF_HIT_INVALID_BVH;
        cursor = blob_align(cursor, BF_BVH_ARRAY_ALIGNMENT);
        if (d.offset_bytes != cursor || counts[a] > max / sizes[a]) return BF_HIT_INVALID_BVH;
        const uint64_t bytes_in_array = counts[a] * sizes[a];
        if (cursor > max - bytes_in_array) return BF_HIT_INVALID_BVH;
        cursor += bytes_in_array;
    }
    return cursor == h.total_size_bytes ? BF_HIT_MISS : BF_HIT_INVALID_BVH;
}

/* intersect_bounds (:407-455): the node's box, validated, in the reference's binary64 slab */
BF_D uint32_t blob_box(const bf_bvh_node& n, const trav_space& s, float t_min, float t_max, bool& hit, float& nearv) {
    if (!bf_isfinite(n.min_x) || !bf_isfinite(n.min_y) || !bf_isfinite(n.min_z) || !bf_isfinite(n.max_x) ||
        !bf_isfinite(n.max_y) || !bf_isfinite(n.max_z) || n.min_x > n.max_x || n.min_y > n.max_y || n.min_z > n.max_z)
        return BF_HIT_INVALID_TOPOLOGY;
    double v = 0.0;
    const uint32_t st = slab_exact(n.min_x, n.min_y, n.min_z, n.max_x, n.max_y, n.max_z, s, t_min, t_max, hit, v);
    nearv = (float)v;
    return st;
}

/* push_intersecting_children (:466-512) */
BF_D uint32_t blob_push_children(const bf_bvh_node* nodes, const bf_bvh_node& n, uint32_t begin, uint32_t count,
                                 const trav_space& s, float t_min, float t_max, uint32_t* stack, uint32_t& size) {
    const uint64_t end = (uint64_t)begin + count;
    const uint32_t a = n.first_child, b = n.second_child;
    if (a == b || a < begin || b < begin || a >= end || b >= end) return BF_HIT_INVALID_TOPOLOGY;
    bool ha, hb;
    float na = 0.0f, nb = 0.0f;
    uint32_t st = blob_box(nodes[a], s, t_min, t_max, ha, na);
    if (st != BF_HIT_MISS) return st;
    st = blob_box(nodes[b], s, t_min, t_max, hb, nb);
    if (st != BF_HIT_MISS) return st;
    if (!ha && !hb) return BF_HIT_MISS;
    if (ha != hb) {
        if (size >= BF_STRUCTURE_STACK) return BF_HIT_STACK_OVERFLOW;
        stack[(size++) * BF_API_BLOCK] = ha ? a : b;
        return BF_HIT_MISS;
    }
    const bool a_near = na < nb || (na == nb && a < b);
    if (size >= BF_STRUCTURE_STACK) return BF_HIT_STACK_OVERFLOW;
    stack[(size++) * BF_API_BLOCK] = a_near ? b : a;
    if (size >= BF_STRUCTURE_STACK) return BF_HIT_STACK_OVERFLOW;
    stack[(size++) * BF_API_BLOCK] = a_near ? a : b;
    return BF_HIT_MISS;
}

/* a 3x4 affine matrix from one of the scene's 16-element matrix column groups (:513-537) */
BF_D uint32_t blob_matrix(const blob_view& b, uint32_t first_column, uint32_t instance, float* m) {
    float full[16];
    for (uint32_t e = 0; e < 16u; ++e) {
        full[e] = soa_col<float>(b, first_column + e)[instance];
        if (!bf_isfinite(full[e])) return BF_HIT_NUMERICAL_FAILURE;
    }
    if (full[12] != 0.0f || full[13] != 0.0f || full[14] != 0.0f || full[15] != 1.0f) return BF_HIT_INVALID_TOPOLOGY;
    for (uint32_t e = 0; e < 12u; ++e) m[e] = full[e];
    return BF_HIT_MISS;
}

struct blob_candidate {
    bool present;
    float t;
    uint32_t instance_id, primitive;
    bf_closest_hit hit;
};

/* traverse_blas (:895-1085) */
template <bool ANY>
BF_D uint32_t blob_blas(const blob_view& b, const bf_bvh_instance_ref& ref, const bf_transport_ray& ray, v3f lo, v3f ld,
                        uint32_t* stack, blob_candidate& best, bool& occluded) {
    const bf_bvh_blas* blases = bvh_arr<bf_bvh_blas>(b, 0);
    const bf_bvh_node* nodes = bvh_arr<bf_bvh_node>(b, 1);
    const uint32_t* prims = bvh_arr<uint32_t>(b, 2);
    if (ref.blas_index >= b.bh->blas_count || ref.scene_geometry_index >= b.sh->geometry_count)
        return BF_HIT_INVALID_TOPOLOGY;
    const bf_bvh_blas B = blases[ref.blas_index];
    const uint64_t node_end = (uint64_t)B.node_offset + B.node_count;
    const uint64_t ref_end = (uint64_t)B.primitive_reference_offset + B.primitive_reference_count;
    if (B.reserved[0] != 0u || B.reserved[1] != 0u || B.geometry_id != ref.geometry_id || B.root_node != B.node_offset ||
        B.node_count == 0u || node_end > b.bh->blas_node_count ||
        B.node_count != (uint64_t)B.primitive_reference_count * 2u - 1u || ref_end > b.bh->primitive_reference_count)
        return BF_HIT_INVALID_TOPOLOGY;
    const uint32_t g = ref.scene_geometry_index;
    const uint64_t vertex_offset = soa_col<uint64_t>(b, bf_soa::C_GEOMETRY_VERTEX_OFFSET)[g];
    const uint64_t vertex_count = soa_col<uint64_t>(b, bf_soa::C_GEOMETRY_VERTEX_COUNT)[g];
    const uint64_t triangle_offset = soa_col<uint64_t>(b, bf_soa::C_GEOMETRY_TRIANGLE_OFFSET)[g];
    const uint64_t triangle_count = soa_col<uint64_t>(b, bf_soa::C_GEOMETRY_TRIANGLE_COUNT)[g];
    if (soa_col<uint32_t>(b, bf_soa::C_GEOMETRY_ID)[g] != ref.geometry_id || triangle_count != B.primitive_reference_count ||
        vertex_count == 0u || vertex_offset > b.sh->vertex_count || vertex_count > b.sh->vertex_count - vertex_offset ||
        triangle_offset > b.sh->triangle_count || triangle_count > b.sh->triangle_count - triangle_offset)
        return BF_HIT_INVALID_TOPOLOGY;
    trav_space s;
    make_space(lo, ld, s);
    trav_shear sh;
    make_shear(ld, sh);
    uint32_t size = 0, visited = 0;
    stack[(size++) * BF_API_BLOCK] = B.root_node;
    while (size != 0u) {
        if (visited++ >= B.node_count) return BF_HIT_INVALID_TOPOLOGY;
        const uint32_t index = stack[(--size) * BF_API_BLOCK];
        if (index < B.node_offset || index >= node_end) return BF_HIT_INVALID_TOPOLOGY;
        const bf_bvh_node n = nodes[index];
        const float t_max = ANY ? ray.t_max : best.t;
        bool h;
        float nearv;
        uint32_t st = blob_box(n, s, ray.t_min, t_max, h, nearv);
        if (st != BF_HIT_MISS) return st;
        if (!h) continue;
        if (n.kind == 0u) {
            if (n.split_axis > 2u || n.reference_offset != 0u || n.reference_count != 0u) return BF_HIT_INVALID_TOPOLOGY;
            st = blob_push_children(nodes, n, B.node_offset, B.node_count, s, ray.t_min, t_max, stack, size);
            if (st != BF_HIT_MISS) return st;
            continue;
        }
        if (n.kind != 1u || n.split_axis != BF_INVALID_INDEX || n.first_child != BF_INVALID_INDEX ||
            n.second_child != BF_INVALID_INDEX || n.reference_count != 1u || n.reference_offset < B.primitive_reference_offset ||
            n.reference_offset >= ref_end)
            return BF_HIT_INVALID_TOPOLOGY;
        const uint32_t prim = prims[n.reference_offset];
        if (prim >= triangle_count) return BF_HIT_INVALID_TOPOLOGY;
        const uint64_t tri = triangle_offset + prim;
        v3f v[3];
        for (uint32_t c = 0; c < 3u; ++c) {
            const uint32_t local = soa_col<uint32_t>(b, bf_soa::C_TRIANGLE_VERTEX_0 + c)[tri];
            if (local >= vertex_count) return BF_HIT_INVALID_TOPOLOGY;
            const uint64_t gv = vertex_offset + local;
            v[c] = mk(soa_col<float>(b, bf_soa::C_POSITION_X)[gv], soa_col<float>(b, bf_soa::C_POSITION_X + 1)[gv],
                      soa_col<float>(b, bf_soa::C_POSITION_X + 2)[gv]);
            if (!fin3(v[c])) return BF_HIT_NUMERICAL_FAILURE;
        }
        tri_result tr;
        tr.hit = false;
        st = watertight<!ANY>(v[0], v[1], v[2], lo, ld, sh, ray.t_min, t_max, tr);
        if (st != BF_HIT_MISS) return st;
        if (!tr.hit) continue;
        if (ANY) {
            occluded = true;
            return BF_HIT_MISS;
        }
        if (best.present && !(tr.t < best.t ||
                              (tr.t == best.t && (ref.instance_id < best.instance_id ||
                                                  (ref.instance_id == best.instance_id && prim < best.primitive)))))
            continue;
        float m[12];
        st = blob_matrix(b, bf_soa::C_INSTANCE_LOCAL_TO_WORLD, ref.scene_instance_index, m);
        if (st != BF_HIT_MISS) return st;
        v3f nrm;
        if (!world_normal(m, v[0], v[1], v[2], nrm)) return BF_HIT_NUMERICAL_FAILURE;
        const uint32_t inst = ref.scene_instance_index;
        if (soa_col<uint32_t>(b, bf_soa::C_INSTANCE_ID)[inst] != ref.instance_id ||
            soa_col<uint32_t>(b, bf_soa::C_INSTANCE_GEOMETRY_ID)[inst] != ref.geometry_id)
            return BF_HIT_INVALID_TOPOLOGY;
        best.present = true;
        best.t = tr.t;
        best.instance_id = ref.instance_id;
        best.primitive = prim;
        bf_closest_hit& hr = best.hit;
        memset(&hr, 0, sizeof hr);
        hr.parameter = tr.t;
        hr.barycentric0 = tr.b0;
        hr.barycentric1 = tr.b1;
        hr.barycentric2 = tr.b2;
        hr.normal_x = nrm.x;
        hr.normal_y = nrm.y;
        hr.normal_z = nrm.z;
        hr.ids.object = soa_col<uint32_t>(b, bf_soa::C_INSTANCE_OBJECT_ID)[inst];
        hr.ids.instance = ref.instance_id;
        hr.ids.geometry = ref.geometry_id;
        hr.ids.primitive = prim;
        hr.ids.material = soa_col<uint32_t>(b, bf_soa::C_INSTANCE_MATERIAL_ID)[inst];
    }
    return BF_HIT_MISS;
}

/* trace_scene (:1087-1186) */
template <bool ANY>
BF_D uint32_t blob_trace(const blob_view& b, const bf_transport_ray& ray, uint32_t* tlas_stack, uint32_t* blas_stack,
                         blob_candidate& best, bool& occluded) {
    if (b.bh->tlas_node_count == 0u) return BF_HIT_MISS;
    const bf_bvh_node* nodes = bvh_arr<bf_bvh_node>(b, 3);
    const bf_bvh_instance_ref* refs = bvh_arr<bf_bvh_instance_ref>(b, 4);
    const uint32_t tlas_count = (uint32_t)b.bh->tlas_node_count;
    trav_space world;
    const v3f o = mk(ray.origin_x, ray.origin_y, ray.origin_z), d = mk(ray.direction_x, ray.direction_y, ray.direction_z);
    make_space(o, d, world);
    uint32_t size = 0, visited = 0;
    tlas_stack[(size++) * BF_API_BLOCK] = b.bh->tlas_root_node;
    while (size != 0u) {
        if (visited++ >= tlas_count) return BF_HIT_INVALID_TOPOLOGY;
        const uint32_t index = tlas_stack[(--size) * BF_API_BLOCK];
        if (index >= tlas_count) return BF_HIT_INVALID_TOPOLOGY;
        const bf_bvh_node n = nodes[index];
        const float t_max = ANY ? ray.t_max : best.t;
        bool h;
        float nearv;
        uint32_t st = blob_box(n, world, ray.t_min, t_max, h, nearv);
        if (st != BF_HIT_MISS) return st;
        if (!h) continue;
        if (n.kind == 0u) {
            if (n.split_axis > 2u || n.reference_offset != 0u || n.reference_count != 0u) return BF_HIT_INVALID_TOPOLOGY;
            st = blob_push_children(nodes, n, 0u, tlas_count, world, ray.t_min, t_max, tlas_stack, size);
            if (st != BF_HIT_MISS) return st;
            continue;
        }
        if (n.kind != 1u || n.split_axis != BF_INVALID_INDEX || n.first_child != BF_INVALID_INDEX ||
            n.second_child != BF_INVALID_INDEX || n.reference_count != 1u ||
            n.reference_offset >= b.bh->instance_reference_count)
            return BF_HIT_INVALID_TOPOLOGY;
        const bf_bvh_instance_ref ref = refs[n.reference_offset];
        if (ref.reserved[0] != 0u || ref.reserved[1] != 0u || ref.scene_instance_index >= b.sh->instance_count ||
            ref.scene_geometry_index >= b.sh->geometry_count || ref.blas_index >= b.bh->blas_count)
            return BF_HIT_INVALID_TOPOLOGY;
        const uint32_t inst = ref.scene_instance_index;
        if (soa_col<uint32_t>(b, bf_soa::C_INSTANCE_ID)[inst] != ref.instance_id ||
            soa_col<uint32_t>(b, bf_soa::C_INSTANCE_GEOMETRY_ID)[inst] != ref.geometry_id ||
            soa_col<uint32_t>(b, bf_soa::C_INSTANCE_VISIBILITY_MASK)[inst] != ref.visibility_mask)
            return BF_HIT_INVALID_TOPOLOGY;
        if ((ray.visibility_mask & ref.visibility_mask) == 0u) continue;
        float m[12];
        st = blob_matrix(b, bf_soa::C_INSTANCE_WORLD_TO_LOCAL, inst, m);
        if (st != BF_HIT_MISS) return st;
        const v3f lo = xform_point(m, o), ld = xform_vector(m, d);
        if (!fin3(lo) || !fin3(ld) || (ld.x == 0.0f && ld.y == 0.0f && ld.z == 0.0f)) return BF_HIT_NUMERICAL_FAILURE;
        st = blob_blas<ANY>(b, ref, ray, lo, ld, blas_stack, best, occluded);
        if (st != BF_HIT_MISS) return st;
        if (ANY && occluded) return BF_HIT_MISS;
    }
    return BF_HIT_MISS;
}

template <bool ANY>
__global__ __launch_bounds__(BF_API_BLOCK) void k_blob_traverse(const uint8_t* scene_bytes, size_t scene_size,
                                                                const uint8_t* bvh_bytes, size_t bvh_size,
                                                                const bf_transport_ray* rays, uint32_t count,
                                                                void* results) {
    __shared__ uint32_t s_layout;
    __shared__ uint32_t s_tlas[BF_STRUCTURE_STACK * BF_API_BLOCK];
    __shared__ uint32_t s_blas[BF_STRUCTURE_STACK * BF_API_BLOCK];
    if (threadIdx.x == 0u) {
        uint32_t st = blob_scene_layout(scene_bytes, scene_size);
        if (st == BF_HIT_MISS) st = blob_bvh_layout(bvh_bytes, bvh_size, *(const bf_scene_soa_header*)scene_bytes);
        s_layout = st;
    }
    __syncthreads();
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count) return;
    uint32_t status = s_layout;
    blob_candidate best;
    best.present = false;
    bool occluded = false;
    if (status == BF_HIT_MISS) {
        const bf_transport_ray r = rays[i];
        if (!valid_traversal_ray(r)) {
            status = BF_HIT_INVALID_RAY;
        } else {
            const blob_view b{scene_bytes, (const bf_scene_soa_header*)scene_bytes, bvh_bytes,
                              (const bf_bvh_header*)bvh_bytes};
            best.t = r.t_max;
            status = blob_trace<ANY>(b, r, s_tlas + threadIdx.x, s_blas + threadIdx.x, best, occluded);
        }
    }
    if (ANY) {
        bf_occlusion_result out;
        memset(&out, 0, sizeof out);
        out.status = status != BF_HIT_MISS ? status : (occluded ? BF_OCCLUDED : BF_VISIBLE);
        ((bf_occlusion_result*)results)[i] = out;
    } else {
        bf_closest_hit_result out;
        memset(&out, 0, sizeof out);
        if (status != BF_HIT_MISS) out.status = status;
        else if (best.present) {
            out.status = BF_HIT_HIT;
            out.hit = best.hit;
        }
        ((bf_closest_hit_result*)results)[i] = out;
    }
}

/* Workgroups of one persistent traversal launch of a kind (0 closest hit, 1 shadow, 2 counting): as
 * many as the device holds at once, and no more than one wave per `wave_rays` items. */
static uint32_t trace_blocks(const bf_transport_params* P, uint32_t max_count, uint32_t block, uint32_t wave_rays,
                             uint32_t kind) {
    const uint32_t needed = blocks_for(blocks_for(max_count, wave_rays), block / 64u);
    const uint32_t resident = P->trace_lanes[kind] / block;
    return needed < resident ? needed : resident;
}

template <bool ANY, bool BATCH, uint32_t BLOCK>
static void launch_trace(const bf_transport_params* P, uint32_t max_count, const uint32_t* q, const uint32_t* n,
                         uint8_t* route, unsigned long long* counters, bool exact, hipStream_t s) {
    (void)bfk_set_words(P->fetch + (ANY ? BF_CLAIM_SEGMENTS * BF_CLAIM_STRIDE : 0u), BF_CLAIM_SEGMENTS * BF_CLAIM_STRIDE, 0u, s);
    /* optional direction-octant order; the route bytes are free until the traversal writes them */
    uint32_t* order = ANY ? P->shadow_order : P->closest_order;
    if (order)
        bfk_work_order(P, ANY ? BF_KEY_SHADOW : BF_KEY_RAY, q, n, max_count, route, order, BATCH, s);
    if (exact)
        hipLaunchKernelGGL((k_trace_counting<ANY, BATCH, BLOCK>), dim3(trace_blocks(P, max_count, BLOCK, 64u, 2u)),
                           dim3(BLOCK), 0, s, *P, q, n, order, route, counters);
    else
        hipLaunchKernelGGL((k_trace<ANY, BATCH, BLOCK>), dim3(trace_blocks(P, max_count, BLOCK, 4u, ANY ? 1u : 0u)),
                           dim3(BLOCK), 0, s, *P, q, n, order, route);
}

template <bool ANY, bool BATCH>
static void launch_trace_block(const bf_transport_params* P, uint32_t max_count, const uint32_t* q, const uint32_t* n,
                               uint8_t* route, unsigned long long* counters, bool exact, hipStream_t s) {
    if (P->trace_block == 64u) launch_trace<ANY, BATCH, 64u>(P, max_count, q, n, route, counters, exact, s);
    else if (P->trace_block == 256u) launch_trace<ANY, BATCH, 256u>(P, max_count, q, n, route, counters, exact, s);
    else launch_trace<ANY, BATCH, 128u>(P, max_count, q, n, route, counters, exact, s);
}

/* Counted launches, and frames outside the bound engine's range (P->exact_walk), take the step-exact
 * walk; its counts go to the workspace's own counters when the caller asked for none. */
template <bool ANY>
static hipError_t trace_stage(const bf_transport_params* P, const uint32_t* queue, const uint32_t* count_ptr,
                              uint32_t max_count, uint8_t* route, unsigned long long* counters, bool batch, hipStream_t s) {
    if (max_count == 0) return hipSuccess;
    const bool exact = counters != nullptr || P->exact_walk != 0u;
    if (!counters) counters = P->step_counters;
    if (batch) launch_trace_block<ANY, true>(P, max_count, queue, count_ptr, route, counters, exact, s);
    else launch_trace_block<ANY, false>(P, max_count, queue, count_ptr, route, counters, exact, s);
    return hipGetLastError();
}

extern "C" {

hipError_t bfk_trace_closest(const bf_transport_params* P, const uint32_t* queue, const uint32_t* count_ptr,
                             uint32_t max_count, uint8_t* route, unsigned long long* counters, bool batch, hipStream_t s) {
    return trace_stage<false>(P, queue, count_ptr, max_count, route, counters, batch, s);
}

hipError_t bfk_trace_shadow(const bf_transport_params* P, const uint32_t* queue, const uint32_t* count_ptr,
                            uint32_t max_count, uint8_t* route, unsigned long long* counters, bool batch, hipStream_t s) {
    return trace_stage<true>(P, queue, count_ptr, max_count, route, counters, batch, s);
}

} /* extern "C" */

/* Lanes the device holds at once for each kind of traversal launch (0 closest hit, 1 shadow, 2
 * counting), the least over its workgroup sizes so that a grid of that many is resident in each;
 * false on error. */
template <uint32_t BLOCK>
static void trace_lanes_of(int device, uint32_t* lanes) {
    const void* kernels[8] = {(const void*)k_trace<false, false, BLOCK>,         (const void*)k_trace<false, true, BLOCK>,
                              (const void*)k_trace<true, false, BLOCK>,          (const void*)k_trace<true, true, BLOCK>,
                              (const void*)k_trace_counting<false, false, BLOCK>, (const void*)k_trace_counting<false, true, BLOCK>,
                              (const void*)k_trace_counting<true, false, BLOCK>, (const void*)k_trace_counting<true, true, BLOCK>};
    for (int k = 0; k < 8; ++k) {
        uint32_t& kind = lanes[std::min(k / 2, 2)];
        kind = std::min(kind, (uint32_t)bfk_max_resident(kernels + k, 1, BLOCK, device) * BLOCK);
    }
}

extern "C" {

bool bfk_trace_resident_lanes(int device, uint32_t* lanes) {
    for (int k = 0; k < 3; ++k) lanes[k] = 0xFFFFFFFFu;
    trace_lanes_of<64u>(device, lanes);
    trace_lanes_of<128u>(device, lanes);
    trace_lanes_of<256u>(device, lanes);
    return lanes[0] != 0u && lanes[1] != 0u && lanes[2] != 0u;
}

} /* extern "C" */

extern "C" {

/* How a stand-alone query of `count` > 0 rays is cut: `chunk` consecutive rays a wave, one wave a
 * workgroup; returns the workgroups. An equal share of 6 waves on each of the 1024 SIMDs of an undivided
 * MI355X, at most 256 rays so that the last waves of a large launch even out. The SIMD count is a tuning
 * constant (results do not depend on the cut), not the device's own. */
uint32_t bfk_ray_grid(uint32_t count, uint32_t* chunk) {
    const uint32_t waves = 6u * 4u * 256u;
    *chunk = std::min(blocks_for(count, waves), 256u);
    return blocks_for(count, *chunk);
}

} /* extern "C" */

template <bool ANY>
static hipError_t scene_trace(const bf_dev_scene* S, const bf_transport_ray* rays, uint32_t count, void* results,
                              uint32_t* counters, hipStream_t s) {
    if (count == 0) return hipSuccess;
    if (counters || S->exact_walk) {
        hipLaunchKernelGGL(k_scene_counting<ANY>, dim3(blocks_for(count, BF_API_BLOCK)), dim3(BF_API_BLOCK), 0, s, *S, rays,
                           count, results, counters);
    } else {
        uint32_t chunk = 0;
        const uint32_t grid = bfk_ray_grid(count, &chunk);
        hipLaunchKernelGGL(k_scene_trace<ANY>, dim3(grid), dim3(BF_API_BLOCK), 0, s, *S, rays, count, chunk, results);
    }
    return hipGetLastError();
}

extern "C" {

hipError_t bfk_scene_closest_hit(const bf_dev_scene* S, const bf_transport_ray* rays, uint32_t count,
                                 bf_closest_hit_result* results, uint32_t* counters, hipStream_t s) {
    return scene_trace<false>(S, rays, count, results, counters, s);
}

hipError_t bfk_blob_traverse(bool any, const uint8_t* scene_bytes, size_t scene_size, const uint8_t* bvh_bytes,
                             size_t bvh_size, const bf_transport_ray* rays, uint32_t count, void* results, hipStream_t s) {
    if (count == 0) return hipSuccess;
    const dim3 grid(blocks_for(count, BF_API_BLOCK)), block(BF_API_BLOCK);
    if (any)
        hipLaunchKernelGGL(k_blob_traverse<true>, grid, block, 0, s, scene_bytes, scene_size, bvh_bytes, bvh_size, rays,
                           count, results);
    else
        hipLaunchKernelGGL(k_blob_traverse<false>, grid, block, 0, s, scene_bytes, scene_size, bvh_bytes, bvh_size, rays,
                           count, results);
    return hipGetLastError();
}

hipError_t bfk_scene_occlusion(const bf_dev_scene* S, const bf_transport_ray* rays, uint32_t count,
                               bf_occlusion_result* results, hipStream_t s) {
    return scene_trace<true>(S, rays, count, results, nullptr, s);
}

} /* extern "C" */
