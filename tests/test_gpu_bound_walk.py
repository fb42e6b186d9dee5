"""The traversal that renders take (binary32 bounds, binary64 only where it can decide the result)
against the oracle's step-by-step binary64 walk, bit for bit, where bounds and exact values part:

  - a lattice of unit boxes and flat quads seen by rays that start on lattice points and run along
    axes, face diagonals and through edges and vertices: zero direction components, origins on box
    planes, degenerate boxes, sibling boxes with equal near planes, shared edges hit twice;
  - the same at scales whose reciprocals, products or coordinates leave binary32's comfortable
    range (subnormal direction components, 2^-60, 2^60, past 2^126 where launches take the
    step-exact walk);
  - item counts around a wave, its refill threshold and the share of a wave in a small launch;
  - stacks deeper than their part in LDS, for closest-hit and any-hit walks of every launch;
  - frames in every workgroup size, with and without orders and counters.
"""
import functools

import numpy as np
import pytest

from path_inputs import as_u32
from rays import result_bytes
from test_gpu_paths import compare
from test_gpu_transport import check_parity, path_arrays

pytestmark = pytest.mark.gpu


def lattice(bf, scale=1.0):
    s = bf.scenes.Scene()
    material = s.add_material(1, [bf.scenes.lambert(0.5)])
    light = s.add_material(2, [bf.scenes.lambert(0.0)], emission=3.0)
    positions, normals, uvs, faces = (np.asarray(a) for a in bf.scenes.unit_box())
    box = s.add_geometry(11, positions * scale, normals, uvs, faces)
    quad = s.add_geometry(12, *bf.scenes.quad([[-8 * scale, 0, -8 * scale], [-8 * scale, 0, 8 * scale],
                                               [8 * scale, 0, 8 * scale], [8 * scale, 0, -8 * scale]], [0, 1, 0]))
    k = 0
    for x in range(-2, 3):
        for y in range(0, 2):
            for z in range(-2, 3):
                s.add_instance(100 + k, 100 + k, box, material,
                               bf.scenes.affine(translation=(x * scale, (y + 0.5) * scale, z * scale)))
                k += 1
    s.add_instance(500, 500, quad, material, bf.scenes.affine())
    if scale <= 1.0:  # a larger emitter's area overflows
        s.add_instance(501, 501, quad, light, bf.scenes.affine(np.diag([1.0, -1.0, -1.0]), (0.0, 6.0 * scale, 0.0)))
    s.set_environment(0.25)
    return s.finalize()


def lattice_rays(abi, n, seed, scale=1.0, tiny=0.0, t_max=np.inf):
    """Rays from half-lattice points toward half-lattice offsets; `tiny` replaces zero components."""
    rng = np.random.default_rng(seed)
    o = rng.integers(-7, 8, size=(n, 3)) * 0.5
    o[:, 1] = rng.integers(-1, 9, size=n) * 0.5
    off = rng.uniform(size=n) < 0.3
    o[off] += rng.uniform(-0.5, 0.5, size=(int(off.sum()), 3))
    d = rng.integers(-2, 3, size=(n, 3)).astype(np.float64)
    d[(d == 0).all(axis=1)] = (0.0, -1.0, 0.0)
    d[d == 0] = tiny
    loose = rng.uniform(size=n) < 0.2
    d[loose] += rng.uniform(-0.4, 0.4, size=(int(loose.sum()), 3))
    rays = (abi.TransportRay * n)()
    view = np.frombuffer(rays, dtype=np.float32).reshape(n, 12)
    view[:, 0:3] = o * scale
    view[:, 4:7] = d
    view[:, 7] = t_max
    view[:, 8] = 0.5
    np.frombuffer(rays, dtype=np.uint32).reshape(n, 12)[:, 9] = 0xFFFFFFFF
    return rays


def path_inputs(abi, rays):
    n = len(rays)
    samples = (abi.SampleStreamIndex * n)(*[abi.SampleStreamIndex(k % 64, k // 64, 0, 5) for k in range(n)])
    cones = (abi.RayCone * n)()
    states = (abi.PathStateLane * n)()
    view = np.frombuffer(states, dtype=np.float32).reshape(n, 32)
    view[:, 0:4] = 1.0
    view[:, 8:12] = [400.0, 500.0, 600.0, 700.0]
    view[:, 12:16] = np.float32(1.0) / np.float32(470.0)
    view[:, 22] = 1.0
    np.frombuffer(states, dtype=np.uint8).reshape(n, 128)[:, 100:104] = abi.WAVELENGTH_MEASURE
    return samples, rays, cones, states


@pytest.mark.parametrize("scale,tiny", [(1.0, 0.0), (1.0, -0.0), (1.0, 1e-42), (2.0 ** -60, 0.0), (2.0 ** 60, 0.0),
                                        (2.0 ** 122, 0.0), (2.0 ** 124, 0.0)])
def test_lattice_paths_match_the_oracle(bf, abi, oracle, hip, scale, tiny):
    rays = lattice_rays(abi, 6000, 3, scale, tiny)
    options = bf.scenes.transport_options(max_depth=3, rr_first_depth=2)
    options.failure_policy = abi.FAILURES_COUNT
    got, report = compare(hip, oracle, lattice(bf, scale), path_inputs(abi, rays), options)
    if scale == 1.0:
        assert report.shadow_queries > 500
        assert len(np.unique(as_u32(got["rays"])[:, 0])) > 100


@pytest.mark.parametrize("count", [1, 2, 63, 64, 65, 255, 257, 4095, 30001])
def test_any_item_count_matches_the_oracle(bf, abi, oracle, hip, count):
    rays = lattice_rays(abi, count, count)
    options = bf.scenes.transport_options(max_depth=2, rr_first_depth=0)
    options.failure_policy = abi.FAILURES_COUNT
    compare(hip, oracle, lattice(bf), path_inputs(abi, rays), options)


@pytest.mark.parametrize("count,tiny", [(1, 0.0), (65, 0.0), (6145, 0.0), (30001, 0.0), (3000, 1e-42)])
def test_ray_queries_match_the_oracle(bf, abi, oracle, hip, count, tiny):
    """Uncounted stand-alone queries; 6145 rays are one more than the waves the share is cut for."""
    scene = lattice(bf)
    xs, want = hip.XpuScene(scene), oracle.scene(scene)
    rays = lattice_rays(abi, count, 7 + count, tiny=tiny)
    rays[count // 2].t_min = -1.0  # an invalid ray answers alone
    assert result_bytes(xs.closest_hit(rays)) == result_bytes(want.closest_hit(rays))
    rays = lattice_rays(abi, count, 8 + count, tiny=tiny, t_max=2.5)
    assert result_bytes(xs.occlusion(rays)) == result_bytes(want.occlusion(rays))


def test_deep_stacks_match_the_oracle(bf, abi, oracle, hip):
    """Closest-hit walks that hold more entries than the 8 in LDS: many overlapping boxes per ray."""
    scene, _ = bf.scenes.icosphere_grid(grid=6, subdivisions=3)
    rng = np.random.default_rng(1)
    n = 8000
    rays = (abi.TransportRay * n)()
    view = np.frombuffer(rays, dtype=np.float32).reshape(n, 12)
    view[:, 0:3] = rng.uniform([-9, -1, -9], [9, 1, 9], size=(n, 3))
    d = rng.normal(size=(n, 3)) * [1.0, 0.02, 1.0]
    view[:, 4:7] = d / np.linalg.norm(d, axis=1, keepdims=True)
    view[:, 7], view[:, 8] = np.inf, 0.5
    np.frombuffer(rays, dtype=np.uint32).reshape(n, 12)[:, 9] = 0xFFFFFFFF
    xs, want = hip.XpuScene(scene), oracle.scene(scene)
    assert result_bytes(xs.closest_hit(rays)) == result_bytes(want.closest_hit(rays))
    assert result_bytes(xs.occlusion(rays)) == result_bytes(want.occlusion(rays))


def stacked_corner(bf, split):
    """Sibling boxes that share their min corner and differ in extent: triangle A, and B1 in A's plane
    with B2 above it. A ray from above enters B's box first and finds B1; A's box is then culled where
    t rounds below it. split: one triangle per instance (siblings in the TLAS) or one geometry."""
    s = bf.scenes.Scene()
    material = s.add_material(1, [bf.scenes.lambert(0.5)])
    triangles = [[[0, 0, 0], [2, 0, 0], [0, 0, 2]], [[0, 0, 0], [6, 0, 0], [0, 0, 2]], [[4, 3, 0], [6, 4, 0], [6, 4, 2]]]
    for k, group in enumerate([[t] for t in triangles] if split else [triangles]):
        corners = np.concatenate(group)
        g = s.add_geometry(11 + k, corners, [[0, 1, 0]] * len(corners), [[0, 0]] * len(corners),
                           np.arange(len(corners)).reshape(-1, 3))
        s.add_instance(100 + k, 100 + k, g, material, bf.scenes.affine())
    s.set_environment(0.25)
    return s.finalize()


@pytest.mark.parametrize("split", [False, True], ids=["blas", "tlas"])
@pytest.mark.parametrize("direction", [(-0.01, -1.0, 1e-42), (-0.01, -1.0, -1e-42), (-1e-42, -1.0, 0.01),
                                       (-0.01 * 2.0 ** 127, -(2.0 ** 127), -0.02 * 2.0 ** 127)],
                         ids=["up", "down", "x", "huge"])
def test_sibling_order_where_bounds_do_not_hold(bf, abi, oracle, hip, split, direction):
    """Directions without binary32 reciprocals (a subnormal component, or past 2^126) and negative others."""
    rng = np.random.default_rng(4)
    n = 4000
    rays = (abi.TransportRay * n)()
    view = np.frombuffer(rays, dtype=np.float32).reshape(n, 12)
    view[:, 0:3] = rng.uniform([0.0, 4.5, 0.0], [2.0, 9.0, 2.0], size=(n, 3))
    view[:, 4:7] = np.array(direction) * rng.uniform(0.7, 1.3, size=(n, 1))
    view[:, 7], view[:, 8] = np.inf, 0.5
    np.frombuffer(rays, dtype=np.uint32).reshape(n, 12)[:, 9] = 0xFFFFFFFF
    scene = stacked_corner(bf, split)
    xs, want = hip.XpuScene(scene), oracle.scene(scene)
    expected = as_u32(want.closest_hit(rays))
    # the order is what decides: both triangles of the plane are answers
    assert len(np.unique(expected[expected[:, 0] == abi.HIT_HIT][:, 13:16], axis=0)) > 1
    differ = np.nonzero((as_u32(xs.closest_hit(rays)) != expected).any(axis=1))[0]
    assert differ.size == 0, f"{differ.size} of {n} hits differ, first {differ[:5].tolist()}"
    options = bf.scenes.transport_options(max_depth=2, rr_first_depth=0)
    options.failure_policy = abi.FAILURES_COUNT
    compare(hip, oracle, scene, path_inputs(abi, rays), options)


SHADOW_STACK = 16  # entries of an any-hit walk in LDS


def sheaf(bf, width, height):
    """256 instances of 512 triangles whose boxes nearly coincide: a ray up through x + z > 1 meets every
    box and misses all but a few triangles. Every third instance is masked. A floor below, a lamp above."""
    rng = np.random.default_rng(11)
    s = bf.scenes.Scene()
    material = s.add_material(1, [bf.scenes.lambert(0.7)])
    lamp = s.add_material(2, [bf.scenes.lambert(0.0)], emission=8.0)
    corners = np.array([[0, 0, 0], [1, 0.5, 0], [0, 1, 1]], dtype=np.float64)
    corners = (corners + rng.uniform(-0.02, 0.02, size=(512, 3, 3))).reshape(-1, 3)
    cloud = s.add_geometry(11, corners, [[0, 1, 0]] * 1536, [[0, 0], [1, 0], [0, 1]] * 512, np.arange(1536).reshape(-1, 3))
    shifts = rng.uniform(-0.02, 0.02, size=(256, 3)).astype(np.float32)
    for k, shift in enumerate(shifts):
        s.add_instance(100 + k, 100 + k, cloud, material, bf.scenes.affine(translation=shift),
                       mask=0xFFFFFFFE if k % 3 == 0 else 0xFFFFFFFF)
    floor = s.add_geometry(12, *bf.scenes.quad([[-4, -1, -4], [-4, -1, 4], [4, -1, 4], [4, -1, -4]], [0, 1, 0]))
    top = s.add_geometry(13, *bf.scenes.quad([[0.7, 3, 0.7], [1, 3, 0.7], [1, 3, 1], [0.7, 3, 1]], [0, -1, 0]))
    s.add_instance(500, 500, floor, material, bf.scenes.affine())
    s.add_instance(501, 501, top, lamp, bf.scenes.affine())
    s.set_environment(0.25)
    camera = bf.scenes.look_at_camera((2.6, -0.4, 2.6), (0.85, -1.0, 0.85), width, height, 0.25)
    camera.visibility_mask = 1
    return s.finalize(), camera


def peak_entries(abi, xs, scene, o, d, enough):
    """Most entries an uncut near-first walk of the canonical BVH holds for a ray, the two that mark the
    ends of the ray and of a BLAS among them, or the first number past `enough`."""
    bvh = xs.bvh()
    trees = [np.frombuffer(bvh[k], dtype=np.uint32).reshape(-1, 12) for k in ("blas_nodes", "tlas_nodes")]
    blases = np.frombuffer(bvh["blas"], dtype=np.uint32).reshape(-1, 8)
    refs = (abi.BvhInstanceRef * bvh["counts"][4]).from_buffer_copy(bvh["instance_refs"])
    roots = [abi.BvhBlas.from_buffer_copy(b.tobytes()).root_node for b in blases]

    def near(tree, node, origin):
        box = trees[tree].view(np.float32)[node][[0, 1, 2, 4, 5, 6]].astype(np.float64)
        t = np.stack([(box[:3] - origin) / d, (box[3:] - origin) / d])
        lo, hi = max(t.min(axis=0).max(), 0.0), t.max(axis=0).min()
        return lo if lo <= hi else None

    def walk(tree, root, origin, held):
        peak, stack = held, [root] if near(tree, root, origin) is not None else []
        while stack and peak <= enough:
            node = stack.pop()
            row = trees[tree][node]
            if row[3] == 0:
                met = sorted(((n, c) for c in (row[8], row[9]) if (n := near(tree, c, origin)) is not None), reverse=True)
                stack += [c for _, c in met]
                peak = max(peak, held + len(stack) - (1 if met else 0))  # the nearer child is walked at once
            elif tree == 1:
                ref = refs[row[10]]
                m = np.array(list(scene.instances[ref.scene_instance_index].local_to_world)).reshape(3, 4)
                peak = max(peak, walk(0, roots[ref.blas_index], origin - m[:, 3], held + len(stack) + 1))
        return peak

    return walk(1, bvh["tlas_root"], np.asarray(o, dtype=np.float64), 1)


def test_any_hit_stacks_past_lds_match_the_oracle(bf, abi, oracle, hip):
    """Rays up through the sheaf: occlusion queries, closest hits, and the shadow rays of path inputs."""
    scene, _ = sheaf(bf, 4, 4)
    xs, want = hip.XpuScene(scene), oracle.scene(scene)
    assert peak_entries(abi, xs, scene, (0.9, -1.0, 0.9), np.array([0.001, 1.0, 0.001]), SHADOW_STACK) > SHADOW_STACK
    rng = np.random.default_rng(12)
    n = 160
    rays = (abi.TransportRay * n)()
    view = np.frombuffer(rays, dtype=np.float32).reshape(n, 12)
    view[:, 0:3] = rng.uniform([0.45, -0.9, 0.5], [0.95, -0.5, 0.95], size=(n, 3))
    view[:, 4:7] = rng.uniform([-0.01, 1.0, -0.01], [0.01, 1.0, 0.01], size=(n, 3))
    view[:, 7], view[:, 8] = 2.5, 0.5
    np.frombuffer(rays, dtype=np.uint32).reshape(n, 12)[:, 9] = 1
    for query in ("occlusion", "closest_hit"):
        expected = as_u32(getattr(want, query)(rays))
        assert len(np.unique(expected[:, 0])) == 2, query  # some rays reach the lamp's height, some do not
        assert np.array_equal(as_u32(getattr(xs, query)(rays)), expected), query
    view[:, 1], view[:, 5], view[:, 7] = -0.5, -1.0, np.inf  # down to the floor, below the sheaf
    options = bf.scenes.transport_options(max_depth=2, rr_first_depth=0)
    options.failure_policy = abi.FAILURES_COUNT
    _, report = compare(hip, oracle, scene, path_inputs(abi, rays), options)
    assert report.shadow_queries >= n


@functools.lru_cache(maxsize=None)
def expected_frame(bf, oracle, name):
    width, height, spp = (12, 8, 2) if name == "sheaf" else (48, 27, 2)
    scene, camera = sheaf(bf, width, height) if name == "sheaf" else bf.scenes.icosphere_grid(width, height, grid=4,
                                                                                               subdivisions=2)
    frame = bf.scenes.frame_desc(camera, spp, seed=11)
    options = bf.scenes.transport_options(max_depth=2 if name == "sheaf" else 16, mis=bf.abi.MIS_POWER)
    options.record_queues = 1
    return scene, frame, options, oracle.scene(scene).render(frame, options, threads=8)


@pytest.mark.parametrize("name,order", [("grid", 0), ("grid", 0x00100000), ("grid", 0x00200000), ("grid", 0x00300000),
                                        ("sheaf", 0)], ids=["grid", "grid-shade", "grid-trace", "grid-both", "sheaf"])
@pytest.mark.parametrize("lanes", [64, 128, 256])
@pytest.mark.parametrize("counters", [False, True], ids=["bound", "counting"])
def test_frames_match_the_oracle_in_every_launch_shape(bf, oracle, hip, name, order, lanes, counters):
    """A frame and a batch of two: uncounted launches take the bound walk, counted ones the step-exact one."""
    scene, frame, options, expected = expected_frame(bf, oracle, name)
    options.launch = bf.abi.launch_trace_block(lanes) | order
    xs = hip.XpuScene(scene)
    n = frame.camera.width * frame.camera.height * frame.samples_per_pixel
    ws = hip.XpuWavefrontTransportWorkspace(2 * n)
    got = hip.trace_xpu_wavefront_transport(ws, xs, frame, options, want_paths=True, want_counters=counters)
    if counters:
        check_parity(expected, got)
    else:
        for b in range(expected["report"].bounces):
            assert got["report"].ray_queue_hash[b] == expected["report"].ray_queue_hash[b], b
            assert got["report"].shadow_queue_hash[b] == expected["report"].shadow_queue_hash[b], b
        assert np.array_equal(path_arrays(got["paths"]), path_arrays(expected["paths"]))
        assert np.array_equal(got["film"].host()["film"], expected["film"])
    batch = hip.trace_xpu_wavefront_batch(ws, [(xs, frame), (xs, frame)], options, want_paths=True, want_counters=counters)
    for k in range(2):
        assert np.array_equal(path_arrays(batch["paths"][k]), path_arrays(expected["paths"])), k
        assert np.array_equal(batch["films"][k].host()["film"], expected["film"]), k
