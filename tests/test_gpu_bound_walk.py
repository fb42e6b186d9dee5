"""The traversal that renders take (binary32 bounds, binary64 only where it can decide the result)
against the oracle's step-by-step binary64 walk, bit for bit, where bounds and exact values part:

  - a lattice of unit boxes and flat quads seen by rays that start on lattice points and run along
    axes, face diagonals and through edges and vertices: zero direction components, origins on box
    planes, degenerate boxes, sibling boxes with equal near planes, shared edges hit twice;
  - the same at scales whose reciprocals, products or coordinates leave binary32's comfortable
    range (subnormal direction components, 2^-60, 2^60, past 2^126 where launches take the
    step-exact walk);
  - item counts around a wave, its refill threshold and the share of a wave in a small launch.
"""
import numpy as np
import pytest

from path_inputs import as_u32
from rays import result_bytes
from test_gpu_paths import compare

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
    """Walks that hold more entries than the LDS part of the stack: many overlapping boxes per ray."""
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
