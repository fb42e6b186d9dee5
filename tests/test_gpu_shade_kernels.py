"""The shade stage's kernels and its rule for them, against the oracle bit for bit: scenes whose
materials send their items to one kernel without an order (one kind of single closure), to the kernel
of single closures through the order, to the general kernel, or to both; item counts that leave the
kinds' ranges of the order with remainders of every size; and uniform selection over light counts on
both sides of the powers of two that the sampler answers from a dimension's leading bits."""
import numpy as np
import pytest

from test_gpu_transport import check_parity

pytestmark = pytest.mark.gpu


def closures(bf, kind):
    s = bf.scenes
    return {
        "lambert": [s.lambert(0.6)],
        "conductor": [s.rough_conductor(1.0, s.GOLD_ETA, s.GOLD_K, 0.2, 0.35)],
        "dielectric": [s.rough_dielectric(1.0, 1.0, 1.5, 0.15)],
        "mirror": [s.specular_reflection(0.8)],
        "diffuse": [s.rough_diffuse(0.5, 0.4)],
        "mixture": [s.lambert(0.5, probability=0.6), s.rough_conductor(0.8, s.COPPER_ETA, s.COPPER_K, 0.3, probability=0.4)],
    }[kind]


def boxes(bf, kinds, lights, width, height):
    """A row of boxes over a floor, their materials in turn; `lights` small quads overhead."""
    s = bf.scenes.Scene()
    materials = [s.add_material(1 + k, closures(bf, kind)) for k, kind in enumerate(kinds)]
    box = s.add_geometry(11, *bf.scenes.unit_box())
    floor = s.add_geometry(12, *bf.scenes.quad([[-8, 0, -8], [-8, 0, 8], [8, 0, 8], [8, 0, -8]], [0, 1, 0]))
    s.add_instance(100, 100, floor, materials[0])
    for k in range(7):
        s.add_instance(101 + k, 101 + k, box, materials[k % len(materials)],
                       bf.scenes.affine(bf.scenes.rotation_y(0.3 * k), (1.3 * (k - 3), 0.55, 0.4 * (k % 3))))
    if lights:
        emitter = s.add_material(90, closures(bf, kinds[0]), emission=9.0)
        # one triangle each, so the selection runs over exactly `lights` of them
        lamp = s.add_geometry(13, [[-0.2, 0, -0.2], [0.2, 0, -0.2], [0, 0, 0.3]], [[0, -1, 0]] * 3,
                              [[0, 0], [1, 0], [0, 1]], [[0, 1, 2]])
        side = int(np.ceil(np.sqrt(lights)))
        for k in range(lights):
            s.add_instance(1000 + k, 1000 + k, lamp, emitter,
                           bf.scenes.affine(translation=(0.5 * (k % side - side / 2), 5.0, 0.5 * (k // side - side / 2))))
    s.set_environment(0.3)
    s.finalize()
    return s, bf.scenes.look_at_camera((0.5, 3.0, 7.5), (0.0, 0.4, 0.0), width, height, 0.8)


def check(bf, oracle, hip, scene_and_camera, width, height, spp, launch=0, **opts):
    scene, camera = scene_and_camera
    frame = bf.scenes.frame_desc(camera, spp)
    options = bf.scenes.transport_options(**opts)
    options.record_queues = 1
    options.launch = launch
    expected = oracle.scene(scene).render(frame, options, threads=8)
    ws = hip.XpuWavefrontTransportWorkspace(width * height * spp)
    got = hip.trace_xpu_wavefront_transport(ws, hip.XpuScene(scene), frame, options, want_paths=True, want_counters=True)
    check_parity(expected, got)


@pytest.mark.parametrize("kinds", [
    ("lambert",), ("conductor",), ("dielectric",),                       # one kind: no order
    ("lambert", "conductor"), ("dielectric", "lambert"), ("conductor", "dielectric"),
    ("lambert", "conductor", "dielectric"),
    ("mirror",), ("diffuse", "mirror"), ("mixture",),                    # the general kernel alone
    ("mixture", "lambert"), ("mirror", "dielectric"),
    ("lambert", "conductor", "dielectric", "diffuse", "mirror", "mixture"),
], ids="-".join)
@pytest.mark.parametrize("launch", ["default", "grouped"])
def test_material_kinds(bf, oracle, hip, kinds, launch):
    check(bf, oracle, hip, boxes(bf, kinds, 1, 33, 17), 33, 17, 3,
          launch=bf.abi.LAUNCH_SHADE_ORDER if launch == "grouped" else 0, mis=1, max_depth=6)


@pytest.mark.parametrize("width,height", [(1, 1), (3, 1), (9, 7), (16, 16), (257, 1), (37, 29)])
def test_remainders_of_the_kinds(bf, oracle, hip, width, height):
    kinds = ("lambert", "conductor", "dielectric", "mixture")
    check(bf, oracle, hip, boxes(bf, kinds, 2, width, height), width, height, 1, max_depth=5)


@pytest.mark.parametrize("lights", [0, 1, 2, 3, 64, 255, 256, 257, 512])
@pytest.mark.parametrize("sampler", [0, 1])
def test_light_counts(bf, oracle, hip, lights, sampler):
    check(bf, oracle, hip, boxes(bf, ("lambert",), lights, 16, 9), 16, 9, 2, sampler=sampler, max_depth=3)


def test_sample_indexes_past_a_byte(bf, oracle, hip):
    check(bf, oracle, hip, boxes(bf, ("lambert", "dielectric"), 4, 2, 2), 2, 2, 515, max_depth=4)


def test_partitions_of_several_tiles_a_workgroup(bf, hip):
    """9.4 M paths in one launch, past one tile of 512 items a workgroup in the compactions (from 1 M) and
    in the shade order (from 256 K), against a launch per sample."""
    width, height, spp = 1025, 1021, 9
    scene, camera = boxes(bf, ("lambert", "conductor", "dielectric", "mixture"), 1, width, height)
    frame = bf.scenes.frame_desc(camera, spp)
    options = bf.scenes.transport_options(max_depth=3)
    device_scene = hip.XpuScene(scene)
    films = []
    for capacity in (width * height * spp, width * height):
        ws = hip.XpuWavefrontTransportWorkspace(capacity)
        films.append(hip.trace_xpu_wavefront_transport(ws, device_scene, frame, options)["film"].host())
        ws.close()
    for name in ("film", "film_counts"):
        assert np.array_equal(films[0][name].view(np.uint32), films[1][name].view(np.uint32)), name
