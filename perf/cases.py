"""What is timed of this renderer: frames, batches, path inputs, ray queries, the texture adjoint
and the texture fit, each through the entry points a program calls.

A case is a dict of plain values. Its "kind" names the entry point:
  frame      trace_xpu_wavefront_transport: one frame (Cornell box, displaced icosphere grid, or a
             Cornell box with normal and bump maps) into a new film
  batch      trace_xpu_wavefront_batch: uneven frames of several scenes in one call
  paths      trace_xpu_wavefront_paths: caller-made primary rays and path states, terminal records out
  closest    blackframe_hip_launch_scene_closest_hit on device rays
  occlusion  blackframe_hip_launch_scene_occlusion on device rays
  adjoint    DifferentiableFrame: taped render and texel gradients of an image gradient
  fit        TextureFit: taped forward, L2 loss and adjoint of several textured scenes

Films, path records and hits are decided bit for bit by the scene and the sample streams, so they
are compared exactly; texel gradients are sums of float atomics in no fixed order.
"""
import ctypes
import importlib
import importlib.util
import math
import sys
from pathlib import Path

import numpy as np
import torch

ROOT = Path(__file__).resolve().parent.parent
PACKAGE = "blackframe_renderer_amd"


def _package():
    """The package (its folder's name is not an identifier) and its HIP module."""
    if PACKAGE not in sys.modules:
        folder = ROOT / "blackframe-renderer_amd"
        spec = importlib.util.spec_from_file_location(PACKAGE, folder / "__init__.py",
                                                      submodule_search_locations=[str(folder)])
        module = importlib.util.module_from_spec(spec)
        sys.modules[PACKAGE] = module
        spec.loader.exec_module(module)
    return sys.modules[PACKAGE], importlib.import_module(PACKAGE + ".hip")


def listed():
    return [
        # the reference's own Cornell frame: small enough that launches and host reads show
        dict(name="frame_cornell_64x64x16", kind="frame", scene="cornell", width=64, height=64, spp=16, depth=8,
             mis="balance", launch=0),
        # one interactive preview pass of a small scene, odd sizes
        dict(name="frame_preview_333x187x1", kind="frame", scene="grid", grid=8, width=333, height=187, spp=1,
             depth=8, mis="power", launch=0),
        # an ordinary offline frame at the default launch word
        dict(name="frame_grid16_640x360x16", kind="frame", scene="grid", grid=16, width=640, height=360, spp=16,
             depth=16, mis="power", launch=0),
        # the headline frame: 1.3 M triangles, 1080p, 64 samples, tuned launch word
        dict(name="frame_grid32_1080p64", kind="frame", scene="grid", grid=32, width=1920, height=1080, spp=64,
             depth=16, mis="power", launch=0x00160004),
        # normal and bump maps (EWA lookups in the shade stage)
        dict(name="frame_mapped_256x256x16", kind="frame", scene="mapped", width=256, height=256, spp=16, depth=8,
             mis="balance", launch=0),
        # several users' frames of unequal size in one set of queues, bounce groups as graphs
        dict(name="batch_6_scenes", kind="batch", scenes=6, max_resolution=512, max_spp=32, depth=16,
             launch=0x80160004),
        # a host renderer that makes its own primary rays, an odd count
        dict(name="paths_grid16_300007", kind="paths", grid=16, count=300007, depth=8),
        # ray queries of a tool or a physics step: a few rays, and a large incoherent set
        dict(name="closest_cornell_777", kind="closest", scene="cornell", grid=0, count=777),
        dict(name="closest_grid32_1000003", kind="closest", scene="grid", grid=32, count=1000003),
        dict(name="occlusion_grid32_2000003", kind="occlusion", scene="grid", grid=32, count=2000003),
        # the differentiable Cornell box: taped render, then texel gradients
        dict(name="adjoint_cornell_256x256x64", kind="adjoint", width=256, height=256, spp=64, texture=512, depth=8),
        # loss and gradients of a texture fit over several scenes
        dict(name="fit_3_scenes", kind="fit", scenes=3, min_resolution=256, max_resolution=320, texture=1024,
             spp=16, depth=8),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["frame", "frame", "frame", "batch", "paths", "closest", "occlusion", "adjoint", "fit"])
    mis = rng.choice(["balance", "power"])
    if kind == "frame":
        scene = rng.choice(["cornell", "grid", "grid", "mapped"])
        width, height = _log_uniform(rng, 33, 1920), _log_uniform(rng, 33, 1080)
        spp = _log_uniform(rng, 1, 64)
        if scene == "mapped":
            spp = max(1, min(spp, 4000000 // (width * height)))
        case = dict(kind=kind, scene=scene, width=width, height=height, spp=spp,
                    depth=rng.randint(1, 16), mis=mis, launch=rng.choice([0, 0x00160004, 0x00080002, 0x80060004]))
        if scene == "grid":
            case["grid"] = _log_uniform(rng, 1, 32)
        return case
    if kind == "batch":
        return dict(kind=kind, scenes=rng.randint(2, 8), max_resolution=_log_uniform(rng, 64, 512),
                    max_spp=_log_uniform(rng, 2, 32), depth=rng.randint(2, 16),
                    launch=rng.choice([0, 0x80160004, 0x80080002]))
    if kind == "paths":
        return dict(kind=kind, grid=_log_uniform(rng, 1, 24), count=_log_uniform(rng, 100, 1000000),
                    depth=rng.randint(1, 12))
    if kind in ("closest", "occlusion"):
        scene = rng.choice(["cornell", "grid", "grid"])
        return dict(kind=kind, scene=scene, grid=_log_uniform(rng, 1, 32) if scene == "grid" else 0,
                    count=_log_uniform(rng, 1, 4000000))
    if kind == "adjoint":
        return dict(kind=kind, width=_log_uniform(rng, 33, 256), height=_log_uniform(rng, 33, 256),
                    spp=_log_uniform(rng, 2, 64), texture=rng.choice([17, 64, 255, 512]), depth=rng.randint(2, 10))
    low = _log_uniform(rng, 48, 256)
    return dict(kind=kind, scenes=rng.randint(1, 3), min_resolution=low, max_resolution=low + rng.randint(0, 64),
                texture=rng.choice([64, 333, 1024]), spp=_log_uniform(rng, 2, 16), depth=rng.randint(2, 8))


# ---- scenes and inputs --------------------------------------------------------------------------
def _mips(image):
    """2x2 box mip chain of a square image whose side is a power of two."""
    levels = [image.astype(np.float32)]
    while levels[-1].shape[0] > 1:
        p = levels[-1]
        n = p.shape[0] // 2
        levels.append(p.reshape(n, 2, n, 2, p.shape[2]).mean(axis=(1, 3)).astype(np.float32))
    return levels


def _mapped_cornell(bf, width, height, seed):
    scene, camera = bf.scenes.cornell(width, height)
    rng = np.random.default_rng(seed)
    n = 128
    y, x = np.mgrid[0:n, 0:n]
    u, v = (x + 0.5) / n, (y + 0.5) / n
    p = rng.uniform(0.0, 2.0 * np.pi, size=5)
    tilt_x = 0.35 * np.sin(2 * np.pi * 3 * u + p[0]) * np.cos(2 * np.pi * 2 * v + p[1])
    tilt_y = 0.35 * np.cos(2 * np.pi * 4 * v + p[2])
    normal = np.stack([tilt_x, tilt_y, np.sqrt(1 - tilt_x ** 2 - tilt_y ** 2)], axis=-1)
    bump = 0.5 + 0.5 * np.sin(2 * np.pi * 5 * u + p[3]) * np.sin(2 * np.pi * 3 * v + p[4])
    t_normal = scene.add_image_texture(_mips(0.5 * (normal + 1.0)))
    t_bump = scene.add_image_texture(_mips(bump[..., None]))
    scene.set_surface_maps(0, normal={"texture": t_normal})
    scene.set_surface_maps(2, bump={"texture": t_bump, "scale": 0.05})
    return scene.finalize(), camera


def _host_scene(bf, case, seed, width=64, height=64):
    if case["scene"] == "cornell":
        return bf.scenes.cornell(width, height)
    if case["scene"] == "mapped":
        return _mapped_cornell(bf, width, height, seed)
    return bf.scenes.icosphere_grid(width, height, grid=case["grid"], seed=0x5EED_1C05 + seed)


def _options(bf, case, mis="power"):
    options = bf.scenes.transport_options(max_depth=case["depth"],
                                          mis=bf.abi.MIS_BALANCE if mis == "balance" else bf.abi.MIS_POWER)
    options.failure_policy = bf.abi.FAILURES_COUNT
    options.launch = case.get("launch", 0)
    return options


def _rays(case, seed, count):
    """Incoherent rays through the scene: origins in its bounds, directions on the sphere (12 words
    a ray: origin, t_min, direction, t_max, time, mask, medium, reserved)."""
    rng = np.random.default_rng(seed)
    if case["scene"] == "cornell":
        lo, hi = np.array([-0.95, -0.95, 0.05]), np.array([0.95, 0.95, 1.95])
        reach = 1.5
    else:
        extent = 1.3 * case["grid"]
        lo, hi = np.array([-extent, -1.5, -extent]), np.array([extent, 6.0, extent])
        reach = 12.0
    rays = np.zeros((count, 12), dtype=np.float32)
    rays[:, 0:3] = rng.uniform(lo, hi, size=(count, 3))
    d = rng.normal(size=(count, 3))
    rays[:, 4:7] = d / np.linalg.norm(d, axis=1, keepdims=True)
    rays[:, 7] = np.inf if case["kind"] == "closest" else rng.uniform(0.1, reach, size=count)
    rays[:, 8] = 0.5
    rays.view(np.uint32)[:, 9] = 0xFFFFFFFF
    return rays


def _path_inputs(bf, camera, case, seed):
    """Sample streams, pinhole rays, cones and initial states of `count` paths over the camera's pixels."""
    n = case["count"]
    rng = np.random.default_rng(seed)
    px, py = np.arange(n) % camera.width, (np.arange(n) // camera.width) % camera.height
    samples = np.zeros(n, dtype=[("x", "<u4"), ("y", "<u4"), ("s", "<u8"), ("seed", "<u8")])
    samples["x"], samples["y"], samples["seed"] = px, py, seed
    samples["s"] = np.arange(n) // (camera.width * camera.height)
    jitter = rng.uniform(size=(n, 2))
    nx = (2.0 * (px + jitter[:, 0]) / camera.width - 1.0) * camera.half_width
    ny = (1.0 - 2.0 * (py + jitter[:, 1]) / camera.height) * camera.half_height
    basis = np.array([list(camera.tangent), list(camera.bitangent), list(camera.normal)])
    d = np.stack([nx, ny, -np.ones(n)], axis=1) @ basis
    rays = np.zeros((n, 12), dtype=np.float32)
    rays[:, 0:3] = list(camera.origin)
    rays[:, 4:7] = d / np.linalg.norm(d, axis=1, keepdims=True)
    rays[:, 7] = np.inf
    rays[:, 8] = 0.5
    rays.view(np.uint32)[:, 9] = 0xFFFFFFFF
    cones = np.zeros((n, 2), dtype=np.float32)
    cones[:, 1] = 1.0e-3
    states = np.zeros((n, 32), dtype=np.float32)
    states[:, 0:4] = 1.0
    states[:, 8:12] = 360.0 + 470.0 * ((rng.uniform(size=(n, 1)) + np.arange(4) / 4.0) % 1.0)
    states[:, 8:12] = np.clip(states[:, 8:12], 360.0, 830.0)
    states[:, 12:16] = np.float32(1.0) / np.float32(470.0)
    states[:, 22] = 1.0
    states.view(np.uint8)[:, 100:104] = bf.abi.WAVELENGTH_MEASURE
    return tuple(torch.from_numpy(a.view(np.uint8).reshape(-1)).cuda() for a in (samples, rays, cones, states))


def _batch_frames(bf, case, seed):
    rng = np.random.default_rng(seed)
    frames = []
    for k in range(case["scenes"]):
        # sizes from the case alone (every seed has the same work), scenes and streams from the seed
        size = max(16, case["max_resolution"] >> (k % 3))
        spp = max(1, case["max_spp"] >> ((2 * k) % 4))
        grid = (20, 3, 12, 6, 16, 9, 4, 14)[k % 8]
        scene, camera = bf.scenes.icosphere_grid(size, max(16, size * 3 // 4 + k), grid=grid,
                                                 seed=int(rng.integers(1 << 32)))
        frames.append((scene, bf.scenes.frame_desc(camera, spp, seed=seed + k)))
    return frames


def prepare(case, seed):
    bf, hip = _package()
    kind = case["kind"]
    state = {"kind": kind, "hip": hip}
    if kind == "frame":
        scene, camera = _host_scene(bf, case, seed, case["width"], case["height"])
        state["scene"] = hip.XpuScene(scene)
        state["frame"] = bf.scenes.frame_desc(camera, case["spp"], seed=seed)
        state["options"] = _options(bf, case, case["mis"])
        state["workspace"] = hip.XpuWavefrontTransportWorkspace(case["width"] * case["height"] * case["spp"])
    elif kind == "batch":
        frames = _batch_frames(bf, case, seed)
        state["items"] = [(hip.XpuScene(scene), frame) for scene, frame in frames]
        state["options"] = _options(bf, case)
        paths = sum(f.camera.width * f.camera.height * f.samples_per_pixel for _, f in frames)
        state["workspace"] = hip.XpuWavefrontTransportWorkspace(paths)
    elif kind == "paths":
        scene, camera = bf.scenes.icosphere_grid(640, 360, grid=case["grid"], seed=0x5EED_1C05 + seed)
        state["scene"] = hip.XpuScene(scene)
        state["inputs"] = _path_inputs(bf, camera, case, seed)
        state["options"] = _options(bf, case)
        state["workspace"] = hip.XpuWavefrontTransportWorkspace(case["count"])
    elif kind in ("closest", "occlusion"):
        scene, _ = _host_scene(bf, case, seed)
        state["scene"] = hip.XpuScene(scene)
        state["rays"] = torch.from_numpy(_rays(case, seed, case["count"])).cuda()
        words = ctypes.sizeof(bf.abi.ClosestHitResult if kind == "closest" else bf.abi.OcclusionResult) // 4
        state["results"] = torch.zeros((case["count"], words), dtype=torch.int32, device="cuda")
        state["library"] = hip.library()
    elif kind == "adjoint":
        autodiff = importlib.import_module(PACKAGE + ".autodiff")
        generator = torch.Generator().manual_seed(seed)
        t = case["texture"]
        albedo = (0.1 + 0.8 * torch.rand((t, t, 3), generator=generator)).cuda().contiguous()
        roughness = torch.full((1, 1, 1), 0.3, device="cuda")
        scene, camera, _ = bf.scenes.textured_cornell(case["width"], case["height"],
                                                      albedo=(albedo.data_ptr(), t, t, 3),
                                                      roughness=(roughness.data_ptr(), 1, 1, 1))
        frame = bf.scenes.frame_desc(camera, case["spp"], seed=seed)
        state["frame"] = autodiff.DifferentiableFrame(hip.XpuScene(scene), frame, _options(bf, case, "balance"),
                                                      [albedo, roughness])
        # dLoss/d(image) of a mean absolute error: one sign a channel
        sign = torch.rand((case["height"], case["width"], 3), generator=generator) < 0.8
        state["image_gradient"] = (sign.to(torch.float32) * 2.0 - 1.0).cuda() / sign.numel()
    else:
        autodiff = importlib.import_module(PACKAGE + ".autodiff")
        options = bf.scenes.transport_options(max_depth=case["depth"], mis=bf.abi.MIS_BALANCE, rr_first_depth=0)
        options.failure_policy = bf.abi.FAILURES_COUNT
        specs = bf.scenes.fit_specs(count=case["scenes"], min_resolution=case["min_resolution"],
                                    max_resolution=case["max_resolution"])
        generator = torch.Generator().manual_seed(seed)
        frames, parameters, size = [], [], case["texture"]
        for k, spec in enumerate(specs):
            albedo, widths = (torch.from_numpy(a).cuda().contiguous()
                              for a in bf.scenes.fit_textures(spec["seed"] + seed, size=size))
            r = spec["resolution"]
            scene, camera = bf.scenes.icosphere_grid(r, r, grid=spec["grid"], seed=spec["seed"] ^ seed,
                                                     materials="textured", albedo=(albedo.data_ptr(), size, size, 3),
                                                     roughness=(widths.data_ptr(), size, size, 2))
            target = torch.rand((r, r, 3), generator=generator).cuda()
            frames.append((hip.XpuScene(scene), bf.scenes.frame_desc(camera, case["spp"], seed=seed + k), target,
                           [albedo, widths]))
            parameters += [(albedo, 0.02, 0.0, 1.0), (widths, 0.01, 0.01, 1.0)]
        paths = sum(f.camera.width * f.camera.height * f.samples_per_pixel for _, f, _, _ in frames)
        state["fit"] = autodiff.TextureFit(frames, options, parameters,
                                           workspace=hip.XpuWavefrontTransportWorkspace(paths))
    return state


def _film(film):
    return [film.float_sum, film.compensated, film.counts]


def run(state):
    hip, kind = state["hip"], state["kind"]
    if kind == "frame":
        r = hip.trace_xpu_wavefront_transport(state["workspace"], state["scene"], state["frame"], state["options"],
                                              synchronize=False)
        return _film(r["film"])
    if kind == "batch":
        r = hip.trace_xpu_wavefront_batch(state["workspace"], state["items"], state["options"], synchronize=False)
        return [t for film in r["films"] for t in _film(film)]
    if kind == "paths":
        r = hip.trace_xpu_wavefront_paths(state["workspace"], state["scene"], state["inputs"], state["options"],
                                          synchronize=False, want_host=False)
        return [t.view(torch.int32) for t in r["device"]]
    if kind in ("closest", "occlusion"):
        rays, results, library = state["rays"], state["results"], state["library"]
        stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
        if kind == "closest":
            status = library.blackframe_hip_launch_scene_closest_hit(
                state["scene"].handle, ctypes.c_void_p(rays.data_ptr()), rays.shape[0],
                ctypes.c_void_p(results.data_ptr()), None, stream)
        else:
            status = library.blackframe_hip_launch_scene_occlusion(
                state["scene"].handle, ctypes.c_void_p(rays.data_ptr()), rays.shape[0],
                ctypes.c_void_p(results.data_ptr()), stream)
        if status != 0:
            raise RuntimeError(library.blackframe_hip_last_error().decode())
        if kind == "occlusion":
            return [results]
        # the record's float words (t, barycentrics, normal) apart from its whole ones (status, ids)
        return [results.view(torch.float32)[:, 4:11], results[:, 0:4], results[:, 11:]]
    if kind == "adjoint":
        image = state["frame"].render()
        return [image, *state["frame"].gradients(state["image_gradient"])]
    fit = state["fit"]
    fit.forward()
    losses = fit.loss()
    fit.adjoint()
    return [losses, *(f["film"].float_sum for f in fit.frames), *(p["gradient"] for p in fit.parameters)]


# ---- what a pass cannot do without --------------------------------------------------------------
def _traversal_flops(triangles):
    """One ray: two box tests (18 operations each) at every level of a median-split tree, twice over
    for the boxes that overlap, and a handful of triangle tests (60)."""
    return 2 * 2 * 18 * max(1.0, math.log2(triangles + 1.0)) + 4 * 60


def _frame_work(paths, pixels, triangles, depth, mean_vertices=1.2, replay=False):
    """Scene once (48 bytes a triangle and 64 a node), film once; per path vertex a closest-hit and
    a shadow ray and about 1500 operations of shading."""
    vertices = paths * min(float(depth) + 1.0, mean_vertices)
    rays = vertices * (1.0 if replay else 2.0)
    return (112.0 * triangles + 64.0 * pixels, rays * _traversal_flops(triangles) + 1500.0 * vertices)


def _triangles(case):
    return 34 if case["scene"] in ("cornell", "mapped") else 1280 * case["grid"] ** 2 + 1


def work(case):
    kind = case["kind"]
    if kind == "frame":
        pixels = case["width"] * case["height"]
        vertices = 1.2 if case["scene"] == "grid" else 2.7
        b, f = _frame_work(pixels * case["spp"], pixels, _triangles(case), case["depth"], vertices)
    elif kind == "batch":
        b = f = 0.0
        for k in range(case["scenes"]):
            size = max(16, case["max_resolution"] >> (k % 3))
            pixels = size * max(16, size * 3 // 4 + k)
            grid = (20, 3, 12, 6, 16, 9, 4, 14)[k % 8]
            db, df = _frame_work(pixels * max(1, case["max_spp"] >> ((2 * k) % 4)), pixels, 1280 * grid * grid,
                                 case["depth"])
            b, f = b + db, f + df
    elif kind == "paths":
        b, f = _frame_work(case["count"], 0, 1280 * case["grid"] ** 2, case["depth"])
        b += (24 + 48 + 8 + 128 + 128 + 48 + 8 + 16) * case["count"]
    elif kind in ("closest", "occlusion"):
        triangles = _triangles(case)
        b = 112.0 * triangles + (48 + (80 if kind == "closest" else 16)) * case["count"]
        f = case["count"] * _traversal_flops(triangles)
    elif kind == "adjoint":
        pixels = case["width"] * case["height"]
        b, f = _frame_work(pixels * case["spp"], pixels, 34, case["depth"], 2.7)
        _, g = _frame_work(pixels * case["spp"], pixels, 34, case["depth"], 2.7, replay=True)
        b, f = b + 24 * case["texture"] ** 2 + 12 * pixels, f + g
    else:
        pixels = case["scenes"] * ((case["min_resolution"] + case["max_resolution"]) // 2) ** 2
        b, f = _frame_work(pixels * case["spp"], pixels, 100000, case["depth"], 2.0)
        _, g = _frame_work(pixels * case["spp"], pixels, 100000, case["depth"], 2.0, replay=True)
        b, f = b * case["scenes"] + 40 * case["scenes"] * case["texture"] ** 2, f + g
    return {"bytes": float(b), "flops": float(f)}


def tolerance(case):
    if case["kind"] in ("adjoint", "fit"):
        # run to run, atomics in another order: 2.4e-7 at worst over these ranges
        return {"rel": 1e-6}
    return "exact"


# ---- 64-bit results -----------------------------------------------------------------------------
def exact(case, seed):
    """Closest hits of a small scene by testing every triangle in float64. A path-traced film is an
    estimate over millions of data-dependent paths and has no such value here."""
    if case["kind"] != "closest" or case["scene"] != "cornell" or case["count"] > 20000:
        return None
    bf, _ = _package()
    scene, _ = _host_scene(bf, case, seed)
    corners, owners = [], []
    positions = np.asarray(scene.positions, dtype=np.float64).reshape(-1, 3)
    faces = np.asarray(scene.indices, dtype=np.int64).reshape(-1, 3)
    for record in scene.instances:
        _, first_vertex, _, first_face, face_count = scene.geometries[record.geometry_index]
        m = np.array(list(record.local_to_world), dtype=np.float64).reshape(3, 4)
        tri = positions[first_vertex + faces[first_face:first_face + face_count]]
        corners.append(tri @ m[:, :3].T + m[:, 3])
    tri = np.concatenate(corners)
    rays = _rays(case, seed, case["count"]).astype(np.float64)
    o, d = rays[:, None, 0:3], rays[:, None, 4:7]
    e1, e2 = tri[:, 1] - tri[:, 0], tri[:, 2] - tri[:, 0]
    with np.errstate(divide="ignore", invalid="ignore"):
        p = np.cross(d, e2[None])
        det = np.sum(e1[None] * p, axis=2)
        s = o - tri[None, :, 0]
        u = np.sum(s * p, axis=2) / det
        q = np.cross(s, e1[None])
        v = np.sum(d * q, axis=2) / det
        t = np.sum(e2[None] * q, axis=2) / det
        ok = (u >= -1e-9) & (v >= -1e-9) & (u + v <= 1 + 1e-9) & (t >= 0.0) & np.isfinite(t)
    t = np.where(ok, t, np.inf)
    best = np.argmin(t, axis=1)
    rows = np.arange(len(best))
    hit = np.isfinite(t[rows, best])
    out = np.zeros((len(best), 7))
    ub, vb = u[rows, best], v[rows, best]
    n = np.cross(e1, e2)
    n /= np.linalg.norm(n, axis=1, keepdims=True)
    out[:, 0], out[:, 1], out[:, 2], out[:, 3] = t[rows, best], 1.0 - ub - vb, ub, vb
    out[:, 4:7] = n[best]
    out[~hit] = 0.0
    return [torch.from_numpy(out), None, None]
