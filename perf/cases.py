"""Performance cases of the renderer, each through the calls a program makes.

A case is a dict of plain values. `kind` says which use it stands for:

  preview   one frame of an interactive viewer: the camera moved, one sample per
            pixel, the display image read for the window (latency and launches)
  final     a still of a closed scene with an area light: next-event estimation
            and MIS, the linear image read at the end (optionally with the
            denoiser's feature images)
  sky       a still of a displaced sphere of many triangles and materials under
            an HDR sky, in any render mode, with or without environment
            importance sampling (`freq` 229 at 1920x1080, 64 spp, hero
            wavelengths is the repository's headline workload)
  stress    incoherent paths among instances and a cloud of small triangles
  textured  textures in every slot, MASK and BLEND alpha, the feature images a
            denoiser takes
  edit      an editor's step: one object moved to two places, each drawn
  inverse   one step of inverse rendering: forward image, loss, gradients
  cache     frames of the neural radiance cache while it trains
  fit       the cache network on host records: inference and a loss gradient
  rays      closest-hit queries on device memory (serving, simulation)
  probe     closest-hit and shadow queries on host arrays (tools, picking)

Scenes, cameras and values come from the seed; resolutions, sample counts and
depths from the case. Every pass of an image case starts its render anew, so a
pass on the same state draws the same image.
"""

from __future__ import annotations

import functools
import math

import numpy as np
import torch

import vkrt_amd as V
from vkrt_amd import autograd, scenes

RGB, SINGLE, HERO = "rgb", "single", "hero"


# ----------------------------------------------------------------- cases --
def listed():
    return [
        # a viewer's frame on the smallest scene: nothing but latency
        {"name": "preview", "kind": "preview", "width": 256, "height": 256, "spp": 1, "depth": 8, "mode": RGB},
        # a still of the same box at the size and quality it is saved with
        {"name": "final", "kind": "final", "width": 1024, "height": 1024, "spp": 16, "depth": 8, "mode": RGB,
         "features": False},
        # the headline workload: 1.05M triangles, 64 materials, sky with sun, hero wavelengths
        {"name": "sky_1080p_hero", "kind": "sky", "freq": 229, "width": 1920, "height": 1080, "spp": 64, "depth": 12,
         "mode": HERO, "env_nee": False},
        # glass and dispersion at one wavelength per path, sky sampled, ragged extent
        {"name": "sky_single_nee", "kind": "sky", "freq": 61, "width": 961, "height": 543, "spp": 8, "depth": 12,
         "mode": SINGLE, "env_nee": True},
        # incoherent traversal over 2.7M triangles, long paths
        {"name": "stress", "kind": "stress", "instances": 16, "freq": 72, "triangles": 1000000, "width": 1280,
         "height": 720, "spp": 8, "depth": 16, "mode": RGB},
        # every texture slot, alpha tests on extension and shadow rays, denoiser features
        {"name": "textured", "kind": "textured", "width": 801, "height": 601, "spp": 8, "depth": 8, "mode": RGB,
         "features": True},
        # a dragged object: transform, scene update with BVH build, frame; twice
        {"name": "edit", "kind": "edit", "objects": 12, "freq": 40, "width": 640, "height": 360, "spp": 2, "depth": 6,
         "mode": RGB},
        # 64 materials and a 512 x 256 sky from a loss on the image
        {"name": "inverse", "kind": "inverse", "width": 512, "height": 512, "spp": 32, "depth": 8},
        # two frames of the cache while it tracks a scene: its default paths, steps and batch
        {"name": "cache", "kind": "cache", "width": 1280, "height": 720, "spp": 1, "depth": 8, "mode": RGB,
         "frames": 2},
        # a tool's pass over recorded radiance, a ragged count above one training slice
        {"name": "fit", "kind": "fit", "records": 100003},
        # 4M incoherent rays against 1.05M triangles, on device memory
        {"name": "rays_device", "kind": "rays", "freq": 229, "rays": 4194304},
        # a tool's 131,071 rays and as many shadow rays, on host arrays
        {"name": "probe_host", "kind": "probe", "freq": 31, "rays": 131071},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _extent(rng, lo, hi):
    """Width and height of about `lo`..`hi` pixels, any aspect from 1:1 to 16:9, odd sizes among them."""
    pixels = _log_int(rng, lo, hi)
    aspect = rng.uniform(1.0, 16.0 / 9.0)
    return max(8, int(math.sqrt(pixels * aspect))), max(8, int(math.sqrt(pixels / aspect)))


def draw(rng):
    kind = rng.choice(["preview", "final", "sky", "sky", "stress", "textured", "edit", "inverse", "cache", "fit",
                       "rays", "probe"])
    mode = rng.choice([RGB, SINGLE, HERO])
    if kind == "preview":
        w, h = _extent(rng, 20000, 2000000)
        return {"kind": kind, "width": w, "height": h, "spp": 1, "depth": rng.randint(3, 12), "mode": mode}
    if kind == "final":
        w, h = _extent(rng, 60000, 2000000)
        return {"kind": kind, "width": w, "height": h, "spp": _log_int(rng, 2, 16), "depth": rng.randint(4, 12),
                "mode": mode, "features": rng.random() < 0.25}
    if kind == "sky":
        w, h = _extent(rng, 60000, 2000000)
        return {"kind": kind, "freq": _log_int(rng, 12, 200), "width": w, "height": h, "spp": _log_int(rng, 1, 24),
                "depth": rng.randint(4, 12), "mode": mode, "env_nee": rng.random() < 0.5}
    if kind == "stress":
        w, h = _extent(rng, 60000, 1000000)
        return {"kind": kind, "instances": rng.randint(2, 16), "freq": _log_int(rng, 12, 72),
                "triangles": _log_int(rng, 20000, 1000000), "width": w, "height": h, "spp": _log_int(rng, 1, 8),
                "depth": rng.randint(4, 16), "mode": mode}
    if kind == "textured":
        w, h = _extent(rng, 60000, 1000000)
        return {"kind": kind, "width": w, "height": h, "spp": _log_int(rng, 1, 8), "depth": rng.randint(4, 10),
                "mode": mode, "features": rng.random() < 0.5}
    if kind == "edit":
        w, h = _extent(rng, 60000, 600000)
        return {"kind": kind, "objects": rng.randint(2, 16), "freq": _log_int(rng, 8, 48), "width": w, "height": h,
                "spp": rng.randint(1, 4), "depth": rng.randint(4, 8), "mode": mode}
    if kind == "inverse":
        w, h = _extent(rng, 16000, 262144)
        return {"kind": kind, "width": w, "height": h, "spp": _log_int(rng, 4, 32), "depth": rng.randint(4, 8)}
    if kind == "cache":
        w, h = _extent(rng, 60000, 2000000)
        return {"kind": kind, "width": w, "height": h, "spp": 1, "depth": rng.randint(5, 10),
                "mode": rng.choice([RGB, HERO]), "frames": rng.randint(1, 3)}
    if kind == "fit":
        return {"kind": kind, "records": _log_int(rng, 500, 200000)}
    if kind == "rays":
        return {"kind": kind, "freq": _log_int(rng, 12, 200), "rays": _log_int(rng, 3000, 4000000)}
    return {"kind": kind, "freq": _log_int(rng, 8, 40), "rays": _log_int(rng, 1000, 200000)}


# ---------------------------------------------------------------- scenes --
@functools.lru_cache(maxsize=16)
def _sphere_topology(freq, parts):
    """Unit sphere vertices, triangles, and for each of `parts` meshes its vertices and local triangles."""
    verts, tris = scenes.geodesic_sphere(freq)
    mesh = (np.arange(len(tris), dtype=np.uint64) * np.uint64(0x9E3779B97F4A7C15) >> np.uint64(40)) % np.uint64(parts)
    pieces = []
    for k in range(parts):
        f = tris[mesh == k]
        if len(f):
            used, local = np.unique(f, return_inverse=True)
            pieces.append((used, local.reshape(-1, 3).astype(np.uint32)))
    return verts, tris, pieces


def _blob(freq, rng, amplitude=0.1):
    """Vertices (20 floats each) of the sphere displaced by a few smooth waves."""
    verts, tris, _ = _sphere_topology(freq, 1)
    k = rng.normal(size=(6, 3)) * np.array([2.0, 3.0, 4.0, 6.0, 8.0, 12.0])[:, None]
    a = np.array([1.0, 0.8, 0.6, 0.35, 0.25, 0.15])
    disp = (np.sin(verts @ k.T + rng.uniform(0, 6.28, 6)) * (a / a.sum())).sum(axis=1)
    pos = verts * (1.0 + amplitude * disp)[:, None]
    fn = np.cross(pos[tris[:, 1]] - pos[tris[:, 0]], pos[tris[:, 2]] - pos[tris[:, 0]])
    nrm = np.stack([sum(np.bincount(tris[:, c], fn[:, x], len(pos)) for c in range(3)) for x in range(3)], axis=1)
    nrm /= np.maximum(np.linalg.norm(nrm, axis=1, keepdims=True), 1e-30)
    return V.make_vertices(pos, nrm)


@functools.lru_cache(maxsize=4)
def _sky(width, height, sun):
    return scenes.sky_environment(width, height, sun_radiance=sun)


def _materials(rng, count):
    """A mix of coated diffuse, metal and (dispersive, sometimes absorbing) glass."""
    out = []
    for _ in range(count):
        m = V.default_material(baseColor=tuple(float(x) for x in rng.uniform(0.05, 0.95, 3)),
                               roughness=float(rng.uniform(0.05, 1.0)), metallic=0.0, specular=0.5)
        pick = rng.random()
        if pick < 0.2:
            m.transmission = 1.0
            m.ior = 1.5
            m.abbeNumber = 0.0 if pick < 0.12 else 32.0
            m.absorptionCoefficient = 0.0 if pick < 0.16 else 0.5
            m.attenuationColor[:] = (0.8, 0.9, 0.7)
        elif pick < 0.3:
            m.metallic = 1.0
        out.append(m)
    return out


def _box_scene(rng):
    """The Cornell box with walls of other colours and another light strength."""
    s = scenes.cornell_box()
    for m in s.materials[1:3]:
        m.baseColor[:] = tuple(float(x) for x in rng.uniform(0.1, 0.7, 3))
    s.materials[3].emissionLuminance = float(rng.uniform(10.0, 20.0))
    x, z = rng.uniform(0.4, 0.6, 2)
    s.camera = ((float(x), -1.35, float(z)), (0.5, 0.5, 0.5), (0.0, 0.0, 1.0), 40.0)
    return s


def _sky_scene(case, rng):
    """The displaced sphere split over 64 materials under a 2048 x 1024 sky with a sun."""
    s = scenes.Scene()
    s.materials = _materials(rng, 64)
    vertices = _blob(case["freq"], rng)
    for m, (used, local) in enumerate(_sphere_topology(case["freq"], 64)[2]):
        s.meshes.append(scenes.MeshData(vertices[used], local, m))
    a = rng.uniform(0, 2 * math.pi)
    s.camera = ((3.4 * math.cos(a), 3.4 * math.sin(a), 1.1), (0.0, 0.0, 0.0), (0.0, 0.0, 1.0), 40.0)
    s.environment = _sky(2048, 1024, 1.0e4)
    return s


def _stress_scene(case, rng):
    s = scenes.Scene()
    s.materials = [scenes.lambert((0.7, 0.7, 0.7)), scenes.lambert((0.5, 0.6, 0.8))]
    vertices = _blob(case["freq"], rng)
    index = _sphere_topology(case["freq"], 1)[1].astype(np.uint32)
    for _ in range(case["instances"]):
        m = np.eye(4)
        q = np.linalg.qr(rng.normal(size=(3, 3)))[0]
        m[:3, :3] = q * np.sign(np.linalg.det(q))
        m[:3, 3] = rng.uniform(-2.5, 3.5, 3)
        s.meshes.append(scenes.MeshData(vertices, index, 0, m))
    s.meshes.append(scenes.random_triangles(case["triangles"], seed=int(rng.integers(1 << 30))))
    s.meshes[-1].material = 1
    s.camera = ((0.5, -4.5, 1.2), (0.5, 0.5, 0.5), (0.0, 0.0, 1.0), 60.0)
    s.environment_color, s.environment_strength = (1.0, 1.0, 1.0), 1.0
    return s


def _edit_scene(case, rng):
    """Objects on a floor under an area light and a dim constant sky; object 0 is the one moved."""
    s = scenes.Scene()
    s.materials = [scenes.lambert((0.6, 0.6, 0.6)), scenes.lambert((0.7, 0.7, 0.7), emission=12.0)]
    s.materials += [V.default_material(baseColor=tuple(float(x) for x in rng.uniform(0.1, 0.9, 3)),
                                       roughness=float(rng.uniform(0.2, 1.0)), specular=0.5, metallic=0.0)
                    for _ in range(4)]
    index = _sphere_topology(case["freq"], 1)[1].astype(np.uint32)
    shapes = [_blob(case["freq"], rng) for _ in range(2)]
    for k in range(case["objects"]):
        s.meshes.append(scenes.MeshData(shapes[k % 2], index, 2 + k % 4, _pose(rng)))
    quad = np.array([[0, 1, 2], [0, 2, 3]], np.uint32)
    floor = np.array([[-6, -6, 0], [6, -6, 0], [6, 6, 0], [-6, 6, 0]], np.float32)
    light = np.array([[-1, -1, 5], [-1, 1, 5], [1, 1, 5], [1, -1, 5]], np.float32)
    up = np.tile(np.array([[0, 0, 1]], np.float32), (4, 1))
    s.meshes.append(scenes.MeshData(V.make_vertices(floor, up), quad, 0))
    s.meshes.append(scenes.MeshData(V.make_vertices(light, -up), quad, 1))
    s.camera = ((0.0, -9.0, 4.0), (0.0, 0.0, 0.7), (0.0, 0.0, 1.0), 45.0)
    s.environment_color, s.environment_strength = (0.6, 0.7, 0.9), 0.3
    return s


def _pose(rng):
    m = np.eye(4)
    a, size = rng.uniform(0, 2 * math.pi), rng.uniform(0.3, 0.8)
    m[:2, :2] = [[math.cos(a), -math.sin(a)], [math.sin(a), math.cos(a)]]
    m[:3, :3] *= size
    m[:3, 3] = [rng.uniform(-3, 3), rng.uniform(-3, 3), 1.1 * size]
    return m


def _renderer(case, scene, seed, tone=V.TONE_NONE):
    w, h = case.get("width", 64), case.get("height", 64)
    r = V.Renderer(w, h)
    scenes.load(r, scene)
    mode = case.get("mode", RGB)
    r.configure(spp=case.get("spp", 1), max_depth=case.get("depth", 8), min_depth=4,
                mode=V.RENDER_MODE_RGB if mode == RGB else V.RENDER_MODE_SPECTRAL,
                spectral=V.SPECTRAL_HERO if mode == HERO else V.SPECTRAL_SINGLE, tone=tone, rng=V.RNG_PCG32,
                seed=1 + seed % 1000003, env_importance=bool(case.get("env_nee")))
    if case.get("features"):
        r.set_denoiser_features(True)
    r.start(w, h, 0)
    return r


def _tint(scene, rng):
    """Another strength for everything a scene emits, so that another seed is another scene."""
    for m in scene.materials:
        m.emissionLuminance *= float(rng.uniform(0.7, 1.3))
        m.baseColor[:] = [float(c) for c in np.clip(np.array(m.baseColor[:]) * rng.uniform(0.8, 1.1), 0.0, 1.0)]
    return scene


def _network(rng):
    """He-initialised weights of the cache network in its documented order (biases ride on the constant input)."""
    w = np.zeros(29696, np.float32)
    w0 = np.zeros((64, 192), np.float32)
    w0[:, :173] = rng.uniform(-1, 1, (64, 173)) * math.sqrt(6 / 173)
    w[:12288] = w0.ravel()
    w[12288:28672] = rng.uniform(-1, 1, 16384) * math.sqrt(6 / 64)
    w[28672:28672 + 192] = rng.uniform(-1, 1, 192) * math.sqrt(6 / 64)
    return w


def _records(case, rng):
    """Cache inputs in [0, 1] and the noisy, non-negative radiance recorded there."""
    n = case["records"]
    x = rng.random((n, 11), dtype=np.float32)
    smooth = np.stack([1 + np.sin(3 * x[:, 0] + c) * np.cos(2 * x[:, 1] - c) for c in range(3)], axis=1)
    target = (smooth * x[:, 8:11] * rng.gamma(2.0, 0.5, (n, 1))).astype(np.float32)
    return x, target


def _rays(rng, n):
    """Rays through the object's ball from all around and from inside it, as 8 floats (origin, tmin, direction, tmax)."""
    d = rng.normal(size=(n, 3)).astype(np.float32)
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    target = rng.uniform(-1.0, 1.0, (n, 3)).astype(np.float32)
    rays = np.empty((n, 8), np.float32)
    rays[:, 0:3] = target - d * rng.uniform(0.0, 4.0, (n, 1)).astype(np.float32)
    rays[:, 3] = 1e-3
    rays[:, 4:7] = d
    rays[:, 7] = 1e4
    return rays


def _ray_scene(case, rng):
    s = scenes.Scene()
    s.materials = [scenes.lambert((0.7, 0.7, 0.7))]
    s.meshes.append(scenes.MeshData(_blob(case["freq"], rng),
                                    _sphere_topology(case["freq"], 1)[1].astype(np.uint32), 0))
    return s


# ------------------------------------------------------------------ runs --
def prepare(case, seed):
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    if kind == "preview":
        return {"case": case, "r": _renderer(case, _box_scene(rng), seed, tone=V.TONE_ACES),
                "pose": ((float(rng.uniform(0.3, 0.7)), -1.35, 0.5), (0.5, 0.5, 0.5), (0.0, 0.0, 1.0), 40.0)}
    if kind in ("final", "cache"):
        r = _renderer(case, _box_scene(rng), seed)
        if kind == "cache":
            r.nrc_reset(1 + seed % 1000003)
            # the rate of a cache that follows a scene it has seen; at the library's starting rate of
            # 1e-2 the order in which the GPU writes records alone moves the weights by 4 %
            r.set_neural_cache(True, learningRate=1e-3)
        return {"case": case, "r": r}
    if kind == "sky":
        return {"case": case, "r": _renderer(case, _sky_scene(case, rng), seed)}
    if kind == "stress":
        return {"case": case, "r": _renderer(case, _stress_scene(case, rng), seed)}
    if kind == "textured":
        return {"case": case, "r": _renderer(case, _tint(scenes.textured_cornell(), rng), seed)}
    if kind == "edit":
        r = _renderer(case, _edit_scene(case, rng), seed)
        return {"case": case, "r": r, "poses": [np.ascontiguousarray(_pose(rng).T, dtype=np.float32) for _ in range(2)]}
    if kind == "inverse":
        scene = scenes.differentiable_cornell(seed)
        r = _renderer(case, scene, seed)
        autograd.forget(r)
        p = autograd.SceneParameters.from_renderer(r, scene.environment)
        p = autograd.SceneParameters(*[t.requires_grad_(True) for t in p.tensors()])
        target = torch.from_numpy(rng.uniform(0.0, 1.0, (case["height"], case["width"], 3)).astype(np.float32))
        return {"case": case, "r": r, "params": p, "view": scenes.prb_views(seed, 1)[0], "target": target}
    if kind == "fit":
        r = V.Renderer(16, 16)
        r.nrc_set_weights(_network(rng))
        x, t = _records(case, rng)
        return {"case": case, "r": r, "inputs": x, "targets": t}
    r = _renderer(case, _ray_scene(case, rng), seed)
    r.draw()  # the scene is on the device before queries are served
    rays = _rays(rng, case["rays"])
    if kind == "probe":
        return {"case": case, "r": r, "rays": rays}
    n = case["rays"]
    dev = {"mesh": torch.empty(n, dtype=torch.int32, device="cuda"),
           "prim": torch.empty(n, dtype=torch.int32, device="cuda"),
           "t": torch.empty(n, dtype=torch.float32, device="cuda"),
           "bary": torch.empty((n, 2), dtype=torch.float32, device="cuda")}
    return {"case": case, "r": r, "rays": torch.from_numpy(rays).cuda(), "out": dev}


def run(state):
    case, r = state["case"], state["r"]
    kind = case["kind"]
    if kind == "preview":
        r.set_camera(*state["pose"])
        r.draw()
        return r.output_image()
    if kind == "edit":
        images = []
        for pose in state["poses"]:
            r.set_mesh_transform_matrix(0, pose.reshape(-1))
            r.start(case["width"], case["height"], 0)
            r.draw()
            images.append(r.output_image())
        return images
    if kind == "inverse":
        p = state["params"]
        for t in p.tensors():
            t.grad = None
        image = autograd.render(r, p, state["view"])
        ((image - state["target"]) ** 2).sum().backward()
        return [image] + [t.grad for t in p.tensors()]
    if kind == "fit":
        grad, loss = r.nrc_gradient(state["inputs"], state["targets"])
        return {"out": r.nrc_infer(state["inputs"]), "gradient": grad, "loss": loss}
    if kind == "rays":
        o = state["out"]
        r.trace_rays_device_noalloc(state["rays"].data_ptr(), case["rays"], o["mesh"].data_ptr(), o["prim"].data_ptr(),
                                    o["t"].data_ptr(), o["bary"].data_ptr())
        return o
    if kind == "probe":
        mesh, prim, t, bary = r.trace_rays(state["rays"])
        return {"mesh": mesh.view(np.int32), "prim": prim.view(np.int32), "t": t, "bary": bary,
                "visible": r.trace_shadow_rays(state["rays"]).view(np.int32)}
    r.start(case["width"], case["height"], 0)
    for _ in range(case.get("frames", 1)):
        r.draw()
    if kind == "cache":
        return {"image": r.accumulation(), "weights": r.nrc_weights()}
    if case.get("features"):
        return [r.accumulation(), *r.denoiser_features()]
    return r.accumulation()


# ------------------------------------------------------------------ work --
def _triangles(case):
    kind = case["kind"]
    sphere = 20 * case.get("freq", 0) ** 2
    return {"sky": sphere, "stress": sphere * case.get("instances", 0) + case.get("triangles", 0),
            "edit": sphere * case.get("objects", 0) + 4, "rays": sphere, "probe": sphere, "inverse": 138}.get(kind, 40)


def _trace_flops(triangles):
    """A closest hit: eight slab tests (about 12 operations each) on every level of an 8-wide tree, one triangle test."""
    return 96.0 * max(1.0, math.log(triangles, 8)) + 60.0


def work(case):
    kind, tris = case["kind"], _triangles(case)
    scene = 112.0 * tris  # 36 bytes of positions, 64 of shading data and 12 of indices per triangle
    if kind == "fit":
        n = case["records"]
        layers = 192 * 64 + 4 * 64 * 64 + 64 * 3
        return {"bytes": n * (2 * 44.0 + 12.0 + 12.0) + 8 * 29696.0, "flops": 4 * 2.0 * n * layers}
    if kind in ("rays", "probe"):
        n = case["rays"]
        each = (32.0 + 20.0) + (32.0 + 4.0 if kind == "probe" else 0.0)
        return {"bytes": n * each + 36.0 * tris, "flops": n * _trace_flops(tris) * (2 if kind == "probe" else 1)}
    pixels = case["width"] * case["height"]
    frames = 2 if kind == "edit" else case.get("frames", 1)
    paths = pixels * case["spp"] * frames
    # path vertices per path: the open scenes lose most paths to the sky, the boxes keep them for a few bounces
    vertices = {"sky": 1.5, "stress": 3.0, "edit": 2.5}.get(kind, min(4.0, case["depth"]))
    lanes = 4 if case.get("mode") == HERO else 1
    shading = 250.0 + 100.0 * lanes
    shadow = 1 if kind in ("preview", "final", "textured", "edit", "inverse", "cache") or case.get("env_nee") else 0
    flops = paths * vertices * (_trace_flops(tris) * (1 + shadow) + shading)
    image = pixels * (8.0 if kind in ("preview", "edit") else 16.0) * (3.0 if case.get("features") else 1.0)
    if kind == "inverse":  # the replay walks the same paths, with the derivatives of every lobe
        flops *= 3.0
        image += pixels * 12.0 + 512 * 256 * 12.0 * 2
    if kind == "cache":
        flops += pixels * 2.0 * 29696.0 * frames
    env = 2048 * 1024 * 16.0 if kind == "sky" else 0.0
    return {"bytes": scene * (2 if kind == "edit" else 1) + image * (2 if kind == "edit" else 1) + env, "flops": flops}


def tolerance(case):
    kind = case["kind"]
    if kind in ("rays", "probe"):
        # whole numbers agree but for rays through a shared edge; t and the barycentrics are 32-bit
        return {"rel": 1e-4, "max": 0.9, "differ": 1e-5}
    if kind == "fit":
        return {"rel": 2e-3, "max": 0.5}
    if kind == "inverse":
        # gradients are sums of 32-bit atomics in any order
        return {"rel": 1e-3, "max": 0.5}
    if kind == "cache":
        # training draws records in the order the GPU wrote them
        return {"rel": 3e-2, "max": 0.9}
    if kind in ("preview", "edit"):
        return {"differ": 1e-3, "rel": 1e-3, "max": 0.5}
    if kind == "sky":
        # a last-place difference in a lobe or the sky lookup sends a path another way, and the sun is 1e4
        return {"rel": 3e-3, "max": 0.9}
    return {"rel": 1e-4, "max": 0.5}


# ----------------------------------------------------------------- exact --
def _exact_rays(case, seed):
    """Closest hits by testing every triangle in 64 bits; None where that is too many pairs."""
    rng = np.random.default_rng(seed)
    scene = _ray_scene(case, rng)
    rays = _rays(rng, case["rays"])
    tris = len(scene.meshes[0].indices)
    if tris * case["rays"] > 4e9:
        return None
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    pos = torch.from_numpy(scene.meshes[0].vertices[:, :3][scene.meshes[0].indices].astype(np.float64)).to(dev)
    v0, e1, e2 = pos[:, 0], pos[:, 1] - pos[:, 0], pos[:, 2] - pos[:, 0]
    r = torch.from_numpy(rays.astype(np.float64)).to(dev)
    t_out, uv_out, hit_out = [], [], []
    step = max(1, int(3e7) // tris)
    for a in range(0, len(r), step):
        o, d, lo, hi = r[a:a + step, 0:3], r[a:a + step, 4:7], r[a:a + step, 3:4], r[a:a + step, 7:8]
        # Moeller and Trumbore, with the products of the triangle taken out of the ray loop
        n = torch.linalg.cross(e1, e2)
        det = -(d @ n.T)
        dao = torch.linalg.cross(o, d)  # o x d
        nd = d @ torch.linalg.cross(v0, e2).T + dao @ e2.T
        ne = -(d @ torch.linalg.cross(v0, e1).T + dao @ e1.T)
        nt = o @ n.T - (v0 * n).sum(1)
        inv = 1.0 / det
        u, v, t = nd * inv, ne * inv, nt * inv
        ok = (u >= 0) & (v >= 0) & (u + v <= 1) & (t > lo) & (t < hi)
        t = torch.where(ok, t, torch.inf)
        best, k = t.min(dim=1)
        got = torch.isfinite(best)
        t_out.append(torch.where(got, best, 0.0))
        row = torch.arange(len(k), device=dev)
        uv = torch.stack([u[row, k], v[row, k]], 1)
        uv_out.append(torch.where(got[:, None], uv, 0.0))
        hit_out.append(got)
    out = {"mesh": None, "prim": None, "t": torch.cat(t_out).cpu(), "bary": torch.cat(uv_out).cpu()}
    if case["kind"] == "probe":
        out["visible"] = None
    return out


def _encode(x):
    """12 octaves of sine and cosine of the first seven inputs, the other four, a constant 1, zero padding."""
    e = np.zeros((len(x), 192))
    for d in range(7):
        for f in range(12):
            a = x[:, d].astype(np.float64) * 2.0 ** f * math.pi
            e[:, 24 * d + 2 * f], e[:, 24 * d + 2 * f + 1] = np.sin(a), np.cos(a)
    e[:, 168:172] = x[:, 7:11]
    e[:, 172] = 1.0
    return e


def _exact_fit(case, seed):
    """The network on its 16-bit weights, forward and backward, in 64 bits."""
    rng = np.random.default_rng(seed)
    w = _network(rng).astype(np.float16).astype(np.float64)
    x, target = _records(case, rng)
    mats = [w[:12288].reshape(64, 192)] + [w[12288 + 4096 * k:16384 + 4096 * k].reshape(64, 64) for k in range(4)]
    mats.append(w[28672:28672 + 192].reshape(3, 64))
    acts = [_encode(x)]
    for m in mats[:-1]:
        acts.append(np.maximum(acts[-1] @ m.T, 0.0))
    y = acts[-1] @ mats[-1].T
    den = y * y + 0.01
    loss = float((((y - target) ** 2) / den).sum())
    d = np.clip(2 * (y - target) / den, -1000, 1000)
    grads = [None] * 6
    for k in range(5, -1, -1):
        grads[k] = (d.T @ acts[k]).ravel()
        if k:
            d = (d @ mats[k]) * (acts[k] > 0)
    flat = np.concatenate(grads + [np.zeros(13 * 64)])
    return {"out": y, "gradient": flat, "loss": loss}


def exact(case, seed):
    """Queries and the network have closed answers; a path-traced image would need the whole renderer again in 64
    bits (and its random decisions flip with the last place), far beyond 20 seconds at these sizes."""
    if case["kind"] in ("rays", "probe"):
        return _exact_rays(case, seed)
    if case["kind"] == "fit":
        return _exact_fit(case, seed)
    return None
