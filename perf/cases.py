"""The work that programs on this framework have it do, as cases to be timed.

A case is one pass of a public entry point at one size:

  frame    a frame of the wavefront pass: begin_frame, render, end_frame, and
           with "measure" the frame's relMSE against a reference image and its
           accumulation, as an offline render does (scenes: the Cornell box,
           the icosphere field, the field with textures, alpha tests, normal
           maps, an environment image and a thin lens, the field in a grid
           medium; "nrc" turns the radiance cache on)
  views    a frame of many camera views in one launch (render_views)
  mega     a frame of the megakernel pass
  trace    closest hits and visibility of a caller's own rays
  rebuild  an acceleration structure built anew, and rays traced through it
           (a scene whose geometry moves)
  infer    radiance-cache queries
  train    radiance-cache training: the gradient of one batch, or with "steps"
           that many Adam steps on it and the weights afterwards

Scenes, resolutions and params are those of bench.py and of the tests, and
sizes between and below them.
"""
import ctypes as C
import math

import numpy as np
import torch

import kiraray_amd as krr
from kiraray_amd import _abi
from kiraray_amd.nrc import NeuralRadianceCache

MAX_VIEWS = 48


# ---------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------

def listed():
    return [
        # the smallest frame: a thumbnail, where launches and latency count
        frame("cornell", 64, 64, spp=4, max_depth=8, name="frame_thumbnail"),
        # the offline reference render of a small scene, measured and accumulated
        frame("cornell", 256, 256, spp=16, max_depth=8, measure=True, name="frame_cornell_measured"),
        # the ordinary interactive frame on a large scene
        frame("field", 1920, 1080, spp=1, max_depth=16, rr_min_depth=3, spheres=1024, level=3, name="frame_field_1080p"),
        # textured materials, alpha tests, an image environment and a lens, at a ragged size
        frame("textured", 853, 479, spp=2, max_depth=10, spheres=300, level=2, clamp=True, name="frame_textured_ragged"),
        # participating media: the largest frame
        frame("volume", 1280, 720, spp=2, max_depth=32, rr_min_depth=3, spheres=1024, level=3, grid=128, name="frame_volume_720p"),
        # the radiance cache in a frame: queries and online training
        frame("field", 960, 540, spp=1, max_depth=16, rr_min_depth=3, spheres=1024, level=3, nrc=True, name="frame_radiance_cache"),
        # many views of uneven, partly odd sizes per frame
        {"name": "views_uneven", "kind": "views", "spheres": 1024, "level": 3, "views": 32, "largest": 512, "spp": 2, "max_depth": 12},
        # the megakernel pass
        {"name": "mega_field", "kind": "mega", "spheres": 256, "level": 3, "width": 960, "height": 540, "spp": 1, "max_depth": 10},
        # rays of a program's own, closest hit and visibility
        {"name": "trace_million", "kind": "trace", "spheres": 1024, "level": 3, "rays": 1 << 20, "bounces": True},
        # geometry that moves: build, then trace
        {"name": "rebuild_mid", "kind": "rebuild", "spheres": 256, "level": 3, "rays": 1 << 16},
        # radiance-cache queries of a whole frame
        {"name": "infer_frame", "kind": "infer", "samples": 1000003},
        # a frame's training: four steps on one mini-batch size
        {"name": "train_steps", "kind": "train", "samples": 16384, "steps": 4},
    ]


def frame(scene, width, height, spp, max_depth, rr_min_depth=0, spheres=0, level=0, grid=0, clamp=False, measure=False, nrc=False, name=None):
    case = {"kind": "frame", "scene": scene, "width": width, "height": height, "spp": spp, "max_depth": max_depth,
            "rr_min_depth": rr_min_depth, "spheres": spheres, "level": level, "grid": grid, "clamp": clamp, "measure": measure, "nrc": nrc}
    return dict(case, name=name) if name else case


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["frame", "frame", "frame", "views", "mega", "trace", "rebuild", "infer", "train"])
    spheres, level = log_int(16, 1024), rng.choice([2, 2, 3])
    if kind == "frame":
        scene = rng.choice(["cornell", "field", "field", "textured", "volume"])
        pixels = log_int(4096, {"volume": 400000}.get(scene, 1500000))
        width = max(16, int(math.sqrt(pixels * rng.uniform(0.7, 2.0))))
        height = max(16, pixels // width)
        spp = rng.choice([1, 2, 3, 4]) if pixels < 400000 else 1
        return frame(scene, width, height, spp=spp, max_depth=rng.randint(4, 16), rr_min_depth=rng.choice([0, 3]),
                     spheres=0 if scene == "cornell" else spheres, level=0 if scene == "cornell" else level,
                     grid=rng.choice([48, 96, 128]) if scene == "volume" else 0, clamp=rng.random() < 0.3,
                     measure=rng.random() < 0.3, nrc=scene in ("cornell", "field") and rng.random() < 0.3)
    if kind == "views":
        return {"kind": "views", "spheres": spheres, "level": level, "views": log_int(2, 32), "largest": log_int(64, 400),
                "spp": rng.choice([1, 2]), "max_depth": rng.randint(4, 12)}
    if kind == "mega":
        return {"kind": "mega", "spheres": spheres, "level": level, "width": log_int(48, 1000), "height": log_int(48, 700),
                "spp": rng.choice([1, 2]), "max_depth": rng.randint(4, 12)}
    if kind == "trace":
        return {"kind": "trace", "spheres": spheres, "level": level, "rays": log_int(100, 2000000), "bounces": rng.random() < 0.5}
    if kind == "rebuild":
        return {"kind": "rebuild", "spheres": log_int(16, 1024), "level": level, "rays": log_int(1000, 200000)}
    if kind == "infer":
        return {"kind": "infer", "samples": log_int(100, 1000000)}
    return {"kind": "train", "samples": log_int(500, 65536), "steps": rng.choice([0, 1, 3, 4])}


# ---------------------------------------------------------------------------
# scenes
# ---------------------------------------------------------------------------

def _scene_config(case, seed):
    if case.get("scene") == "cornell":
        return {"model": [{"type": "cornell_box"}], "camera": {"eye": [0, 1, 2.8], "target": [0, 1, 0]}}
    cfg = {"model": [{"type": "icosphere_field", "count": case["spheres"], "level": case["level"], "seed": 7 + seed % 1000}],
           "camera": {"eye": [0.5, 0.75, 2.3], "target": [0.5, 0.3, 0.45]}}
    if case.get("scene") == "volume":
        cfg["media"] = [{"type": "value_noise_grid", "res": case["grid"], "octaves": 5, "seed": 11 + seed % 1000,
                         "sigma_t_max": 20.0, "albedo": 0.8, "g": 0.3}]
        cfg["camera"]["medium"] = 0
    if case.get("kind") == "views":
        cfg["views"] = {"count": min(case["views"], MAX_VIEWS), "seed": 5 + seed % 1000, "radius": 2.0, "center": [0.5, 0.5, 0.5]}
    return cfg


def _view_size(case, i):
    top = case["largest"]
    side = (top, max(16, top // 4), max(16, top * 3 // 8 + 1), max(16, top // 2))[i % 4]
    return side, side * 9 // 16 if i % 3 == 1 else side


def _pointer(array, ctype):
    return array.ctypes.data_as(C.POINTER(ctype))


class _TexturedScene:
    """The field's geometry in a scene description of the program's own: image
    textures on its materials, alpha tests on every seventh, normal maps on
    every fifth, and an image environment."""

    def __init__(self, base, seed):
        rng = np.random.default_rng(seed)
        self.base = base  # owns the geometry
        src = base.desc
        pos, _, _ = base.arrays()
        self.uv = np.ascontiguousarray(np.stack([pos[:, 0] * 2.5 + pos[:, 1], pos[:, 2] * 2.5 - pos[:, 1]], 1), np.float32)
        colour = np.ones((61, 83, 4), np.float32)
        colour[..., :3] = 0.1 + 0.8 * rng.random((61, 83, 3), dtype=np.float32)
        gloss = np.ones((32, 32, 4), np.float32)
        gloss[..., 3] = 0.3 + 0.6 * rng.random((32, 32), dtype=np.float32)
        clear = np.zeros((16, 16, 4), np.float32)
        clear[..., :3] = (rng.random((16, 16, 1)) < 0.4).astype(np.float32) * 0.9
        bumps = np.ones((40, 40, 4), np.float32)
        bumps[..., :2] = 0.5 + 0.2 * (rng.random((40, 40, 2), dtype=np.float32) - 0.5)
        self.images = [colour, gloss, clear, bumps]
        self.textures = (_abi.krr_texture * len(self.images))()
        for t, image in zip(self.textures, self.images):
            t.height, t.width = image.shape[:2]
            t.rgba = _pointer(image, C.c_float)
        self.materials = (krr.krr_material * src.n_materials)()
        C.memmove(self.materials, src.materials, C.sizeof(self.materials))
        for i, m in enumerate(self.materials):
            if m.type == _abi.KRR_MAT_DIFFUSE:
                m.diffuse_texture = 1
            elif m.type == _abi.KRR_MAT_CONDUCTOR:
                m.specular_texture = 2
            if i % 7 == 3:
                m.transmission_texture = 3
            if i % 5 == 1:
                m.normal_texture = 4
        self.meshes = (krr.krr_mesh * src.n_meshes)()
        C.memmove(self.meshes, src.meshes, C.sizeof(self.meshes))
        for m in self.meshes:
            m.has_texcoords = 1
        self.sky = (0.2 + rng.random((32, 64, 4))).astype(np.float32)
        self.light = (_abi.krr_infinite_light * 1)()
        self.light[0].tint[:] = [1.0, 0.95, 0.9]
        self.light[0].scale = 0.5
        self.light[0].image_height, self.light[0].image_width = self.sky.shape[:2]
        self.light[0].image_rgba = _pointer(self.sky, C.c_float)
        self.desc = krr.krr_scene_desc()
        C.memmove(C.byref(self.desc), C.byref(src), C.sizeof(src))
        self.desc.materials, self.desc.meshes = self.materials, self.meshes
        self.desc.texcoords = _pointer(self.uv, C.c_float)
        self.desc.n_textures, self.desc.textures = len(self.images), self.textures
        self.desc.n_infinite_lights, self.desc.infinite_lights = 1, self.light


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _first_frame(seed):
    return 1 + seed % 4093


# ---------------------------------------------------------------------------
# prepare and run
# ---------------------------------------------------------------------------

def prepare(case, seed):
    torch.cuda.init()
    torch.cuda.current_stream()
    return {"frame": _prepare_frame, "mega": _prepare_frame, "views": _prepare_views, "trace": _prepare_trace, "rebuild": _prepare_trace,
            "infer": _prepare_cache, "train": _prepare_cache}[case["kind"]](case, seed)


def run(state):
    return {"frame": _run_frame, "mega": _run_frame, "views": _run_views, "trace": _run_trace, "rebuild": _run_rebuild,
            "infer": _run_infer, "train": _run_train}[state["case"]["kind"]](state)


def _prepare_frame(case, seed):
    w, h = case["width"], case["height"]
    scene = krr.Scene(_scene_config(case, seed))
    camera = scene.camera(0)
    camera.aspect_ratio = w / h
    params = {"spp": case["spp"], "max_depth": case["max_depth"], "rr": 0.8}
    if case["kind"] == "mega":
        tracer = krr.MegakernelPathTracer(params)
    else:
        params.update(rr_min_depth=case["rr_min_depth"], enable_clamp=case["clamp"], clamp_max=100.0)
        if case["nrc"]:
            params["nrc"] = {"train_mod": 16, "batch": 131072, "steps_per_frame": 1, "lr": 1e-3}
        tracer = krr.WavefrontPathTracer(params)
    if case.get("scene") == "textured":
        scene = _TexturedScene(scene, seed)
        camera.lens_radius = 0.004
        camera.focal_distance = 2.0
    tracer.set_scene(scene.desc)
    tracer.resize(w, h)
    state = {"case": case, "scene": scene, "tracer": tracer, "camera": camera, "frame": _first_frame(seed), "count": 0,
             "film": torch.empty(h, w, 4, device="cuda")}
    if case.get("measure"):
        state["reference"] = torch.rand(h, w, 4, device="cuda", generator=_generator(seed)) + 0.1
        state["sum"] = torch.zeros(h, w, 4, device="cuda", dtype=torch.float64)
    return state


def _run_frame(s):
    tracer, film = s["tracer"], s["film"]
    tracer.begin_frame(s["camera"], s["frame"])
    tracer.render(film.data_ptr(), _stream())
    tracer.end_frame()
    s["frame"] += 1
    if "reference" not in s:
        return {"film": film}
    n = s["case"]["width"] * s["case"]["height"]
    error = krr.error_metric(3, film.data_ptr(), s["reference"].data_ptr(), n, _stream())
    krr.accumulate(s["sum"].data_ptr(), film.data_ptr(), n, s["count"], 0, 0, 64, _stream())
    s["count"] += 1
    return {"film": film, "sum": s["sum"], "relmse": error}


def _prepare_views(case, seed):
    scene = krr.Scene(_scene_config(case, seed))
    tracer = krr.WavefrontPathTracer({"spp": case["spp"], "max_depth": case["max_depth"], "rr": 0.8, "rr_min_depth": 3})
    tracer.set_scene(scene.desc)
    films, views = [], []
    for i in range(scene.n_views):
        w, h = _view_size(case, i)
        camera = scene.camera(i)
        camera.aspect_ratio = w / h
        films.append(torch.empty(h, w, 4, device="cuda"))
        views.append((camera, w, h, films[-1].data_ptr()))
    tracer.set_views(views)
    return {"case": case, "scene": scene, "tracer": tracer, "films": films, "frame": _first_frame(seed)}


def _run_views(s):
    s["tracer"].render_views(s["frame"], _stream())
    s["frame"] += 1
    return s["films"]


def _rays(pos, idx, n, g, towards_lights, bounces):
    """Rays from points just off random triangles (bounces) or from a camera
    in front of the scene, into the scene or to points on its lights."""
    def rand(*shape):
        return torch.rand(*shape, device="cuda", generator=g)

    # the last 16 quads (32 triangles) of the field are its lights
    lights, solid = idx[-32:], idx[:-32]
    tri = solid[torch.randint(len(solid), (n,), device="cuda", generator=g)].long()
    b = rand(n, 3) + 1e-3
    b = b / b.sum(1, keepdim=True)
    at = (pos[tri] * b[:, :, None]).sum(1)
    d = torch.randn(n, 3, device="cuda", generator=g)
    rays = torch.zeros(n, 8, device="cuda")
    if towards_lights:
        tri = lights[torch.randint(len(lights), (n,), device="cuda", generator=g)].long()
        lb = rand(n, 3) + 1e-3
        to = (pos[tri] * (lb / lb.sum(1, keepdim=True))[:, :, None]).sum(1)
        org = at + 1e-4 * (to - at)
        rays[:, 0:3], rays[:, 3], rays[:, 4:7] = org, 0.999, to - org
    elif bounces:
        d = d / d.norm(dim=1, keepdim=True)
        rays[:, 0:3], rays[:, 3], rays[:, 4:7] = at + 1e-4 * d, math.inf, d
    else:
        org = torch.tensor([0.5, 0.75, 2.3], device="cuda")
        side = max(1, int(math.sqrt(n)))
        k = torch.arange(n, device="cuda")
        to = torch.stack([(k % side) / side * 1.2 - 0.1, 1.1 - (k // side) / side * 1.2, torch.zeros(n, device="cuda")], 1) + 1e-3 * rand(n, 3)
        rays[:, 0:3], rays[:, 3], rays[:, 4:7] = org, math.inf, torch.nn.functional.normalize(to - org, dim=1)
    return rays


def _ray_inputs(case, seed):
    scene = krr.Scene(_scene_config(case, seed))
    pos, idx, _ = scene.arrays()
    pos, idx = torch.from_numpy(pos).cuda(), torch.from_numpy(idx).cuda()
    g = _generator(seed)
    n = case["rays"]
    return scene, pos, idx, _rays(pos, idx, n, g, False, case.get("bounces", True)), _rays(pos, idx, n, g, True, True)


def _prepare_trace(case, seed):
    scene, _, _, rays, shadow = _ray_inputs(case, seed)
    n = case["rays"]
    return {"case": case, "scene": scene, "rays": rays, "shadow": shadow, "hits": torch.empty(n, 4, device="cuda"),
            "visible": torch.empty(n, device="cuda", dtype=torch.int32), "accel": krr.Accel(scene.desc) if case["kind"] == "trace" else None}


def _trace(s, accel):
    n, st = s["case"]["rays"], _stream()
    accel.trace_closest(s["rays"].data_ptr(), n, s["hits"].data_ptr(), st)
    accel.trace_any(s["shadow"].data_ptr(), n, s["visible"].data_ptr(), st)
    hits = s["hits"]
    return {"t": hits[:, 0], "prim": hits.view(torch.int32)[:, 1], "b1": hits[:, 2], "b2": hits[:, 3], "visible": s["visible"]}


def _run_trace(s):
    return _trace(s, s["accel"])


def _run_rebuild(s):
    if s["accel"] is not None:
        s["accel"].close()
    s["accel"] = krr.Accel(s["scene"].desc)
    info = s["accel"].info()
    return dict(_trace(s, s["accel"]), triangles=info["leaf_tris"])


def _cache_inputs(case, seed):
    """Vertex records, radiance targets and weights of a cache in use."""
    g = _generator(seed)
    n = case["samples"]
    v = torch.zeros(n, 16, device="cuda")
    v[:, :14] = torch.rand(n, 14, device="cuda", generator=g)
    glossy = (torch.rand(n, device="cuda", generator=g) < 0.3)[:, None]
    v[:, 8:11] = torch.where(glossy, 0.0, v[:, 8:11])
    v[:, 11:14] = torch.where(glossy, v[:, 11:14], 0.0)
    light = 0.5 + 0.5 * torch.sin(6.0 * v[:, 0:3]) * torch.cos(4.0 * v[:, 1:2])
    t = light * (0.2 + v[:, 8:11] + v[:, 11:14]) * torch.exp(0.5 * torch.randn(n, 3, device="cuda", generator=g))
    spread = torch.full((_abi.NRC_PARAMS,), math.sqrt(6.0 / 128.0), device="cuda")
    spread[-64 * 3:] = math.sqrt(6.0 / 67.0)
    w = (2.0 * torch.rand(_abi.NRC_PARAMS, device="cuda", generator=g) - 1.0) * spread
    return v, t.contiguous(), w


def _prepare_cache(case, seed):
    v, t, w = _cache_inputs(case, seed)
    cache = NeuralRadianceCache({"max_batch": max(1024, case["samples"])} if case["kind"] == "train" else None)
    cache.set_weights(w.cpu().numpy())
    state = {"case": case, "cache": cache, "vertices": v, "targets": t, "weights": w.cpu().numpy()}
    state["out"] = torch.empty(case["samples"], 3, device="cuda") if case["kind"] == "infer" else torch.empty(_abi.NRC_PARAMS, device="cuda")
    return state


def _run_infer(s):
    s["cache"].infer(s["vertices"].data_ptr(), s["case"]["samples"], s["out"].data_ptr(), _stream())
    return {"radiance": s["out"]}


def _run_train(s):
    cache, case = s["cache"], s["case"]
    v, t, n = s["vertices"].data_ptr(), s["targets"].data_ptr(), case["samples"]
    if not case["steps"]:  # the gradient, for an optimiser of the program's own
        return {"loss": cache.gradient(v, t, n, s["out"].data_ptr(), _stream()), "gradient": s["out"]}
    cache.set_weights(s["weights"])  # from a stored state, as when training is resumed
    losses = [cache.train_step(v, t, n, _stream()) for _ in range(case["steps"])]
    return {"losses": np.array(losses), "weights": cache.get_weights()}


# ---------------------------------------------------------------------------
# what a pass cannot do without, and how exact its results are
# ---------------------------------------------------------------------------

def _triangles(case):
    return 36 if case.get("scene") == "cornell" else case["spheres"] * 20 * 4 ** case["level"] + 34


def _ray_flops(case):
    # a 4-wide node visit per factor of two in triangles (about 60 flops) and two watertight triangle tests (about 50)
    return 60.0 * math.log2(_triangles(case)) + 100.0


def work(case):
    kind = case["kind"]
    if kind in ("infer", "train"):
        n, macs = case["samples"], 5 * 64 * 64 + 64 * 3
        if kind == "infer":
            return {"bytes": 64.0 * n + 12.0 * n + 2.0 * macs, "flops": 2.0 * macs * n}
        passes = max(1, case["steps"])
        return {"bytes": passes * (76.0 * n + 4.0 * macs), "flops": passes * 3 * 2.0 * macs * n}
    tris = _triangles(case)
    geometry = 48.0 * tris
    if kind == "trace":
        return {"bytes": geometry + case["rays"] * (2 * 32.0 + 16.0 + 4.0), "flops": 2.0 * case["rays"] * _ray_flops(case)}
    if kind == "rebuild":
        # positions, indices in, triangles and nodes out; each triangle binned once per level of the tree, about 60 flops
        return {"bytes": (24.0 + 48.0 + 64.0) * tris + case["rays"] * (2 * 32.0 + 16.0 + 4.0),
                "flops": 60.0 * tris * math.log2(tris) + 2.0 * case["rays"] * _ray_flops(case)}
    if kind == "views":
        pixels = float(sum(w * h for w, h in (_view_size(case, i) for i in range(min(case["views"], MAX_VIEWS)))))
    else:
        pixels = float(case["width"] * case["height"])
    # rays a path traces (closest and shadow), counted on these scenes, and the shading between them
    rays = {"cornell": 4.4, "volume": 5.0, "textured": 3.5}.get(case.get("scene"), 3.2)
    paths = pixels * case["spp"]
    out = 16.0 * pixels * (5 if case.get("measure") else 1)
    return {"bytes": out + geometry, "flops": paths * rays * (_ray_flops(case) + 600.0)}


def tolerance(case):
    kind = case["kind"]
    if kind == "infer":
        return {"rel": 4e-3, "max": 0.1}
    if kind == "train":
        return {"rel": 1e-2, "max": 0.3}
    if case.get("nrc"):
        # training vertices are queued in the order of atomics, so the sums of
        # a training step, and the frames after it, may differ in their rounding
        return {"rel": 2e-3, "max": 0.3}
    # the shading code takes the same decisions in the same float operations
    # whatever the launch; the framework states 1e-4 per pixel against its
    # checker, and whole numbers (primitives, visibility) are the same
    return {"rel": 1e-6, "max": 1e-4}


def exact(case, seed):
    if case["kind"] in ("infer", "train"):
        return _exact_cache(case, seed)
    if case["kind"] in ("trace", "rebuild") and case["rays"] * _triangles(case) < 4e9:
        return _exact_trace(case, seed)
    return None  # a path's decisions follow from its binary32 values: no 64-bit image is this image


def _exact_trace(case, seed):
    _, pos, idx, rays, shadow = _ray_inputs(case, seed)
    p = pos.double()[idx.long()]
    v0, e1, e2 = p[:, 0], p[:, 1] - p[:, 0], p[:, 2] - p[:, 0]
    n = len(rays)
    t = torch.full((n,), math.inf, device="cuda", dtype=torch.float64)
    b1, b2 = torch.zeros_like(t), torch.zeros_like(t)
    step = max(1, (1 << 25) // len(p))
    for i in range(0, n, step):
        o, d = rays[i:i + step, None, 0:3].double(), rays[i:i + step, None, 4:7].double()
        pv = torch.linalg.cross(d.expand(-1, len(p), -1), e2.expand(len(d), -1, -1))
        det = (pv * e1).sum(-1)
        tv = o - v0
        u = (tv * pv).sum(-1) / det
        del pv
        qv = torch.linalg.cross(tv, e1.expand(len(d), -1, -1))
        v = (d * qv).sum(-1) / det
        at = (qv * e2).sum(-1) / det
        del qv, tv
        at = torch.where((u >= 0) & (v >= 0) & (u + v <= 1) & (at > 0), at, math.inf)
        best, k = at.min(1)
        hit = torch.isfinite(best)
        t[i:i + step] = best
        b1[i:i + step] = torch.where(hit, u.gather(1, k[:, None])[:, 0], 0.0)
        b2[i:i + step] = torch.where(hit, v.gather(1, k[:, None])[:, 0], 0.0)
    return {"t": t, "prim": None, "b1": b1, "b2": b2, "visible": None, **({"triangles": None} if case["kind"] == "rebuild" else {})}


def _encode(v):
    """The 64 inputs of the network: five octaves of sin / cos of the position
    and two ones; the position, one-blob(4) of the angles and the roughness,
    the albedos, three zeros.  Slot q = 4s + j of half g is input 8s + 4g + j."""
    v = v.double()
    n = len(v)
    octaves = (2.0 ** torch.arange(5, device=v.device, dtype=torch.float64)) * math.pi
    a = v[:, 0:3, None] * octaves
    half0 = torch.cat([torch.stack([a.sin(), a.cos()], -1).reshape(n, 30), torch.ones(n, 2, device=v.device, dtype=torch.float64)], 1)
    centres = (torch.arange(4, device=v.device, dtype=torch.float64) + 0.5) / 4
    blobs = torch.exp(-0.5 * (4 * (v[:, 3:8, None] - centres)) ** 2).reshape(n, 20)
    half1 = torch.cat([v[:, 0:3], blobs, v[:, 8:14], torch.zeros(n, 3, device=v.device, dtype=torch.float64)], 1)
    return torch.stack([half0.reshape(n, 8, 4), half1.reshape(n, 8, 4)], 2).reshape(n, 64)


def _layers(w):
    return [w[4096 * i:4096 * (i + 1)].reshape(64, 64) for i in range(5)] + [w[5 * 4096:].reshape(64, 3)]


def _exact_cache(case, seed):
    v, t, w = _cache_inputs(case, seed)
    w, t = w.double(), t.double()

    def forward(x):
        xs = [x]
        for m in _layers(w)[:-1]:
            xs.append((xs[-1] @ m).clamp_min(0.0))
        return xs, xs[-1] @ _layers(w)[-1]

    if case["kind"] == "infer":
        return {"radiance": torch.cat([forward(_encode(part))[1] for part in v.split(1 << 19)])}
    x = _encode(v)
    moment, second, losses = torch.zeros_like(w), torch.zeros_like(w), []
    for step in range(1, max(1, case["steps"]) + 1):
        xs, y = forward(x)
        scale = (y * y + 0.01) * y.numel()
        losses.append(float(((y - t) ** 2 / scale).sum()))
        dz = 2.0 * (y - t) / scale
        grads = [None] * 6
        for i in range(5, -1, -1):
            grads[i] = (xs[i].T @ dz).reshape(-1)
            dz = (dz @ _layers(w)[i].T) * (xs[i] > 0)
        gradient = torch.cat(grads)
        if not case["steps"]:
            return {"loss": losses[0], "gradient": gradient}
        moment = 0.9 * moment + 0.1 * gradient
        second = 0.99 * second + 0.01 * gradient * gradient
        w = w - 1e-3 * (moment / (1 - 0.9 ** step)) / ((second / (1 - 0.99 ** step)).sqrt() + 1e-8)
    return {"losses": np.array(losses), "weights": w}
