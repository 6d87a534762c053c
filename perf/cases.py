"""What a user of the renderer has it do, as cases that can be timed and compared.

A case is a plain dict.  `prepare` makes what a program holds before a frame (models, textures,
canvases, the renderer), `run` draws once through the public entry points and returns the
canvases, `exact` gives the floating-point results in 64 bits from the same inputs, computed here
from the geometry alone.  Kinds:

  frame   renderer_begin / giveTask / end into a colour and a depth canvas, cleared by the frame.
          scene: soup (loose triangles in a cube), terrain (textured height field), objects (many
          instances of one box model with diffuse and light map over a ground), alpha (a terrain
          behind translucent triangles), all under a perspective camera unless ortho is set.
  depth   model_renderDepth of a terrain into a depth canvas the caller clears.
  batch   dfpsr_hip_batch_render of uneven jobs.
  fit     one differentiable step: forward of all views, adjoint into texture (and multipliers).
"""
from __future__ import annotations

import copy
import math

import numpy as np
import torch

from dfpsr_amd import _lib, api, scenes

TILE = {"16x16": 0, "32x16": 1, "32x32": 2}


def listed():
    return [
        # The smallest call: a thumbnail of a hundred triangles with the renderer's default tuning.
        # Latency and launches are all there is.
        {"name": "thumbnail", "kind": "frame", "scene": "soup", "width": 64, "height": 48, "size": 100, "texture": 0, "tile": "16x16",
         "host": False, "ortho": False},
        # A program of the reference that swapped its renderer: 2,000 vertex-coloured triangles into
        # 640x480 images in host memory, copied up and down by the frame.
        {"name": "soup_host", "kind": "frame", "scene": "soup", "width": 640, "height": 480, "size": 2000, "texture": 0, "tile": "16x16",
         "host": True, "ortho": False},
        # The headline frame: 1080p terrain of 256x256 points with a 1024^2 texture.
        {"name": "terrain_1080p", "kind": "frame", "scene": "terrain", "width": 1920, "height": 1080, "size": 256, "texture": 1024,
         "light": False, "tile": "32x16", "host": False, "ortho": False},
        # A window of any size: odd width and height, a grid that fills no block evenly, light map on.
        {"name": "window_odd", "kind": "frame", "scene": "terrain", "width": 1365, "height": 767, "size": 151, "texture": 512,
         "light": True, "tile": "32x16", "host": False, "ortho": False},
        # The largest frame: 4K, half a million triangles, a 2048^2 texture.
        {"name": "terrain_4k", "kind": "frame", "scene": "terrain", "width": 3840, "height": 2160, "size": 512, "texture": 2048,
         "light": False, "tile": "32x16", "host": False, "ortho": False},
        # A game level: 200 instances of a box model (one task each) over a ground, diffuse and light.
        {"name": "objects_720p", "kind": "frame", "scene": "objects", "width": 1280, "height": 720, "size": 200, "texture": 256,
         "tile": "32x16", "host": False, "ortho": False},
        # Glass, smoke, leaves: 1,500 translucent triangles (Filter::Alpha) in front of a terrain.
        {"name": "alpha_720p", "kind": "frame", "scene": "alpha", "width": 1280, "height": 720, "size": 1500, "texture": 256,
         "tile": "32x16", "host": False, "ortho": False},
        # The isometric view of a strategy game: an orthogonal camera over a terrain.
        {"name": "ortho_720p", "kind": "frame", "scene": "terrain", "width": 1280, "height": 720, "size": 192, "texture": 512,
         "light": False, "tile": "32x16", "host": False, "ortho": True},
        # Shadow maps and picking: the terrain's depth alone at 1080p.
        {"name": "depth_1080p", "kind": "depth", "width": 1920, "height": 1080, "size": 256, "ortho": False},
        # Data generation: 384 uneven jobs in one call, as the autotuner sets it.
        {"name": "batch_384", "kind": "batch", "jobs": 384, "layout": 2, "max_triangles": 20000},
        # Fitting a texture and per-point colours to eight 720p views of a 50,000-triangle surface.
        {"name": "fit_8_views", "kind": "fit", "views": 8, "width": 1280, "height": 720, "frequency": 50, "texture": 512,
         "multipliers": True, "tile": "32x16"},
        # Fitting a texture to many small views: 96 of 256x256, a 1024^2 texture.
        {"name": "fit_96_views", "kind": "fit", "views": 96, "width": 256, "height": 256, "frequency": 32, "texture": 1024,
         "multipliers": False, "tile": "16x16"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["soup", "terrain", "terrain", "terrain", "objects", "alpha", "depth", "batch", "fit"])
    width, height = _log(rng, 64, 3840), 0
    height = max(40, min(2160, int(width * rng.uniform(0.5, 0.8))))
    tile = rng.choice(sorted(TILE))
    if kind == "batch":
        return {"kind": "batch", "jobs": _log(rng, 8, 300), "layout": rng.randint(3, 1000), "max_triangles": _log(rng, 1000, 20000)}
    if kind == "fit":
        views = _log(rng, 1, 64)
        width = min(_log(rng, 96, 1280), int(math.sqrt(5e6 / views)))
        return {"kind": "fit", "views": views, "width": width, "height": max(64, int(width * rng.uniform(0.55, 1.0))),
                "frequency": rng.randint(6, 50), "texture": rng.choice([128, 256, 512, 1024]), "multipliers": rng.random() < 0.5,
                "tile": rng.choice(["16x16", "32x16"])}
    if kind == "depth":
        return {"kind": "depth", "width": width, "height": height, "size": rng.randint(20, 300), "ortho": rng.random() < 0.3}
    case = {"kind": "frame", "scene": kind, "width": width, "height": height, "tile": tile, "host": rng.random() < 0.1, "ortho": False}
    if kind == "soup":
        case.update(size=_log(rng, 50, 20000), texture=rng.choice([0, 0, 128, 256]))
    elif kind == "terrain":
        case.update(size=rng.randint(20, 400), texture=rng.choice([128, 256, 512, 1024]), light=rng.random() < 0.3, ortho=rng.random() < 0.25)
    elif kind == "objects":
        case.update(size=rng.randint(10, 250), texture=rng.choice([64, 128, 256]))
    else:
        case.update(size=_log(rng, 50, 1500), texture=rng.choice([128, 256]))
    return case


# ---------------------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------------------

def _terrain(case, seed):
    sc = scenes.terrain(width=case["width"], height=case["height"], grid=case["size"], seed=seed % 100003,
                        texture_size=case.get("texture") or 64, resolutions=(case.get("texture") or 64).bit_length(),
                        uv_repeat=4.0 * case["size"] / 256)
    if case["size"] < 256:  # the same slope of the view whatever the grid's size
        half, scale = (case["size"] - 1) / 2.0, case["size"] / 256.0
        sc.cam_location = scenes.look_transform((0.0, 30.0 * scale + 8.0, -half - 10.0 * scale), 0.0, math.radians(35.0))
    if case.get("light"):
        sc.textures.append(scenes.noise_checker_texture(128, seed % 100003 + 5, 1, check=8))
        sc.texcoords[:, :, 2:4] = sc.texcoords[:, :, 0:2] * np.float32(0.25)
        sc.parts[0].light = 1
    if case.get("ortho"):
        half = (case["size"] - 1) / 2.0
        sc.perspective = False
        sc.cam_location = scenes.look_transform((-0.6 * half, 0.9 * half, -0.6 * half), math.radians(45.0), math.radians(45.0))
        sc.width_slope = float(np.float32(0.45 * half))
    return sc


def _box(side, seed):
    """A unit box of 6 x side x side quads wound to face outwards, uv per face, light uv over the face."""
    pts, quads, tex = [], [], []
    g = np.linspace(-1.0, 1.0, side + 1)
    for axis in range(3):
        for sign in (-1.0, 1.0):
            base = len(pts)
            for v in g:
                for u in g:
                    p = [0.0, 0.0, 0.0]
                    p[axis], p[(axis + 1) % 3], p[(axis + 2) % 3] = sign, u, v
                    pts.append(p)
            for j in range(side):
                for i in range(side):
                    a = base + j * (side + 1) + i
                    q = [a, a + 1, a + side + 2, a + side + 1] if sign > 0 else [a, a + side + 1, a + side + 2, a + 1]
                    quads.append(q)
                    local = [(k - base) for k in q]
                    tex.append([[(k % (side + 1)) / side, (k // (side + 1)) / side] * 2 for k in local])
    shade = scenes.Rng(seed).uniform(len(quads) * 4, 0.5, 1.0).reshape(len(quads), 4, 1)
    colors = np.ones((len(quads), 4, 4), np.float32)
    colors[:, :, :3] = shade
    return np.array(pts, np.float32), np.array(quads, np.int32), colors, np.array(tex, np.float32)


def _scenes_of(case, seed):
    """The scenes whose models one frame draws in turn (all under the first one's camera)."""
    s = seed % 100003
    if case["scene"] == "soup":
        sc = scenes.cube_soup(width=case["width"], height=case["height"], triangles=case["size"], seed=seed)
        if case["texture"]:
            sc.texcoords[:, :3, :2] = scenes.Rng(seed + 77).uniform(case["size"] * 6, -1.0, 2.0).reshape(-1, 3, 2)
            sc.textures = [scenes.noise_checker_texture(case["texture"], s, case["texture"].bit_length(), check=16)]
            sc.parts = [scenes.Part(0, case["size"], diffuse=0)]
        return [sc]
    if case["scene"] == "terrain":
        return [_terrain(case, seed)]
    if case["scene"] == "objects":
        ground = _terrain({**case, "size": 64, "light": False}, seed)
        pts, quads, colors, tex = _box(4, s + 3)
        rng = scenes.Rng(seed + 11)
        place = rng.uniform(case["size"] * 3, -1.0, 1.0).reshape(-1, 3)
        yaw = rng.uniform(case["size"], 0.0, 2.0 * math.pi)
        inst = np.zeros((case["size"], 12), np.float32)
        for i in range(case["size"]):
            c, n, k = math.cos(yaw[i]), math.sin(yaw[i]), 0.5 + 0.5 * abs(float(place[i, 1]))
            inst[i] = [place[i, 0] * 28, 3.0 + 6.0 * place[i, 1], place[i, 2] * 28, c * k, 0, -n * k, 0, k, 0, n * k, 0, c * k]
        boxes = copy.copy(ground)
        boxes.points, boxes.indices, boxes.colors, boxes.texcoords, boxes.instances = pts, quads, colors, tex, inst
        boxes.textures = [scenes.noise_checker_texture(case["texture"], s + 7, case["texture"].bit_length(), check=16),
                          scenes.noise_checker_texture(64, s + 9, 1, check=8)]
        boxes.parts = [scenes.Part(0, quads.shape[0], diffuse=0, light=1)]
        return [ground, boxes]
    ground = _terrain({**case, "size": 96, "light": False}, seed)
    soup = scenes.cube_soup(width=case["width"], height=case["height"], triangles=case["size"], seed=seed, alpha=0.5)
    glass = copy.copy(ground)
    glass.points = (soup.points * np.float32(18.0) + np.array([0.0, 8.0, -14.0], np.float32)).astype(np.float32)
    glass.indices, glass.colors, glass.texcoords = soup.indices, soup.colors, soup.texcoords
    glass.textures, glass.parts, glass.filter = [], [scenes.Part(0, case["size"])], api.Filter_Alpha
    return [ground, glass]


class _State:
    pass


def _far(case):
    return float("inf") if case.get("ortho") else 0.0


def _fit_inputs(case, seed):
    views = scenes.sphere_views(case["frequency"], case["views"], case["width"], case["height"], seed=seed % 100003)
    g = torch.Generator().manual_seed(seed)
    tex = torch.from_numpy(scenes.float_texture(case["texture"], seed % 100003, smooth=16))
    mul = torch.rand((views[0].points.shape[0], 3), generator=g) + 0.5 if case["multipliers"] else None
    return views, tex, mul


def _jobs(case, seed):
    """The jobs of one layout (canvas sizes, triangle counts), each object turned and recoloured by the seed."""
    jobs = scenes.batch_jobs(case["jobs"], seed=case["layout"], max_tris=case["max_triangles"])
    rng = scenes.Rng(seed)
    for sc, turn, shade in zip(jobs, rng.uniform(len(jobs), 0.0, 2.0 * math.pi), rng.uniform(len(jobs), 0.6, 1.0)):
        c, n = math.cos(turn), math.sin(turn)
        sc.instances = np.array([[0, 0, 0, c, 0, -n, 0, 1, 0, n, 0, c]], np.float32)
        sc.colors[..., :3] *= shade
    return jobs


def _grad_image(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed + 1)
    return torch.randn((case["views"], case["height"], case["width"], 4), generator=g, device="cuda") * 1e-3


def prepare(case, seed):
    s = _State()
    s.case = case
    h, w = case.get("height", 0), case.get("width", 0)
    if case["kind"] == "frame":
        s.gpu = [api.GpuScene(sc) for sc in _scenes_of(case, seed)]
        for g in s.gpu[1:]:
            g.camera = s.gpu[0].camera
        s.renderer = api.renderer_create()
        api.renderer_setTuning(s.renderer, api.tuning(tile_config=TILE[case["tile"]], clear=True, clear_depth=_far(case)))
        if case["host"]:
            s.color, s.depth = np.zeros((h, w), np.uint32), np.zeros((h, w), np.float32)
            s.images = api.host_image(s.color), api.host_image(s.depth)
        else:
            s.color = torch.zeros((h, w), dtype=torch.int32, device="cuda")
            s.depth = torch.zeros((h, w), dtype=torch.float32, device="cuda")
            s.images = api.device_image(s.color), api.device_image(s.depth)
    elif case["kind"] == "depth":
        s.gpu = api.GpuScene(_terrain(case, seed))
        s.depth = torch.zeros((h, w), dtype=torch.float32, device="cuda")
        s.image = api.device_image(s.depth)
    elif case["kind"] == "batch":
        jobs = _jobs(case, seed)
        s.jobs = api.GpuJobs(jobs)
        # One allocation for all canvases, as a program that hands the images on keeps them.
        ends = np.cumsum([0] + [j.width * j.height for j in jobs])
        s.color = torch.zeros(int(ends[-1]), dtype=torch.int32, device="cuda")
        s.depth = torch.zeros(int(ends[-1]), dtype=torch.float32, device="cuda")
        for i, j in enumerate(jobs):
            a, b = int(ends[i]), int(ends[i + 1])
            s.jobs.jobs[i].color = api.device_image(s.color[a:b].view(j.height, j.width))
            s.jobs.jobs[i].depth = api.device_image(s.depth[a:b].view(j.height, j.width))
        s.jobs.colors, s.jobs.depths = [], []
        s.batch = api.Batch()
        s.tuning = api.tuning(tile_config=1, persistent_per_cu=8, use_graph=True, clear=True)
    else:
        views, tex, mul = _fit_inputs(case, seed)
        s.model = api.model_create(0)
        api.model_setPoints(s.model, views[0].points)
        api.model_addPart(s.model, views[0].indices, views[0].colors, views[0].texcoords)
        n = case["views"]
        s.color = torch.zeros((n, h, w, 4), device="cuda")
        s.visibility = torch.full((n, h, w), -1, dtype=torch.int32, device="cuda")
        s.depth = torch.zeros((n, h, w), device="cuda")
        s.grad = _grad_image(case, seed)
        s.views = (_lib.View * n)()
        for i, sc in enumerate(views):
            v = s.views[i]
            v.color, v.visibility = s.color[i].data_ptr(), s.visibility[i].data_ptr()
            v.depth, v.grad_color = s.depth[i].data_ptr(), s.grad[i].data_ptr()
            v.width, v.height, v.stride_pixels = w, h, w
            v.transform[:] = [float(x) for x in sc.instances[0]]
            v.camera = api.camera_create(True, sc.cam_location, w, h, sc.width_slope, sc.near_clip, sc.far_clip)
        s.texture = tex.cuda()
        s.multipliers = mul.cuda() if mul is not None else None
        s.grad_texture = torch.zeros_like(s.texture)
        s.grad_multipliers = torch.zeros_like(s.multipliers) if mul is not None else None
        s.diff = api.DiffRenderer()
        tile = TILE[case["tile"]]
        s.forward = api.tuning(clear=True, tile_config=tile, use_graph=True)
        s.backward = api.tuning(tile_config=tile, persistent_per_cu=4, use_graph=True)
    return s


def run(s):
    kind = s.case["kind"]
    if kind == "frame":
        api.renderer_begin(s.renderer, *s.images)
        for g in s.gpu:
            g.give(s.renderer)
        api.renderer_end(s.renderer)
        return {"color": s.color, "depth": s.depth}
    if kind == "depth":
        s.depth.fill_(_far(s.case))
        api.model_renderDepth(s.gpu.model, s.gpu.scene.instances[0], s.image, s.gpu.camera)
        return {"depth": s.depth}
    if kind == "batch":
        s.batch.render(s.jobs.jobs, s.tuning)
        return {"color": s.color, "depth": s.depth}
    s.diff.forward(s.model, s.views, s.texture, s.multipliers, s.forward)
    s.grad_texture.zero_()
    if s.grad_multipliers is not None:
        s.grad_multipliers.zero_()
    s.diff.backward(s.grad_texture, s.grad_multipliers, s.backward)
    out = {"color": s.color, "depth": s.depth, "visibility": s.visibility, "grad_texture": s.grad_texture}
    if s.grad_multipliers is not None:
        out["grad_multipliers"] = s.grad_multipliers
    return out


# ---------------------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------------------

def work(case):
    """Bytes: canvases written once, texels of the sampled levels, 12 per point, 84 per triangle.
    Operations: about 120 per triangle (projection, planes) and 60 per shaded pixel."""
    px = case.get("width", 0) * case.get("height", 0)
    texels = (case.get("texture") or 0) ** 2 * 4 // 3
    n = case.get("size", 0)
    if case["kind"] == "batch":
        # Canvases average 352 x 264 pixels; triangle counts are log-uniform from 100 up.
        m = case["max_triangles"]
        tris = int(case["jobs"] * (m - 100) / math.log(m / 100))
        px = case["jobs"] * 352 * 264
        return {"bytes": 8 * px + 16 * 4 * 65536 * 4 // 3 + 100 * tris, "flops": 120 * tris + 60 * px}
    if case["kind"] == "fit":
        px *= case["views"]
        tris = 20 * case["frequency"] ** 2
        # Forward writes colour, depth and id; the adjoint reads the gradient and the id.
        return {"bytes": (24 + 20) * px + 2 * 16 * case["texture"] ** 2 + 60 * tris,
                "flops": 120 * tris * case["views"] + 100 * px}
    if case["kind"] == "depth":
        tris = 2 * (n - 1) ** 2
        return {"bytes": 4 * px + 12 * n * n + 16 * tris, "flops": 120 * tris + 4 * px}
    tris = {"soup": n, "terrain": 2 * (n - 1) ** 2, "objects": n * 192 + 2 * 63 ** 2, "alpha": n + 2 * 95 ** 2}[case["scene"]]
    stored = 192 + 2 * 63 ** 2 if case["scene"] == "objects" else tris
    return {"bytes": (16 if case["host"] else 8) * px + 4 * texels + 96 * stored, "flops": 120 * tris + 60 * px}


# ---------------------------------------------------------------------------------------
# The same results in 64 bits
# ---------------------------------------------------------------------------------------

def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _camera_space(points, transform, location, real):
    t, c = transform.to(real), location.to(real)
    p = points.to(real)
    w = ((p[:, 0:1] * t[3:6] + p[:, 1:2] * t[6:9]) + p[:, 2:3] * t[9:12]) + t[0:3]
    d = w - c[0:3]
    return torch.stack([(d[:, 0] * c[3 * k] + d[:, 1] * c[3 * k + 1]) + d[:, 2] * c[3 * k + 2] for k in (1, 2, 3)], 1)


def _screen(cs, sc, real):
    w, h = (torch.tensor(float(v), dtype=real, device=cs.device) for v in (sc.width, sc.height))
    slope = torch.tensor(float(sc.width_slope), dtype=torch.float32, device=cs.device).to(real)
    sx, sy = 0.5 / slope, 0.5 / (slope * h / w)
    x, y, z = cs.unbind(1)
    if not sc.perspective:
        return torch.stack([(x * sx + 0.5) * w, (-y * sy + 0.5) * h], 1)
    inv = 1.0 / z
    mid = z * 0.5
    return torch.stack([((x * sx + mid) * w) * inv, ((-y * sy + mid) * h) * inv], 1)


def _fragments(sc, instances):
    """The pixels that the scene's triangles cover (from corners rounded to 1/256 pixel, whole-number
    arithmetic), with their corner weights and depth in 64 bits: one dict of flat tensors, in drawing
    order; None when a visible triangle reaches the near or far plane."""
    dev = _device()
    idx = torch.from_numpy(sc.indices).to(dev).long()
    fan = torch.stack([torch.cat([idx[:, :3], torch.arange(len(idx), device=dev)[:, None], torch.zeros_like(idx[:, :1])], 1),
                       torch.cat([idx[:, [0, 2, 3]], torch.arange(len(idx), device=dev)[:, None], torch.ones_like(idx[:, :1])], 1)], 1)
    fan = fan.reshape(-1, 5)[torch.stack([torch.ones(len(idx), dtype=torch.bool, device=dev), idx[:, 3] >= 0], 1).reshape(-1)]
    points, location = torch.from_numpy(sc.points).to(dev), torch.from_numpy(np.asarray(sc.cam_location, np.float32)).to(dev)
    found = []
    for t in instances:
        t = torch.from_numpy(np.asarray(t, np.float32)).to(dev)
        cs = _camera_space(points, t, location, torch.float64)
        scr = _screen(cs, sc, torch.float64)
        rounded = _screen(_camera_space(points, t, location, torch.float32), sc, torch.float32)
        z = cs[:, 2][fan[:, :3]]
        p, q = scr[fan[:, :3]], rounded[fan[:, :3]]
        if sc.perspective:
            slope_x, slope_y = sc.width_slope, sc.width_slope * sc.height / sc.width
            corner = cs[fan[:, :3]]
            outside = ((z <= sc.near_clip).all(1) | (z >= sc.far_clip).all(1)
                       | (corner[..., 0] < -slope_x * z).all(1) | (corner[..., 0] > slope_x * z).all(1)
                       | (corner[..., 1] < -slope_y * z).all(1) | (corner[..., 1] > slope_y * z).all(1))
            if bool((((z <= sc.near_clip) | (z >= sc.far_clip)).any(1) & ~outside).any()):
                return None
        else:
            outside = ((p[..., 0] < 0).all(1) | (p[..., 0] > sc.width).all(1) | (p[..., 1] < 0).all(1) | (p[..., 1] > sc.height).all(1))
        f = torch.where(outside[:, None, None], torch.zeros_like(q), q * 256.0).trunc().long()
        a, b, c = f.unbind(1)
        front = ((c[:, 0] - a[:, 0]) * (b[:, 1] - a[:, 1]) + (c[:, 1] - a[:, 1]) * (a[:, 0] - b[:, 0])) < 0
        keep = torch.nonzero(front & ~outside).reshape(-1)
        f, p, z, tri = f[keep], p[keep], z[keep], fan[keep]
        if not len(keep):
            continue
        top = ((f[..., 1].amin(1) + 128).div(256, rounding_mode="trunc") - 1).clamp(min=0)
        bottom = ((f[..., 1].amax(1) + 128).div(256, rounding_mode="trunc") + 1).clamp(max=sc.height)
        x0 = ((f[..., 0].amin(1) + 128).div(256, rounding_mode="trunc") - 1).clamp(min=0)
        x1 = ((f[..., 0].amax(1) + 128).div(256, rounding_mode="trunc") + 1).clamp(max=sc.width)
        rows = (bottom - top).clamp(min=0) * (x1 > x0)
        r = torch.repeat_interleave(torch.arange(len(f), device=dev), rows)
        y = top[r] + torch.arange(len(r), device=dev) - (torch.cumsum(rows, 0) - rows)[r]
        left, right = x0[r], x1[r]
        for k in range(3):
            s, e = f[:, k][r], f[:, (k + 1) % 3][r]
            nx, ny = e[:, 1] - s[:, 1], s[:, 0] - e[:, 0]
            limit = torch.where((s[:, 0] > e[:, 0]) | ((s[:, 0] == e[:, 0]) & (s[:, 1] > e[:, 1])), -1, 0)
            value = (128 - s[:, 0]) * nx + (256 * y + 128 - s[:, 1]) * ny
            by = torch.where(nx == 0, 1, 256 * nx)
            right = torch.where(nx > 0, torch.minimum(right, (limit - value).div(by, rounding_mode="trunc") + 1), right)
            left = torch.where(nx < 0, torch.maximum(left, (limit - value + 1).div(by, rounding_mode="trunc") + 1), left)
            right = torch.where((nx == 0) & (ny != 0) & (value > limit), left, right)
        n = (right - left).clamp(min=0)
        i = torch.repeat_interleave(torch.arange(len(r), device=dev), n)
        x = left[i] + torch.arange(len(i), device=dev) - (torch.cumsum(n, 0) - n)[i]
        y, r = y[i], r[i]
        # Corner weights on the screen, then through 1 / z.
        px, py = x.double() + 0.5, y.double() + 0.5
        A, B, C = p.unbind(1)
        area = (B[:, 0] - A[:, 0]) * (C[:, 1] - A[:, 1]) - (B[:, 1] - A[:, 1]) * (C[:, 0] - A[:, 0])
        wb = ((px - A[r, 0]) * (C[r, 1] - A[r, 1]) - (py - A[r, 1]) * (C[r, 0] - A[r, 0])) / area[r]
        wc = ((B[r, 0] - A[r, 0]) * (py - A[r, 1]) - (B[r, 1] - A[r, 1]) * (px - A[r, 0])) / area[r]
        wa = 1.0 - wb - wc
        zi = 1.0 / z[r] if sc.perspective else z[r]
        depth = wa * zi[:, 0] + wb * zi[:, 1] + wc * zi[:, 2]
        if sc.perspective:
            wb, wc = wb * zi[:, 1] / depth, wc * zi[:, 2] / depth
        found.append({"pixel": y * sc.width + x, "depth": depth, "wb": wb, "wc": wc, "triangle": tri[r]})
    if not found:
        return {"pixel": torch.zeros(0, dtype=torch.long, device=dev), "depth": torch.zeros(0, dtype=torch.float64, device=dev)}
    return {k: torch.cat([f[k] for f in found]) for k in found[0]}


def _depth_image(sc, parts, far):
    image = torch.full((sc.height * sc.width,), float(far), dtype=torch.float64, device=_device())
    for f in parts:
        image.scatter_reduce_(0, f["pixel"], f["depth"], "amax" if sc.perspective else "amin")
    return image


def _exact_fit(case, seed):
    views, tex, mul = _fit_inputs(case, seed)
    dev, size = _device(), case["texture"]
    tex = tex.to(dev).double().reshape(-1, 4)
    mul = mul.to(dev).double() if mul is not None else None
    grad = _grad_image(case, seed).double()
    out = {"color": torch.zeros((len(views), case["height"], case["width"], 4), dtype=torch.float64, device=dev),
           "depth": torch.zeros((len(views), case["height"], case["width"]), dtype=torch.float64, device=dev), "visibility": None,
           "grad_texture": torch.zeros_like(tex)}
    if mul is not None:
        out["grad_multipliers"] = torch.zeros_like(mul)
    for i, sc in enumerate(views):
        f = _fragments(sc, sc.instances)
        if f is None:
            return None
        depth = _depth_image(sc, [f], 0.0)
        out["depth"][i] = depth.reshape(sc.height, sc.width)
        order = torch.arange(len(f["pixel"]), device=dev)
        first = torch.full((sc.height * sc.width,), len(order), dtype=torch.long, device=dev)
        best = f["depth"] == depth[f["pixel"]]
        first.scatter_reduce_(0, f["pixel"][best], order[best], "amin")
        won = torch.nonzero(best & (first[f["pixel"]] == order)).reshape(-1)
        px, wb, wc, tri = f["pixel"][won], f["wb"][won], f["wc"][won], f["triangle"][won]
        w = torch.stack([1.0 - wb - wc, wb, wc], 1)
        corner = torch.stack([torch.zeros_like(tri[:, 4]), 1 + tri[:, 4], 2 + tri[:, 4]], 1)
        uv = torch.from_numpy(sc.texcoords).to(dev).double()[tri[:, 3:4], corner][..., :2]
        uv = (uv * w[..., None]).sum(1)
        sub = ((uv + 256.0) * (256 * size)).trunc().long() - 128
        part = (sub & 255).double() / 256.0
        at = (sub >> 8) & (size - 1)
        nxt = (at + 1) & (size - 1)
        taps = [(at[:, 1], at[:, 0], (1 - part[:, 0]) * (1 - part[:, 1])), (at[:, 1], nxt[:, 0], part[:, 0] * (1 - part[:, 1])),
                (nxt[:, 1], at[:, 0], (1 - part[:, 0]) * part[:, 1]), (nxt[:, 1], nxt[:, 0], part[:, 0] * part[:, 1])]
        sample = sum(k[:, None] * tex[ty * size + tx] for ty, tx, k in taps)
        m = (mul[tri[:, :3]] * w[..., None]).sum(1) if mul is not None else torch.ones_like(sample[:, :3])
        out["color"][i].view(-1, 4)[px] = torch.cat([sample[:, :3] * m, sample[:, 3:]], 1)
        g = grad[i].reshape(-1, 4)[px]
        gt = torch.cat([g[:, :3] * m, g[:, 3:]], 1)
        for ty, tx, k in taps:
            out["grad_texture"].index_add_(0, ty * size + tx, gt * k[:, None])
        if mul is not None:
            for k in range(3):
                out["grad_multipliers"].index_add_(0, tri[:, k], g[:, :3] * sample[:, :3] * w[:, k:k + 1])
    out["grad_texture"] = out["grad_texture"].reshape(size, size, 4)
    return out


def exact(case, seed):
    if case["kind"] == "fit":
        return _exact_fit(case, seed)
    if case["kind"] == "batch":
        images = []
        for sc in _jobs(case, seed):
            f = _fragments(sc, sc.instances)
            if f is None:
                return None
            images.append(_depth_image(sc, [f], 0.0))
        return {"color": None, "depth": torch.cat(images)}
    every = [_terrain(case, seed)] if case["kind"] == "depth" else _scenes_of(case, seed)
    parts = []
    for sc in every:
        if sc.filter == api.Filter_Alpha:  # translucent triangles leave the depth as it is
            continue
        f = _fragments(sc, sc.instances)
        if f is None:
            return None
        parts.append(f)
    depth = _depth_image(every[0], parts, _far(case)).reshape(every[0].height, every[0].width)
    if case["kind"] == "depth":
        return {"depth": depth}
    return {"color": None, "depth": depth.cpu().numpy() if case["host"] else depth}
