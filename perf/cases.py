"""Performance cases of the probe-update engine: the calls a renderer makes per frame.

A case is a dict with a ``kind`` and its sizes:

* ``update``    one frame of a probe grid: optionally the scene's instances move (LBVH refit
                or rebuild) and the atlas follows the camera, then ``ProbeGrid.update`` of one
                probe layer (the reference renderer's schedule) or of the whole grid
* ``convolve``  ``ProbeGrid.convolve`` over radiance the program set itself
* ``gi``        the deferred GI lookup of a G-buffer
* ``mask``      RT hard shadows of a depth buffer
* ``mirror``    mirror reflections of a depth and normal buffer
* ``lights``    point-light shadow moments
* ``rays``      closest or any hits of the program's own device-resident rays

The screen-space passes and ray queries go through the C-ABI on device pointers, as a
renderer with its buffers in HBM calls them.
"""
import ctypes
import math

import numpy as np
import torch

from anerend_amd import native, scenegen
from anerend_amd.types import FLAG_BAKE, Config

FP32, BF16, FP8, FP16 = 0, 1, 2, 3
FRAMES = 24  # frames a state prepares; passes walk over them in turn


def _update(name=None, family="terrain", boxes=0, cells=0, instances=0, subdiv=1, grid=(8, 8, 8), rays=256,
            precision=FP32, layers=0, sun="static", motion="none"):
    c = {"kind": "update", "family": family, "boxes": boxes, "cells": cells, "instances": instances,
         "subdiv": subdiv, "nx": grid[0], "ny": grid[1], "nz": grid[2], "rays": rays, "precision": precision,
         "layers": layers, "sun": sun, "motion": motion}
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest call: one probe layer (64 probes) of the 780-triangle room per frame
        _update("room_layer", family="room", boxes=64, grid=(8, 8, 8), rays=256, layers=1),
        # the whole room grid, 131k rays
        _update("room_update", family="room", boxes=64, grid=(8, 8, 8), rays=256),
        # the reference's schedule on the production grid: one of its 16 layers per frame
        _update("terrain_layer", cells=512, instances=10000, grid=(32, 16, 32), rays=512, layers=1),
        # the production update: 16,384 probes x 512 rays over 984k triangles, a static sun
        _update("terrain_update", cells=512, instances=10000, grid=(32, 16, 32), rays=512),
        # the same scene under a sun that moves with every frame, 16-bit radiance
        _update("terrain_sun", cells=512, instances=10000, grid=(32, 16, 32), rays=512, precision=FP16, sun="moving"),
        # instances move and the hierarchy is rebuilt each frame (the reference's TLAS build), then one layer
        _update("town_rebuild", cells=256, instances=2501, grid=(16, 8, 16), rays=256, precision=BF16, layers=1,
                motion="rebuild"),
        # the largest: 4.04M triangles of which 20,000 instances move, refits with a rebuild every 4
        # frames, a following camera and a full FP8 update of 131,072 probes x 256 rays
        _update("dynamic_frame", cells=600, instances=20000, subdiv=2, grid=(64, 32, 64), rays=256, precision=FP8,
                motion="refit"),
        # the convolution alone, production shape
        {"name": "convolve", "kind": "convolve", "nx": 32, "ny": 16, "nz": 32, "rays": 512, "precision": FP32},
        # screen-space passes of a full-HD frame
        {"name": "gi_1080p", "kind": "gi", "nx": 32, "ny": 16, "nz": 32, "width": 1920, "height": 1080},
        {"name": "mask_1080p", "kind": "mask", "cells": 512, "instances": 10000, "width": 1920, "height": 1080},
        {"name": "mirror_1080p", "kind": "mirror", "cells": 512, "instances": 10000, "nx": 32, "ny": 16, "nz": 32,
         "width": 1920, "height": 1080},
        # an ordinary number of point lights around the camera
        {"name": "lights_64", "kind": "lights", "cells": 512, "instances": 10000, "lights": 64},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["update"] * 6 + ["convolve", "gi", "mask", "mirror", "lights", "rays"])
    cells = _log(rng, 48, 700)
    world = {"cells": cells, "instances": _log(rng, 1, 12000)}
    grid = (rng.randint(3, 32), rng.randint(2, 16), rng.randint(3, 32))
    image = {"width": _log(rng, 160, 2560), "height": _log(rng, 90, 1440)}
    if kind == "update":
        room = rng.random() < 0.25
        precision = rng.choice([FP32, FP32, BF16, FP16, FP8])
        # whole multiples of 32 for the matrix formats, any count in FP32
        rays = 32 * rng.randint(1, 20) if precision != FP32 or rng.random() < 0.6 else rng.randint(16, 700)
        layers = rng.choice([0, 1, rng.randint(1, grid[1])])
        motion = rng.choice(["none", "none", "refit", "rebuild"])
        sun = rng.choice(["static", "static", "moving"])
        if room:
            return _update(family="room", boxes=_log(rng, 1, 400), grid=grid, rays=rays, precision=precision,
                           layers=layers, sun=sun)
        return _update(grid=grid, rays=rays, precision=precision, layers=layers, sun=sun, motion=motion, **world)
    if kind == "convolve":
        precision = rng.choice([FP32, BF16, FP16, FP8])
        rays = 32 * rng.randint(1, 24) if precision != FP32 or rng.random() < 0.6 else rng.randint(16, 700)
        return {"kind": kind, "nx": grid[0], "ny": grid[1], "nz": grid[2], "rays": rays, "precision": precision}
    if kind == "gi":
        return {"kind": kind, "nx": grid[0], "ny": grid[1], "nz": grid[2], **image}
    if kind == "mask":
        return {"kind": kind, **world, **image}
    if kind == "mirror":
        return {"kind": kind, **world, "nx": grid[0], "ny": grid[1], "nz": grid[2], **image}
    if kind == "lights":
        return {"kind": kind, **world, "lights": _log(rng, 1, 1024)}
    return {"kind": "rays", **world, "count": _log(rng, 1000, 3000000), "any": rng.random() < 0.5}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _triangles(c):
    if c.get("family") == "room":
        return 12 * (1 + c["boxes"])
    n = c["instances"]
    return 2 * c["cells"] ** 2 + 12 * ((n + 1) // 2) + 20 * 4 ** c.get("subdiv", 1) * (n // 2)


def _scene(c, seed):
    if c.get("family") == "room":
        return scenegen.room_scene(1 + seed, num_boxes=c["boxes"])
    spread = min(60.0, c["cells"] / 2.0 - 4.0) if c.get("motion", "none") != "none" else None
    return scenegen.terrain_scene(2 + seed, cells=c["cells"], num_instances=c["instances"],
                                  ico_subdiv=c.get("subdiv", 1), spread=spread)


def _config(c):
    step = (1.0, 1.0, 1.0) if c.get("family") == "room" else (1.0, 2.0, 1.0)
    return Config.make((c["nx"], c["ny"], c["nz"]), step=step, rays=c.get("rays", 256), hysteresis=0.96,
                       precision=c.get("precision", FP32))


def _layer_range(c, k):
    """Probe layers of frame k: a window that walks over the grid, or all of them."""
    n = c["layers"] or c["ny"]
    return (k * n) % (c["ny"] - n + 1 if n > 1 else c["ny"]), n


def _frame(c, seed, cfg, k):
    height = 1.5 if c.get("family") == "room" else 12.0
    x = 0.5
    if c.get("motion", "none") != "none":  # there and back, a cell every third frame
        x += (k if k < FRAMES // 2 else FRAMES - k) / 3.0
    f = scenegen.make_frame(1 + seed, camera=(x, height, 0.5), config=cfg, iteration=k)
    if c.get("sun") == "moving":
        a = 0.01 * k
        lx, _, lz = f.light_dir[0], f.light_dir[1], f.light_dir[2]
        f.light_dir[0] = lx * math.cos(a) - lz * math.sin(a)
        f.light_dir[2] = lx * math.sin(a) + lz * math.cos(a)
    if c.get("layers"):
        f.layer_begin, f.layer_count = _layer_range(c, k)
    return f


class _DeviceArray:
    """Device memory of the library as torch sees it; its owner lives as long as a tensor over it."""

    def __init__(self, owner, ptr, shape):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": "<f4", "data": (ptr, False), "version": 3}


def _atlas(s):
    """The grid's current atlas, as the lighting pass reads it (it alternates between two buffers)."""
    ptr, w, h = s["grid"].atlas_device()
    if ptr not in s["views"]:
        s["views"][ptr] = torch.as_tensor(_DeviceArray(s["grid"], ptr, (h, w, 4)), device="cuda")
    return s["views"][ptr]


def _prepare_update(c, seed):
    scene, cfg = _scene(c, seed), _config(c)
    s = {"case": c, "scene": native.DeviceScene(scene), "grid": native.ProbeGrid(cfg), "views": {}, "pass": 0,
         "frames": [_frame(c, seed, cfg, k) for k in range(FRAMES)]}
    if c["motion"] != "none":
        g = scenegen.PCG32(seed, np.arange(c["instances"]) + 300000)
        vel = np.zeros((c["instances"] + 1, 3))
        vel[1:, 0], vel[1:, 2] = g.uniform(-1.0, 1.0), g.uniform(-1.0, 1.0)
        s["instances"] = [scenegen.dynamic_instances(scene, vel, k) for k in range(8)]
    return s


def _run_update(s):
    k, c = s["pass"], s["case"]
    s["pass"] = k + 1
    f = s["frames"][k % FRAMES]
    if c["motion"] != "none":
        inst = s["instances"][k % 8]
        if c["motion"] == "rebuild" or k % 4 == 3:
            s["scene"].rebuild(inst)
        else:
            s["scene"].refit(inst)
        s["grid"].translate(f.camera_pos)
    s["grid"].update(s["scene"], f)
    return _atlas(s)


def _radiance(c, seed, device="cuda"):
    """[probe][3][ray]: log-uniform on [1e-3, 50], with a run of rays that see one sky value."""
    p = c["nx"] * c["ny"] * c["nz"]
    g = torch.Generator(device=device).manual_seed(seed)
    u = torch.rand((p, 3, c["rays"]), generator=g, device=device)
    r = torch.exp(math.log(1e-3) + u * math.log(5e4))
    r[:, :, : c["rays"] // 3] = 0.3
    return r


def _prepare_convolve(c, seed):
    cfg = _config(c)
    s = {"grid": native.ProbeGrid(cfg), "views": {}, "frame": scenegen.make_frame(1 + seed, config=cfg, iteration=seed)}
    s["grid"].set_radiance(s["frame"], _radiance(c, seed).cpu().numpy())
    return s


def _run_convolve(s):
    s["grid"].convolve(s["frame"])
    return _atlas(s)


CAMERA = (0.5, 12.0, 0.5)


def _surface(c, seed):
    """G-buffer [n][12] of a view over rolling ground (y = 1.5 + 1.5 sin cos) with detailed
    normals; pixels above the horizon lie far out, beyond the probes' range."""
    w, h = c["width"], c["height"]
    g = torch.Generator(device="cuda").manual_seed(seed)
    phase = torch.rand(4, generator=g, device="cuda", dtype=torch.float64) * 6.283
    y, x = torch.meshgrid(torch.arange(h, device="cuda", dtype=torch.float64),
                          torch.arange(w, device="cuda", dtype=torch.float64), indexing="ij")
    a, b = ((2 * x + 1) / w - 1) * 0.577 * 16 / 9, (1 - (2 * y + 1) / h) * 0.577
    yaw, pitch = phase[0], -0.6
    cp, sp = math.cos(pitch), math.sin(pitch)
    up, fwd = b * cp + sp, cp - b * sp
    dx, dz = fwd * torch.cos(yaw) - a * torch.sin(yaw), fwd * torch.sin(yaw) + a * torch.cos(yaw)
    t = torch.where(up < -0.02, (1.5 - CAMERA[1]) / up.clamp(max=-0.02), torch.full_like(up, 500.0)).clamp(max=500.0)
    px, pz = CAMERA[0] + t * dx, CAMERA[2] + t * dz
    sx, cx = torch.sin(0.7 * px + phase[1]), torch.cos(0.7 * px + phase[1])
    sz, cz = torch.sin(0.5 * pz + phase[2]), torch.cos(0.5 * pz + phase[2])
    n = torch.stack([-1.05 * cx * cz, torch.ones_like(px), 0.75 * sx * sz], -1)
    n = n + 0.15 * torch.randn(n.shape, generator=g, device="cuda", dtype=torch.float64)
    n = n / n.norm(dim=-1, keepdim=True)
    buf = torch.empty((h, w, 12), device="cuda", dtype=torch.float64)
    buf[..., 0], buf[..., 1], buf[..., 2] = px, 1.5 + 1.5 * sx * cz, pz
    buf[..., 3] = (torch.sin(0.9 * px) > 0).double()
    buf[..., 4:7] = n
    buf[..., 7] = (torch.sin(0.3 * pz + phase[3]) > 0.6).double()
    buf[..., 8:11] = 0.15 + 0.7 * torch.rand((h, w, 3), generator=g, device="cuda", dtype=torch.float64)
    buf[..., 11] = 0.6 + 0.35 * sx
    return buf.reshape(-1, 12).float()


def _probe_atlas(c, seed):
    """A plausible atlas: a level per probe, shaded over its tile."""
    p = c["nx"] * c["ny"] * c["nz"]
    g = torch.Generator(device="cuda").manual_seed(seed + 1000003)
    level = torch.exp(1.5 * torch.randn((p, 1, 1, 3), generator=g, device="cuda"))
    tile = level * (0.4 + torch.rand((p, 10, 10, 3), generator=g, device="cuda"))
    a = torch.ones((p, 10, 10, 4), device="cuda")
    a[..., :3] = tile
    rows = c["ny"] * c["nz"]
    return a.reshape(rows, c["nx"], 10, 10, 4).permute(0, 2, 1, 3, 4).reshape(10 * rows, 10 * c["nx"], 4).contiguous()


def _prepare_gi(c, seed):
    cfg = _config(c)
    s = {"grid": native.ProbeGrid(cfg), "frame": scenegen.make_frame(1 + seed, camera=CAMERA, config=cfg),
         "gbuf": _surface(c, seed)}
    s["grid"].atlas = _probe_atlas(c, seed).cpu().numpy()
    s["out"] = torch.empty((len(s["gbuf"]), 4), device="cuda")
    return s


def _run_gi(s):
    native.check(native.load().ane_ddgi_gi_lookup(s["grid"].handle, ctypes.byref(s["frame"]), s["gbuf"].data_ptr(),
                                                  len(s["gbuf"]), s["out"].data_ptr(), None))
    return s["out"]


def _view(c, scene):
    """Depth [h][w], normals [h][w][4] and the column-major inverse view-projection of a view over
    the scene, from camera rays; normals are the position gradients, facing the camera."""
    w, h = c["width"], c["height"]
    eye = torch.tensor([0.5, 20.0, 0.5], dtype=torch.float64)
    f = torch.tensor([60.0, 0.0, 60.0], dtype=torch.float64) - eye
    f = f / f.norm()
    r = torch.linalg.cross(f, torch.tensor([0.0, 1.0, 0.0], dtype=torch.float64))
    r = r / r.norm()
    u = torch.linalg.cross(r, f)
    view = torch.eye(4, dtype=torch.float64)
    view[0, :3], view[1, :3], view[2, :3] = r, u, -f
    view[:3, 3] = -view[:3, :3] @ eye
    near, far, t = 0.1, 500.0, 1.0 / math.tan(math.radians(30.0))
    proj = torch.zeros((4, 4), dtype=torch.float64)
    proj[0, 0], proj[1, 1] = t * h / w, t
    proj[2, 2], proj[2, 3], proj[3, 2] = far / (near - far), -far * near / (far - near), -1.0
    vp = proj @ view
    ivp = torch.linalg.inv(vp)
    vp, inv, eye = vp.cuda(), ivp.cuda(), eye.cuda()
    y, x = torch.meshgrid(torch.arange(h, device="cuda", dtype=torch.float64),
                          torch.arange(w, device="cuda", dtype=torch.float64), indexing="ij")
    clip = torch.stack([(2 * x + 1) / w - 1, (2 * y + 1) / h - 1, torch.ones_like(x), torch.ones_like(x)], -1)
    p = (clip.reshape(-1, 4) @ inv.T.contiguous())
    d = p[:, :3] / p[:, 3:] - eye
    d = (d / d.norm(dim=1, keepdim=True)).float().contiguous()
    o = eye.float().expand(len(d), 3).contiguous()
    hits = _trace(scene, o, d, 0.0, 490.0)
    hit = hits[:, 0].view(torch.int32) >= 0
    pos = eye + d.double() * hits[:, 1:2].double()
    ndc = torch.cat([pos, torch.ones_like(pos[:, :1])], 1) @ vp.T.contiguous()
    depth = torch.where(hit, ndc[:, 2] / ndc[:, 3].where(hit, torch.ones_like(ndc[:, 3])), torch.ones_like(ndc[:, 2]))
    img = pos.reshape(h, w, 3)
    gy, gx = torch.gradient(img, dim=(0, 1))
    n = torch.linalg.cross(gy, gx)
    n = n * torch.where((n * (eye - img)).sum(-1, keepdim=True) < 0, -1.0, 1.0)
    ln = n.norm(dim=-1, keepdim=True)
    n = torch.where(ln > 1e-12, n / ln.clamp(min=1e-12), torch.tensor([0.0, 1.0, 0.0], device="cuda").double())
    normal = torch.zeros((h, w, 4), device="cuda")
    normal[..., :3] = n.float()
    return depth.float().reshape(h, w).contiguous(), normal, ivp.T.contiguous().numpy().astype(np.float32).ravel()


def _trace(scene, orig, dirs, tmin, tmax, any_hit=0, out=None):
    hits = torch.empty((len(orig), 4), device="cuda") if out is None else out
    native.check(native.load().ane_scene_trace_rays_noalloc(scene.handle, orig.data_ptr(), dirs.data_ptr(), len(orig),
                                                            tmin, tmax, any_hit, hits.data_ptr(), None, None))
    return hits


def _prepare_mask(c, seed):
    scene = native.DeviceScene(_scene(c, seed))
    depth, _, ivp = _view(c, scene)
    light = np.array(scenegen.make_frame(1 + seed).light_dir[:3], np.float32)
    return {"scene": scene, "depth": depth, "ivp": ivp, "light": light, "out": torch.empty_like(depth)}


def _run_mask(s):
    h, w = s["depth"].shape
    native.check(native.load().ane_scene_shadow_mask(s["scene"].handle, s["depth"].data_ptr(), w, h, s["ivp"].ctypes.data,
                                                     s["light"].ctypes.data, s["out"].data_ptr(), None, None))
    return s["out"]


def _prepare_mirror(c, seed):
    cfg = _config(c)
    scene = native.DeviceScene(_scene(c, seed))
    depth, normal, ivp = _view(c, scene)
    grid = native.ProbeGrid(cfg)
    grid.atlas = _probe_atlas(c, seed).cpu().numpy()
    return {"scene": scene, "grid": grid, "depth": depth, "normal": normal, "ivp": ivp,
            "frame": scenegen.make_frame(1 + seed, camera=(0.5, 20.0, 0.5), config=cfg), "out": torch.empty_like(normal)}


def _run_mirror(s):
    h, w = s["depth"].shape
    native.check(native.load().ane_ddgi_mirror_reflections(
        s["grid"].handle, s["scene"].handle, ctypes.byref(s["frame"]), s["depth"].data_ptr(), s["normal"].data_ptr(),
        w, h, s["ivp"].ctypes.data, s["out"].data_ptr(), None, None))
    return s["out"]


def _prepare_lights(c, seed):
    n, half = c["lights"], c["cells"] / 2.0 - 4.0
    rng = np.random.default_rng(seed)
    lights = np.ones((n, 8), np.float32)
    lights[:, 0], lights[:, 2] = rng.uniform(-half, half, n), rng.uniform(-half, half, n)
    lights[:, 1], lights[:, 3] = rng.uniform(1.0, 12.0, n), rng.uniform(5.0, 30.0, n)
    # the moments image's border columns are the caller's: they are not written
    return {"scene": native.DeviceScene(_scene(c, seed)), "lights": lights,
            "dist": torch.zeros((32, 32 * n), device="cuda"), "moments": torch.zeros((8, 10 * n, 2), device="cuda")}


def _run_lights(s):
    native.check(native.load().ane_scene_light_shadows(s["scene"].handle, s["lights"].ctypes.data, len(s["lights"]),
                                                       s["dist"].data_ptr(), s["moments"].data_ptr(), None, None))
    return s["dist"], s["moments"]


def _prepare_rays(c, seed):
    n, half = c["count"], c["cells"] / 2.0
    g = torch.Generator(device="cuda").manual_seed(seed)
    o = (torch.rand((n, 3), generator=g, device="cuda") * 2 - 1) * torch.tensor([half, 4.0, half], device="cuda")
    o[:, 1] += 12.0
    d = torch.randn((n, 3), generator=g, device="cuda")
    d = d / d.norm(dim=1, keepdim=True)
    hits = torch.empty((n, 4), device="cuda")
    return {"scene": native.DeviceScene(_scene(c, seed)), "orig": o, "dirs": d, "any": int(c["any"]), "hits": hits,
            "tri": hits.view(torch.int32)[:, 0], "tuv": hits[:, 1:]}


def _run_rays(s):
    _trace(s["scene"], s["orig"], s["dirs"], 0.1, 50.0, s["any"], s["hits"])
    # of an any-hit query only whether there is a hit is defined
    return s["tri"] >= 0 if s["any"] else (s["tri"], s["tuv"])


_PREPARE = {"update": _prepare_update, "convolve": _prepare_convolve, "gi": _prepare_gi, "mask": _prepare_mask,
            "mirror": _prepare_mirror, "lights": _prepare_lights, "rays": _prepare_rays}
_RUN = {"update": _run_update, "convolve": _run_convolve, "gi": _run_gi, "mask": _run_mask, "mirror": _run_mirror,
        "lights": _run_lights, "rays": _run_rays}


def prepare(case, seed):
    s = _PREPARE[case["kind"]](case, seed)
    s["run"] = _RUN[case["kind"]]
    return s


def run(state):
    return state["run"](state)


def work(case):
    """A ray cannot do with fewer box pairs than the depth of a balanced hierarchy (2 x 24
    operations each) and one triangle test; inputs are read and outputs written once."""
    def traced(n, tris):
        return n * (48.0 * math.log2(max(tris, 2)) + 60.0)

    k = case["kind"]
    if k in ("convolve", "update"):
        probes = case["nx"] * case["nz"] * ((case["layers"] or case["ny"]) if k == "update" else case["ny"])
        n = probes * case["rays"]
        gemm, atlas = 2.0 * 64 * 3 * n, probes * 64 * 16 * 2.0
        if k == "convolve":
            return {"bytes": n * 3.0 * {FP32: 4, BF16: 2, FP16: 2, FP8: 1}[case["precision"]] + atlas, "flops": gemm}
        # the triangles of the scene, moved ones read and written
        tris = _triangles(case)
        return {"bytes": 48.0 * tris * (2 if case["motion"] != "none" else 1) + atlas,
                "flops": traced(n, tris) + gemm + 200.0 * n}
    if k == "lights":
        tris, n = _triangles(case), 1024 * case["lights"]
        return {"bytes": 48.0 * min(tris, n) + n * 4.0 + 64 * 8.0 * case["lights"], "flops": traced(n, tris)}
    if k == "rays":
        tris = _triangles(case)
        return {"bytes": 48.0 * min(tris, case["count"]) + 40.0 * case["count"], "flops": traced(case["count"], tris)}
    n = case["width"] * case["height"]
    if k == "gi":
        return {"bytes": 64.0 * n + case["nx"] * case["ny"] * case["nz"] * 1024.0, "flops": 500.0 * n}
    tris = _triangles(case)
    if k == "mask":
        return {"bytes": 8.0 * n + 48.0 * min(tris, n), "flops": traced(n, tris)}
    return {"bytes": 36.0 * n + 48.0 * min(tris, n) + case["nx"] * case["ny"] * case["nz"] * 1024.0,
            "flops": 1.5 * traced(n, tris) + 700.0 * n}


# ---------------------------------------------------------------------------
# the same results in 64 bits
# ---------------------------------------------------------------------------
def exact(case, seed):
    if case["kind"] == "convolve":
        return _exact_convolve(case, seed)
    if case["kind"] == "gi":
        return _exact_gi(case, seed)
    # brute force over all triangles: a room's; a terrain's million would take minutes
    if case["kind"] == "update" and case["family"] == "room" and _triangles(case) < 5000:
        return _exact_room(case, seed)
    return None


def _rotated_dirs(n, frame):
    i = torch.arange(n, dtype=torch.float64)
    theta, phi = 2 * 3.14159265359 * i / 1.6180339887, torch.acos(1 - 2 * (i + 0.5) / n)
    d = torch.stack([torch.cos(theta) * torch.sin(phi), torch.sin(theta) * torch.sin(phi), torch.cos(phi)], -1)
    d = d / d.norm(dim=1, keepdim=True)
    m = torch.tensor(list(frame.rotation), dtype=torch.float64).reshape(4, 4)[:3, :3]  # rows: columns of the matrix
    return (d @ m).cuda()


def _texel_dirs():
    t = (2 * torch.arange(8, dtype=torch.float64) + 1) / 8 - 1
    y, x = torch.meshgrid(t, t, indexing="ij")
    z = 1 - x.abs() - y.abs()
    fx, fy = (1 - y.abs()) * torch.where(x >= 0, 1.0, -1.0), (1 - x.abs()) * torch.where(y >= 0, 1.0, -1.0)
    x, y = torch.where(z < 0, fx, x), torch.where(z < 0, fy, y)
    d = torch.stack([x, z, y], -1).reshape(64, 3)
    return (d / d.norm(dim=1, keepdim=True)).cuda()


def _blend(case, cfg, frame, radiance):
    """The atlas after one convolution of ``radiance`` ([probe][3][ray], the frame's layers) into a
    cleared atlas."""
    w = (_texel_dirs() @ _rotated_dirs(case["rays"], frame).T.contiguous()).clamp(min=0.0)
    w = torch.where(w > 1e-6, w, torch.zeros_like(w))
    total = w.sum(1)
    e = (radiance.reshape(-1, case["rays"]) @ (w / total[:, None]).T.contiguous()).reshape(-1, 3, 8, 8)
    h = float(cfg.hysteresis)
    rows = frame.layer_count * case["nz"]
    tile = torch.zeros((rows, case["nx"], 10, 10, 4), dtype=torch.float64, device="cuda")
    tile[..., 3] = 1.0
    tile[:, :, 1:9, 1:9, :3] = (1 - h) * e.permute(0, 2, 3, 1).reshape(rows, case["nx"], 8, 8, 3)
    tile[:, :, 1:9, 1:9, 3] = (1 - h) * total.reshape(8, 8) + h
    out = torch.zeros((10 * case["ny"] * case["nz"], 10 * case["nx"], 4), dtype=torch.float64, device="cuda")
    out[..., 3] = 1.0
    r0 = 10 * frame.layer_begin * case["nz"]
    out[r0:r0 + 10 * rows] = tile.permute(0, 2, 1, 3, 4).reshape(10 * rows, 10 * case["nx"], 4)
    return out


def _exact_convolve(case, seed):
    cfg = _config(case)
    return _blend(case, cfg, scenegen.make_frame(1 + seed, config=cfg, iteration=seed), _radiance(case, seed).double())


def _exact_gi(case, seed):
    cfg, buf = _config(case), _surface(case, seed).double()
    f = scenegen.make_frame(1 + seed, camera=CAMERA, config=cfg)
    atlas = _probe_atlas(case, seed).double()
    cam = torch.tensor(list(f.camera_pos)[:3], dtype=torch.float64, device="cuda")
    outs = [_gi(case, cfg, f, atlas, cam, part) for part in buf.split(1 << 18)]
    return torch.cat(outs)


def _gi(case, cfg, f, atlas, cam, b):
    pos, shadow, nrm, metal = b[:, :3], b[:, 3:4].clamp(0.3, 1.0), b[:, 4:7], b[:, 7:8]
    albedo, rough = b[:, 8:11], b[:, 11:12]
    v = cam - pos
    dist = v.norm(dim=1, keepdim=True)
    v = v / dist
    f0 = 0.04 * (1 - metal) + albedo * metal
    p5 = (1 - (nrm * v).sum(1, keepdim=True).clamp(min=0.0)).clamp(0.0, 1.0) ** 5
    ks = f0 + (torch.maximum(1 - rough * rough, f0) - f0) * p5
    near = (1 - ks) * (1 - metal) * _sample(case, cfg, atlas, cam, pos, nrm) * albedo
    far = 0.3 * f.sky_intensity * albedo * shadow
    amb = torch.where(dist > case["nx"] * cfg.probe_step[0] / 2, far, near)
    return torch.cat([amb, torch.zeros_like(dist)], 1)


def _sample(case, cfg, atlas, cam, pos, nrm):
    num = torch.tensor([case["nx"], case["ny"], case["nz"]], dtype=torch.float64, device="cuda")
    step = torch.tensor(list(cfg.probe_step), dtype=torch.float64, device="cuda")
    off = torch.trunc(cam / step) * step - step * num / 2
    off[1] = 0.0
    cell = torch.minimum(torch.floor((pos - off) / step).clamp(min=0.0), num - 1)
    base = cell * step + off
    alpha = ((pos - base) / step).clamp(0.0, 1.0)
    n = nrm / nrm.norm(dim=1, keepdim=True)
    q = n / n.abs().sum(1, keepdim=True)
    ox, oy, oz = q[:, 0], q[:, 2], q[:, 1]
    fx, fy = (1 - oy.abs()) * torch.where(ox >= 0, 1.0, -1.0), (1 - ox.abs()) * torch.where(oy >= 0, 1.0, -1.0)
    ox, oy = (torch.where(oz < 0, fx, ox) + 1) / 2, (torch.where(oz < 0, fy, oy) + 1) / 2
    height, width = atlas.shape[:2]
    total, weight = torch.zeros_like(pos), torch.zeros_like(pos[:, :1])
    for k in range(8):
        corner = torch.tensor([k & 1, (k >> 1) & 1, (k >> 2) & 1], dtype=torch.float64, device="cuda")
        c = cell + corner
        x = 10 * c[:, 0] + 1 + 7 * ox
        y = 10 * (c[:, 1] * case["nz"] + c[:, 2]) + 1 + 7 * oy
        # texel centres: the tile's texture bounds run from centre 1 to centre 8
        x0, y0 = torch.floor(x), torch.floor(y)
        ax, ay = (x - x0)[:, None], (y - y0)[:, None]
        xi = [(x0.long() + d) % width for d in (0, 1)]
        yi = [(y0.long() + d) % height for d in (0, 1)]
        texel = (1 - ay) * ((1 - ax) * atlas[yi[0], xi[0], :3] + ax * atlas[yi[0], xi[1], :3]) + \
            ay * ((1 - ax) * atlas[yi[1], xi[0], :3] + ax * atlas[yi[1], xi[1], :3])
        d = base + corner * step - pos
        wrap = (((d * nrm).sum(1, keepdim=True) / d.norm(dim=1, keepdim=True) + 1) / 2).clamp(min=0.0001)
        w = wrap * wrap + 0.2
        w = w * torch.where(corner > 0, alpha, 1 - alpha).prod(1, keepdim=True)
        total, weight = total + w * texel.sqrt(), weight + w
    return (total / weight) ** 2 * 0.5 * 3.1415926


def _nearest(o, d, tri, tmin, tmax):
    """Index, distance and barycentrics of the closest of ``tri`` [n][3][3] per ray (index -1: none)."""
    a, e1, e2 = tri[:, 0], tri[:, 1] - tri[:, 0], tri[:, 2] - tri[:, 0]
    best = []
    for po, pd in zip(o.split(4096), d.split(4096)):
        h = torch.linalg.cross(pd[:, None], e2[None])
        det = (e1 * h).sum(-1)
        s = po[:, None] - a
        u = (s * h).sum(-1) / det
        q = torch.linalg.cross(s, e1[None].expand_as(s))
        v = (pd[:, None] * q).sum(-1) / det
        t = (e2 * q).sum(-1) / det
        ok = (u >= 0) & (v >= 0) & (u + v <= 1) & (t >= tmin) & (t <= tmax)
        t = torch.where(ok, t, torch.full_like(t, math.inf))
        m, i = t.min(1)
        best.append((torch.where(m < math.inf, i, -1), m, u.gather(1, i[:, None])[:, 0], v.gather(1, i[:, None])[:, 0]))
    return [torch.cat(x) for x in zip(*best)]


def _exact_room(case, seed):
    """The first update of a cleared atlas: closest hits, sun shadows, direct light and emission in 64
    bits (the indirect term is zero while the atlas is black), then the convolution."""
    cfg, sc = _config(case), _scene(case, seed)
    f = _frame(case, seed, cfg, 0)
    if f.flags & FLAG_BAKE:
        return None
    tri, nrm, mat = [], [], []
    for inst in sc.instances:
        m = sc.meshes[(int(inst["custom_index_and_mask"]) >> 10) & 0x3FFF]
        i = sc.indices[m["index_offset"]:m["index_offset"] + m["index_count"]].astype(np.int64) + int(m["vertex_offset"])
        t = inst["transform"].astype(np.float64).reshape(3, 4)
        tri.append((sc.vertices[i, :3].astype(np.float64) @ t[:, :3].T + t[:, 3]).reshape(-1, 3, 3))
        n = sc.vertices[i, 6:9].astype(np.float64) @ np.linalg.inv(t[:, :3])
        nrm.append(n.reshape(-1, 3, 3))
        mat += [int(inst["custom_index_and_mask"]) & 0x3FF] * (len(i) // 3)
    tri, nrm = torch.tensor(np.concatenate(tri)).cuda(), torch.tensor(np.concatenate(nrm)).cuda()
    rec = sc.materials[np.array(mat)]
    albedo, metal = torch.tensor(rec["base_col_fac"][:, :3]).double().cuda(), torch.tensor(rec["met_rough"]).double().cuda()
    emit = torch.tensor(rec["emissive"]).double().cuda()
    nx, nz, ny, rays = case["nx"], case["nz"], f.layer_count, case["rays"]
    y, z, x = torch.meshgrid(torch.arange(f.layer_begin, f.layer_begin + ny), torch.arange(nz), torch.arange(nx), indexing="ij")
    step = torch.tensor(list(cfg.probe_step), dtype=torch.float64)
    off = torch.trunc(torch.tensor(list(f.camera_pos)[:3], dtype=torch.float64) / step) * step \
        - step * torch.tensor([nx, 0, nz], dtype=torch.float64) / 2
    off[1] = 0.0
    org = (torch.stack([x, y, z], -1).reshape(-1, 3).double() * step + off).cuda()
    o = org[:, None].expand(-1, rays, -1).reshape(-1, 3)
    d = _rotated_dirs(rays, f)[None].expand(len(org), -1, -1).reshape(-1, 3)
    k, t, u, v = _nearest(o, d, tri, float(cfg.t_min), float(cfg.t_max))
    hit = k >= 0
    sky = f.sky_intensity * f.sky_color[0]
    sky = sky / 12.92 if sky < 0.04045 else ((sky + 0.055) / 1.055) ** 2.4
    out = torch.full_like(o, sky)
    ki, b = k[hit], torch.stack([1 - u - v, u, v], -1)[hit][:, :, None]
    p = (tri[ki] * b).sum(1)
    n = (nrm[ki] * b).sum(1)
    n = n / n.norm(dim=1, keepdim=True)
    sun = -torch.tensor(list(f.light_dir)[:3], dtype=torch.float64, device="cuda")
    sun = (sun / sun.norm()).expand_as(p)
    lit = _nearest(p, sun, tri, float(cfg.t_min), float(cfg.t_max))[0] < 0
    view = o[hit] - p
    view = view / view.norm(dim=1, keepdim=True)
    half = view + sun
    half = half / half.norm(dim=1, keepdim=True)
    al, met, ro = albedo[ki], metal[ki, 0:1], metal[ki, 1:2]

    def dot(a, c):
        return (a * c).sum(1, keepdim=True).clamp(min=0.0)

    a2, nl, nv = ro ** 4, dot(n, sun), dot(n, view)
    ndf = (a2 + 0.001) / (3.14159265359 * (dot(n, half) ** 2 * (a2 - 1) + 1) ** 2)
    g = (ro + 1) ** 2 / 8
    g = nl / (nl * (1 - g) + g) * nv / (nv * (1 - g) + g)
    f0 = 0.04 * (1 - met) + al * met
    fr = f0 + (1 - f0) * (1 - dot(half, view)).clamp(0.0, 1.0) ** 5
    spec = (fr * ndf * g / (4 * nv * nl + 0.0001)).clamp(0.0, 1.0)
    direct = ((1 - fr) * (1 - met) * al / 3.14159265359 + spec) * f.sun_intensity * nl
    out[hit] = direct * lit[:, None] + emit[ki, :3] * emit[ki, 3:4]
    return _blend(case, cfg, f, out.reshape(-1, rays, 3).permute(0, 2, 1).contiguous())
