"""The closest-hit traversal of grid nodes against the counting traversal of the full and
quantized nodes (bit-exact with the oracle): ordinary rays, rays in box faces, tiny and huge
components, far origins, scenes that outgrow the grid at a build or at a refit."""
import numpy as np
import pytest

from anerend_amd import native, scenegen
from anerend_amd.types import Config
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def moved(scene, offset=(0, 0, 0), scale=1.0):
    t = scene.instances["transform"].reshape(-1, 3, 4)
    t *= np.float32(scale)
    t[:, :, 3] += np.float32(offset)
    return scene


def duplicated():
    """Every triangle twice: equal distances, the lower id is the hit."""
    s = scenegen.room_scene(3, num_boxes=6)
    s.instances = np.concatenate([s.instances, s.instances])
    return s


def detail():
    """Two far-apart clusters of millimetre triangles: far below 2^-16 of the extent."""
    s = moved(scenegen.room_scene(3, num_boxes=40), scale=1e-3)
    s.instances["transform"].reshape(-1, 3, 4)[::2, 0, 3] += np.float32(5000.0)
    return s


SCENES = {
    "room": lambda: scenegen.room_scene(1),
    "one_box": lambda: scenegen.room_scene(1, num_boxes=0),
    "duplicated": duplicated,
    "terrain": lambda: scenegen.terrain_scene(9, cells=48, num_instances=200, spread=18.0),
    "far": lambda: moved(scenegen.terrain_scene(9, cells=48, num_instances=200, spread=18.0), offset=(3e5, 0.0, -2e5)),
    "large": lambda: moved(scenegen.terrain_scene(9, cells=48, num_instances=200, spread=18.0), scale=1e4),
    "detail": detail,
}


def rays(ds, n=6000, seed=5):
    v = ds.world_tris().reshape(-1, 3).astype(np.float64)
    lo, hi = v.min(0), v.max(0)
    rng = np.random.default_rng(seed)
    o = rng.uniform(lo - 0.1 * (hi - lo), hi + 0.1 * (hi - lo), (n, 3))
    d = rng.normal(size=(n, 3))
    pick = v[rng.integers(0, len(v), n)]
    d[: n // 3] = pick[: n // 3] - o[: n // 3]             # through vertices
    k = slice(n // 3, n // 2)                              # along axes, from vertex coordinates (box faces)
    o[k] = np.where(rng.random((k.stop - k.start, 3)) < 0.6, pick[k], o[k])
    d[k] = np.eye(3)[rng.integers(0, 3, k.stop - k.start)] * rng.choice([-1, 1], (k.stop - k.start, 1))
    z = slice(n // 2, 2 * n // 3)                          # one zero component
    d[z][np.arange(z.stop - z.start), rng.integers(0, 3, z.stop - z.start)] = 0.0
    d[z, 1] *= rng.choice([0.0, 1e-20, 1e-28, 1e-32, 1e-40], z.stop - z.start)
    f = slice(2 * n // 3, 2 * n // 3 + 300)                # far origins
    o[f] += d[f] * -1e3 * np.linalg.norm(hi - lo)
    d[f.stop: f.stop + 200] *= 1e-18                       # lengths
    d[f.stop + 200: f.stop + 400] *= 1e18
    d[-3:] = [[0, 0, 0], [np.nan, 0, 1], [np.inf, 0, 0]]
    return o.astype(np.float32), d.astype(np.float32)


def same_hits(ds, o, d, tmax):
    want, _ = ds.trace_rays(o, d, tmin=0.0, tmax=tmax, count=True)
    got = ds.trace_rays(o, d, tmin=0.0, tmax=tmax)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    return int((want["tri"] >= 0).sum())


@pytest.mark.parametrize("fmt", [native.DeviceScene.NODES_FULL, native.DeviceScene.NODES_QUANTIZED])
@pytest.mark.parametrize("name", sorted(SCENES))
def test_closest_hits_equal_the_counting_traversal(name, fmt):
    scene = SCENES[name]()
    ds = native.DeviceScene(scene)
    ds.set_node_format(fmt)
    o, d = rays(ds)
    assert same_hits(ds, o, d, 1e30) > 100
    same_hits(ds, o, d, 5.0)
    if name in ("room", "terrain", "far"):  # the counting traversal is the oracle's
        osc = O.OracleScene(scene)
        if fmt == native.DeviceScene.NODES_FULL:
            assert np.array_equal(ds.trace_rays(o, d, tmax=1e30), osc.trace(o, d, tmax=1e30)[0])
    inst = scene.instances.copy()                          # one instance far out: a refit, then a build
    inst["transform"].reshape(-1, 3, 4)[-1, :, 3] += np.float32(1e6)
    ds.refit(inst)
    same_hits(ds, o, d, 1e30)
    ds.rebuild(inst)
    same_hits(ds, o, d, 1e30)
    ds.rebuild(scene.instances)
    same_hits(ds, o, d, 1e30)


@pytest.mark.parametrize("name", ["room", "terrain", "detail"])
def test_probe_and_shadow_rays_equal_the_counting_traversal(name):
    ds = native.DeviceScene(SCENES[name]())
    cfg = Config.make((5, 3, 4), step=(1.0, 1.0, 1.0), rays=96)
    a, b = native.ProbeGrid(cfg), native.ProbeGrid(cfg)
    b.set_counting(1)
    for k in range(4):  # a new sun each time: the shadow rays follow in the traversal's lanes
        f = scenegen.make_frame(20 + k, camera=(0.5, 1.5, 0.5), config=cfg, iteration=k)
        if k == 2:
            f.rotation[:] = scenegen.rotation_matrix(90.0, 1).tolist()
            f.light_dir[:] = (0.0, -1.0, 0.0, 0.0)
        a.update(ds, f)
        b.update(ds, f)
        (ha, sa), (hb, sb) = a.debug_rays(f), b.debug_rays(f)
        assert np.array_equal(ha.view(np.uint32), hb.view(np.uint32)) and np.array_equal(sa, sb)
        assert np.array_equal(a.atlas, b.atlas)


@pytest.mark.parametrize("tris", [1, 2, 3])
def test_smallest_hierarchies(tris):
    scene = scenegen.room_scene(1, num_boxes=0)
    scene.meshes["index_count"][0] = 3 * tris
    scene.indices = scene.indices.copy()
    ds = native.DeviceScene(scene)
    assert ds.info()["num_triangles"] == tris
    o, d = rays(ds, 1200)
    same_hits(ds, o, d, 1e30)
