"""The two-level grid nodes at the shapes where they can go wrong: leaf children beside
internal ones (empty entries), origins so far out that an empty entry could be hit, and a
launch of more rays than its waves start with.  Bit-exact with the counting traversal."""
import numpy as np
import pytest

from anerend_amd import native, scenegen
from anerend_amd.types import Config

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tris", [2, 3, 4, 5, 6, 7, 9, 12])
def test_small_hierarchies_from_near_and_far(tris):
    scene = scenegen.room_scene(2, num_boxes=0)
    scene.meshes["index_count"][0] = 3 * tris
    ds = native.DeviceScene(scene)
    assert ds.info()["num_triangles"] == tris
    v = ds.world_tris().reshape(-1, 3).astype(np.float64)
    rng = np.random.default_rng(tris)
    n = 1024
    target = v[rng.integers(0, len(v), n)] * 0.5 + v[rng.integers(0, len(v), n)] * 0.5
    away = rng.normal(size=(n, 3))
    away /= np.linalg.norm(away, axis=1, keepdims=True)
    size = np.linalg.norm(v.max(0) - v.min(0))
    dist = size * 10.0 ** rng.integers(-1, 8, (n, 1))
    o = (target + away * dist).astype(np.float32)
    d = (target - o).astype(np.float32)
    d[::7] *= -1.0
    want, _ = ds.trace_rays(o, d, tmin=0.0, tmax=1e30, count=True)
    got = ds.trace_rays(o, d, tmin=0.0, tmax=1e30)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("shape", [(16, 8, 8), (17, 9, 7)])
def test_launches_with_chunks_left_to_claim(shape):
    ds = native.DeviceScene(scenegen.terrain_scene(9, cells=48, num_instances=60, spread=18.0))
    cfg = Config.make(shape, step=(1.0, 1.0, 1.0), rays=512)
    a, b = native.ProbeGrid(cfg), native.ProbeGrid(cfg)
    b.set_counting(1)
    for k in range(2):
        f = scenegen.make_frame(40 + k, camera=(0.5, 1.5, 0.5), config=cfg, iteration=k)
        a.update(ds, f)
        b.update(ds, f)
        (ha, sa), (hb, sb) = a.debug_rays(f), b.debug_rays(f)
        assert np.array_equal(ha.view(np.uint32), hb.view(np.uint32)) and np.array_equal(sa, sb)
