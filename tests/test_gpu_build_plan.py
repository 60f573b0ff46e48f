"""Builds at the sizes where the plan's scan and treelets turn over: one section or tile more
or less, one treelet, the first crossing node.  Depth and hits are the oracle's, and a
rebuild with moved instances is a new scene's."""
import numpy as np
import pytest

from anerend_amd import native, scenegen
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def scene_of(tris, shift=0.0, cells=64):
    s = scenegen.terrain_scene(9, cells=cells, num_instances=1, spread=18.0)
    s.meshes["index_count"][0] = 3 * tris
    s.instances = s.instances[:1].copy()
    s.instances["transform"].reshape(-1, 3, 4)[:, :, 3] += np.float32([shift, 0.0, -shift])
    return s


@pytest.mark.parametrize("tris", [1, 2, 3, 682, 683, 1023, 1024, 1025, 2047, 2049, 6000])
def test_plan_sizes(tris):
    scene, moved = scene_of(tris), scene_of(tris, 0.75)
    ds, osc = native.DeviceScene(scene), O.OracleScene(scene)
    assert ds.info()["num_triangles"] == tris
    if tris > 1:
        assert ds.info()["bvh_depth"] == osc.max_depth
    v = ds.world_tris().reshape(-1, 3).astype(np.float64)
    rng = np.random.default_rng(tris)
    o = (v[rng.integers(0, len(v), 500)] + rng.uniform(-2, 2, (500, 3)) + [0.0, 1.0, 0.0]).astype(np.float32)
    d = (v[rng.integers(0, len(v), 500)] - o).astype(np.float32)
    assert np.array_equal(ds.trace_rays(o, d, tmax=1e30), osc.trace(o, d, tmax=1e30)[0])
    ds.rebuild(moved.instances)
    fresh = native.DeviceScene(moved)
    assert ds.info()["bvh_depth"] == fresh.info()["bvh_depth"]
    assert np.array_equal(ds.world_tris(), fresh.world_tris())
    assert np.array_equal(ds.trace_rays(o, d, tmax=1e30), fresh.trace_rays(o, d, tmax=1e30))
    ds.refit(scene.instances)
    assert np.array_equal(ds.trace_rays(o, d, tmax=1e30), osc.trace(o, d, tmax=1e30)[0])


@pytest.mark.parametrize("tris", [131071, 131072, 131073, 524288, 524289])
def test_sort_tiles(tris):
    """Sizes around those at which the sort's tiles grow."""
    scene = scene_of(tris, cells=520)
    ds, osc = native.DeviceScene(scene), O.OracleScene(scene)
    assert ds.info()["num_triangles"] == tris
    assert ds.info()["bvh_depth"] == osc.max_depth
    v = ds.world_tris().reshape(-1, 3)
    rng = np.random.default_rng(tris)
    o = (v[rng.integers(0, len(v), 500)] + rng.uniform(-2, 2, (500, 3)) + [0.0, 1.0, 0.0]).astype(np.float32)
    d = (v[rng.integers(0, len(v), 500)] - o).astype(np.float32)
    assert np.array_equal(ds.trace_rays(o, d, tmax=1e30), osc.trace(o, d, tmax=1e30)[0])
