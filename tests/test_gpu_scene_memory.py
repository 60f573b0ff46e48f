"""The device memory of a scene, and the build's buffers in the grid nodes' place."""
import numpy as np
import pytest

from anerend_amd import native, scenegen
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def test_bytes_per_triangle():
    """382.3 bytes in full nodes and 414.6 with quantized ones are what a scene of terrain took
    before it held grid nodes."""
    for cells, most in ((400, 383), (1100, 415)):
        i = native.DeviceScene(scenegen.terrain_scene(9, cells=cells, num_instances=100, spread=18.0)).info()
        assert i["device_bytes"] <= most * i["num_triangles"]


@pytest.mark.parametrize("tris", [1, 2, 3, 4, 5, 1025, 1026, 4096])
def test_rebuilds_and_inspection_leave_the_hits_alone(tris):
    """The smallest scenes, whose build buffers are larger than their grid nodes, and odd counts."""
    scene = scenegen.terrain_scene(9, cells=64, num_instances=1, spread=18.0)
    scene.meshes["index_count"][0] = 3 * tris
    scene.instances = scene.instances[:1].copy()
    ds, osc = native.DeviceScene(scene), O.OracleScene(scene)
    v = ds.world_tris()
    assert np.array_equal(v.view(np.uint32), osc.world_tris().view(np.uint32).reshape(v.shape))
    rng = np.random.default_rng(tris)
    p = v.reshape(-1, 3)
    o = (p[rng.integers(0, len(p), 400)] + rng.uniform(-2, 2, (400, 3)) + [0.0, 1.0, 0.0]).astype(np.float32)
    d = (p[rng.integers(0, len(p), 400)] - o).astype(np.float32)
    want = osc.trace(o, d, tmax=1e30)[0]
    for step in (None, ds.rebuild, ds.refit, ds.rebuild):
        if step:
            step(scene.instances)
        assert np.array_equal(ds.trace_rays(o, d, tmax=1e30), want)
        assert np.array_equal(ds.world_tris().view(np.uint32), v.view(np.uint32))
        assert np.array_equal(ds.trace_rays(o, d, tmax=1e30), want)
