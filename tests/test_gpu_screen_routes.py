"""The screen passes' routes: row order, tiles and cut tiles of a mirror image, and the
traversal, undecided-grid and known-grid calls of a shadow mask, all with one answer."""
import numpy as np
import pytest

from anerend_amd import native, scenegen
from anerend_amd.types import Config
from oracle import oracle as O
from tests.test_oracle_shading import _view_proj

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def world():
    scene = scenegen.terrain_scene(9, cells=48, num_instances=200, spread=18.0)
    return scene, native.DeviceScene(scene), O.OracleScene(scene)


CAM = (2.0, 14.0, 18.0)


def view(w, h):
    """Random depths of a view of the scene, a fifth of them sky."""
    rng = np.random.default_rng(1000 * w + h)
    depth = rng.uniform(0.97, 0.9995, (h, w)).astype(np.float32)
    depth[rng.random((h, w)) < 0.2] = 1.0
    return depth, rng.normal(size=(h, w, 4)).astype(np.float32), _view_proj(CAM, (0.0, 0.0, 0.0))[1].T.ravel().astype(np.float32)


# under 64 a side; exact tiles; cut tiles; one more than the threshold each way
@pytest.mark.parametrize("w,h", [(1, 1), (63, 200), (200, 63), (64, 64), (65, 64), (64, 71), (129, 97)])
def test_every_route_of_the_screen_passes_agrees(world, w, h):
    scene, ds, osc = world
    cfg = Config.make((4, 3, 4), step=(4.0, 4.0, 4.0), rays=64)
    frame = scenegen.make_frame(4, camera=CAM, config=cfg)
    depth, normal, ivp = view(w, h)
    light = np.array(frame.light_dir[:3], np.float32)
    want, _ = osc.shadow_mask(depth, ivp, light)
    for _ in range(4):  # traversal, a grid of unknown validity, a known grid
        assert np.array_equal(ds.shadow_mask(depth, ivp, light), want)
        ds.check()
    grid = native.ProbeGrid(cfg)
    ref, _ = osc.mirror_reflections(cfg, frame, O.new_atlas(cfg), depth, normal, ivp)
    first = None
    for _ in range(4):
        got = grid.mirror_reflections(ds, frame, depth, normal, ivp)
        assert np.max(np.abs(got - ref) / np.maximum(np.abs(ref), 1e-3), initial=0.0) < 1e-4
        first = got if first is None else first
        assert np.array_equal(got, first)
        grid.check()
