"""A sun that moves with every update: the grid built at once for each new direction gives
the decisions of the traversal, and is left alone where it does not pay."""
import math

import numpy as np
import pytest

from anerend_amd import native, scenegen
from anerend_amd.types import Config

pytestmark = pytest.mark.gpu


def frames(cfg, n):
    for k in range(n):
        f = scenegen.make_frame(4, camera=(0.5, 12.0, 0.5), config=cfg, iteration=k)
        f.light_dir[:] = (math.cos(0.1 * k), -1.0, math.sin(0.1 * k) + 0.3, 0.0)
        yield f


# 1.05M rays (built from the second update on), 131k rays (traversed)
@pytest.mark.parametrize("grid,builds", [((16, 8, 16), True), ((8, 8, 8), False)])
def test_moving_sun_decides_as_the_traversal(grid, builds):
    scene = scenegen.terrain_scene(9, cells=48, num_instances=200, spread=18.0)
    cfg = Config.make(grid, step=(2.0, 2.0, 2.0), rays=512 if builds else 256)
    for _ in range(2):  # a second scene may take the address of the first
        ds = native.DeviceScene(scene)
        a, b = native.ProbeGrid(cfg), native.ProbeGrid(cfg)
        b.set_counting(1)  # every ray traverses
        for k, f in enumerate(frames(cfg, 6)):
            a.update(ds, f)
            b.update(ds, f)
            (ha, sa), (hb, sb) = a.debug_rays(f), b.debug_rays(f)
            assert np.array_equal(ha, hb) and np.array_equal(sa, sb)
            assert np.array_equal(a.atlas, b.atlas)
            assert a.stats()["sun_grid_state"] == (1 if builds and k > 0 else 0)
            assert a.stats()["calls"]["sungrid"] == (k if builds else 0)
        # the sun stands still: one more build where none was made, then none
        for _ in range(3):
            a.update(ds, f)
        assert a.stats()["calls"]["sungrid"] == (5 if builds else 1)
        f.light_dir[:] = (1.0, -1.0, 1.0, 0.0)
        scene.instances["transform"][1:, 3] += 0.5  # another scene in the next round
        ds.close()
