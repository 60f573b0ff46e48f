"""Shadow rays through the sun grid's bounds check against the traversal, at scales and
offsets where cells, margins and 256ths of a cell meet the rounding of the coordinates."""
import numpy as np
import pytest

from anerend_amd import native, scenegen
from anerend_amd.types import Config

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scale,offset", [(1.0, 0.0), (1e-2, 0.0), (40.0, 0.0), (1.0, 3000.0), (1.0, 3e5)])
def test_sun_grid_decides_as_the_traversal(scale, offset):
    scene = scenegen.terrain_scene(9, cells=48, num_instances=200, spread=18.0)
    t = scene.instances["transform"].reshape(-1, 3, 4)
    t *= np.float32(scale)
    t[:, 0, 3] += np.float32(offset)
    ds = native.DeviceScene(scene)
    cfg = Config.make((9, 5, 7), step=(3.0 * scale,) * 3, rays=160, t_min=0.1 * scale, t_max=50.0 * scale)
    a, b = native.ProbeGrid(cfg), native.ProbeGrid(cfg)
    b.set_counting(1)  # every ray traverses
    used = False
    for sun in ((0.3, -1.0, 0.2), (2.0, -1.0, 0.7), (1e-3, -1.0, 1e-3), (-5.0, -0.5, 4.0)):
        for k in range(2):
            f = scenegen.make_frame(4, camera=(offset, 12.0 * scale, 0.5), config=cfg, iteration=k)
            f.light_dir[:] = (*sun, 0.0)
            a.update(ds, f)
            b.update(ds, f)
            (ha, sa), (hb, sb) = a.debug_rays(f), b.debug_rays(f)
            assert np.array_equal(ha, hb) and np.array_equal(sa, sb)
        used = used or a.stats()["sun_grid_state"] == 1
    # 3e5 m out the margin is 6 m, a cell's candidates are too many and the traversal is kept
    assert used == (offset < 1e5)
    assert (sb == 0).any() and (sb == 1).any()
