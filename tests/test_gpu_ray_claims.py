"""Every ray of a traversal launch is traced exactly once, whatever share of the rays
lies in the waves' own first chunks and whatever is claimed from the launch's counters."""
import numpy as np
import pytest

from anerend_amd import native, scenegen
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def room():
    scene = scenegen.room_scene(1)
    return native.DeviceScene(scene), O.OracleScene(scene)


# one ray; the edges of a 64-ray chunk and of a block's two; around the first chunks of a
# full launch (7168 waves at most, 458,752 rays) and beyond them, off the counters' stride
@pytest.mark.parametrize("n", [1, 63, 64, 65, 127, 129, 4096, 458751, 458752, 458753, 459777, 600001])
def test_every_ray_is_traced_once(room, n):
    ds, osc = room
    rng = np.random.default_rng(n)
    o = rng.uniform(-4.5, 4.5, (n, 3)).astype(np.float32)
    o[:, 1] = rng.uniform(-0.4, 3.4, n)
    d = rng.normal(size=(n, 3)).astype(np.float32)
    assert np.array_equal(ds.trace_rays(o, d), osc.trace(o, d)[0])
