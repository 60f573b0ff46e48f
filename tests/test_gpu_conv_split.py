"""The convolution at the probe counts where its work is split another way (row tiles per
block, rays over waves, streaming), against a float64 contraction."""
import numpy as np
import pytest

from anerend_amd import native, scenegen
from anerend_amd.types import PRECISION_BF16, PRECISION_FP8, PRECISION_FP16, PRECISION_FP32, Config

pytestmark = pytest.mark.gpu

# per operand rounding: radiance, weights and their sum's correction, then FP32 sums
UNIT = {PRECISION_FP32: 0.0, PRECISION_BF16: 2.0 ** -9, PRECISION_FP16: 2.0 ** -11, PRECISION_FP8: 2.0 ** -4}


def texel_dirs():
    t = (2 * np.arange(8) + 1) / 8 - 1
    y, x = np.meshgrid(t, t, indexing="ij")
    z = 1 - abs(x) - abs(y)
    fx, fy = (1 - abs(y)) * np.where(x >= 0, 1, -1), (1 - abs(x)) * np.where(y >= 0, 1, -1)
    d = np.stack([np.where(z < 0, fx, x), z, np.where(z < 0, fy, y)], -1).reshape(64, 3)
    return d / np.linalg.norm(d, axis=1, keepdims=True)


@pytest.mark.parametrize("precision", sorted(UNIT))
# 1 and 17 probes; 256 blocks of one row tile, of two, and one block more; the streaming threshold
@pytest.mark.parametrize("grid", [(1, 1, 1), (17, 1, 1), (32, 2, 16), (41, 5, 5), (32, 4, 16), (3, 683, 1),
                                  (32, 8, 32), (3, 2731, 1)])
def test_split_convolution_matches_float64(grid, precision):
    rays = 96
    cfg = Config.make(grid, rays=rays, hysteresis=0.5, precision=precision)
    g = native.ProbeGrid(cfg)
    frame = scenegen.make_frame(3, config=cfg)
    p = cfg.num_probes
    rad = np.random.default_rng(p).uniform(0.5, 2.0, (p, 3, rays)).astype(np.float32)
    g.set_radiance(frame, rad)
    g.convolve(frame)
    w = np.maximum(texel_dirs() @ native.ray_directions(rays, frame.rotation[:]).astype(np.float64).T, 0.0)
    w[w <= 1e-6] = 0.0
    want = 0.5 * np.einsum("tr,pcr->ptc", w / w.sum(1, keepdims=True), rad.astype(np.float64))
    nx, rows = grid[0], grid[1] * grid[2]
    a = g.atlas.reshape(rows, 10, nx, 10, 4).transpose(0, 2, 1, 3, 4)
    got = a[:, :, 1:9, 1:9, :3].reshape(p, 64, 3)
    assert np.max(np.abs(got - want) / want) < 3 * UNIT[precision] + 1e-5
    border = a.copy()
    border[:, :, 1:9, 1:9] = (0, 0, 0, 1)
    assert np.array_equal(border, np.broadcast_to(np.float32([0, 0, 0, 1]), border.shape))
