"""The streaming convolution (more than 8,192 probes): blocks of 64 probes partly empty, every
prefetch depth, ray counts on both sides of what the weights may fill of the LDS, its stage
clock, and the request loop's batches of such updates beside small ones."""
import numpy as np
import pytest

from anerend_amd import native, scenegen, serving
from anerend_amd.types import PRECISION_BF16, PRECISION_FP8, PRECISION_FP16, PRECISION_FP32, Config
from tests.conftest import bits
from tests.test_gpu_conv_split import UNIT, texel_dirs

pytestmark = pytest.mark.gpu


def interior(atlas, dims):
    a = atlas.reshape(dims[1] * dims[2], 10, dims[0], 10, 4).transpose(0, 2, 1, 3, 4)
    return a[:, :, 1:9, 1:9, :3].reshape(-1, 64, 3), a


# 8,193 and 8,255 probes: one probe, and all but one, in the last block; 8,256: full.  1, 2, 3, 4, 5
# and 8 steps of 32 rays: prefetch depths 1, 2 and 4.  608 and 1,248 rays: the largest weights in
# FP32 and in 16 bits; 640 and 1,280: split rays.
@pytest.mark.parametrize("precision", sorted(UNIT))
@pytest.mark.parametrize("dims,rays", [((3, 2731, 1), 32), ((5, 13, 127), 64), ((8, 24, 43), 96), ((3, 1, 2731), 128),
                                       ((5, 127, 13), 160), ((3, 2731, 1), 256), ((5, 127, 13), 608),
                                       ((5, 127, 13), 640), ((3, 2731, 1), 1248), ((3, 2731, 1), 1280)])
def test_streaming_convolution_matches_float64(dims, rays, precision):
    cfg = Config.make(dims, rays=rays, hysteresis=0.5, precision=precision)
    g = native.ProbeGrid(cfg)
    frame = scenegen.make_frame(3, config=cfg)
    rng = np.random.default_rng(rays + cfg.num_probes)
    rad = rng.uniform(0.5, 2.0, (cfg.num_probes, 3, rays)).astype(np.float32)
    old = rng.uniform(0.5, 2.0, cfg.atlas_shape).astype(np.float32)
    g.atlas = old
    g.set_radiance(frame, rad)
    g.convolve(frame)
    w = np.maximum(texel_dirs() @ native.ray_directions(rays, frame.rotation[:]).astype(np.float64).T, 0.0)
    w[w <= 1e-6] = 0.0
    w /= w.sum(1, keepdims=True)
    fresh = (rad.reshape(-1, rays).astype(np.float64) @ w.T).reshape(-1, 3, 64).transpose(0, 2, 1)
    before, kept = interior(old, dims)
    want = 0.5 * fresh + 0.5 * before.astype(np.float64)
    got, a = interior(g.atlas, dims)
    # operand rounding of the fresh half alone, as in the split convolution's test
    assert np.max(np.abs(got - want) / want) < 3 * UNIT[precision] + 1e-5
    border = a.copy()
    border[:, :, 1:9, 1:9] = kept[:, :, 1:9, 1:9]
    assert np.array_equal(border, kept)


def test_stage_clock_of_a_streaming_convolution():
    ds = native.DeviceScene(scenegen.room_scene(1, num_boxes=4))
    cfg = Config.make((3, 2731, 1), rays=64)
    grid, frame = native.ProbeGrid(cfg), scenegen.make_frame(1, config=cfg)
    total = 0.0
    for n in range(1, 5):
        grid.update(ds, frame)
        s = grid.stats()
        assert s["calls"]["convolve"] == n and 0.0 < s["last_ms"]["convolve"] < 50.0
        total += s["last_ms"]["convolve"]
        assert s["mean_ms"]["convolve"] * n == pytest.approx(total, rel=1e-4)


@pytest.mark.parametrize("precision", [PRECISION_FP32, PRECISION_FP16, PRECISION_BF16, PRECISION_FP8])
def test_fused_batches_of_streaming_convolutions_equal_alone(precision):
    """Streaming updates of several ray counts (their greatest common divisor sets the batch's
    prefetch depth) and split-ray ones in the same batches, bit for bit their own updates."""
    shapes = [((16, 33, 16), 128), ((65, 127, 1), 64), ((16, 8, 8), 128), ((3, 2731, 1), 96), ((4, 4, 4), 640)]
    ds = native.DeviceScene(scenegen.room_scene(1, num_boxes=8))
    cfgs = [Config.make(d, step=(0.5, 0.25, 0.5), rays=n, precision=precision) for d, n in shapes]
    for count in (2, len(cfgs)):
        srv = serving.Server(hbm_budget_bytes=64 << 30, max_inflight=8, num_streams=2, capture_graphs=False,
                             fuse_stages=True)
        ids = [srv.add_session(ds, c) for c in cfgs[:count]]
        frames = [[scenegen.make_frame(7 + k, camera=(0.5, 1.0, 0.5), config=c, iteration=i)
                   for k, c in enumerate(cfgs[:count])] for i in range(4)]
        tickets = [srv.submit(ids[k], f) for per in frames for k, f in enumerate(per)]
        assert all(srv.poll(t, timeout_ms=-1)["status"] == 0 for t in tickets)
        mixed = [srv.atlas(i) for i in ids]
        srv.close()
        for k, c in enumerate(cfgs[:count]):
            grid = native.ProbeGrid(c)
            for per in frames:
                grid.update(ds, per[k])
            assert np.array_equal(bits(grid.atlas), bits(mixed[k])), f"{shapes[k]} differs alone vs mixed"
            grid.close()
