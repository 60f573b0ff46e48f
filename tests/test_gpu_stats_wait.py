"""Reading or resetting a context's statistics waits for the context's own calls, not for
other work on the device."""
import ctypes

import numpy as np
import pytest

from anerend_amd import native, scenegen
from anerend_amd.types import Config

pytestmark = pytest.mark.gpu

NOT_READY = 600


def new_stream(flags):
    hip = native.DeviceBuffer(1) and native.DeviceBuffer._hip
    s = ctypes.c_void_p()
    assert hip.hipStreamCreateWithFlags(ctypes.byref(s), flags) == 0
    return s


@pytest.mark.parametrize("flags", [0, 1])  # of the context's stream: blocking, non-blocking
def test_statistics_do_not_wait_for_other_streams(flags):
    ds = native.DeviceScene(scenegen.terrain_scene(9, cells=48, num_instances=200, spread=18.0))
    small = Config.make((4, 4, 4), step=(1.0, 1.0, 1.0), rays=64)
    large = Config.make((32, 16, 32), step=(1.0, 1.0, 1.0), rays=512)
    a, other = native.ProbeGrid(small), native.ProbeGrid(large)
    fa, fo = scenegen.make_frame(1, config=small), scenegen.make_frame(2, config=large)
    hip = native.DeviceBuffer(1) and native.DeviceBuffer._hip
    for _ in range(2):  # allocations and the first grids
        other.update(ds, fo)
        a.update(ds, fa)
    native.synchronize()
    word, made = native.DeviceBuffer(4), []
    for n in range(1, 9):  # streams that share no hardware queue with each other and the null stream
        stream, busy_stream = new_stream(flags), new_stream(1)
        made += [stream, busy_stream]
        for _ in range(400):  # about half a second
            other.update(ds, fo, busy_stream)
        a.update(ds, fa, stream)
        native.synchronize(stream)
        word.download(np.zeros(1, np.uint32))
        if hip.hipStreamQuery(busy_stream) == NOT_READY:
            break
        native.synchronize(busy_stream)
    else:
        pytest.skip("the streams share a hardware queue")
    s = a.stats()
    busy = hip.hipStreamQuery(busy_stream)
    a.reset_stats()
    busy_after = hip.hipStreamQuery(busy_stream)
    native.synchronize(busy_stream)
    assert busy == NOT_READY and busy_after == NOT_READY
    assert s["calls"]["trace"] == 2 + n and 0.0 < s["last_ms"]["convolve"] < 50.0
    assert other.stats()["calls"]["convolve"] == 2 + 400 * n
    for st in made:
        assert hip.hipStreamDestroy(st) == 0


@pytest.mark.parametrize("flags", [0, 1])
def test_statistics_wait_for_their_own_calls(flags):
    ds = native.DeviceScene(scenegen.terrain_scene(9, cells=48, num_instances=200, spread=18.0))
    cfg = Config.make((16, 16, 16), step=(1.0, 1.0, 1.0), rays=256)
    grid, frame, stream = native.ProbeGrid(cfg), scenegen.make_frame(1, config=cfg), new_stream(flags)
    for k in range(20):
        grid.update(ds, frame, stream)
        grid.trace(ds, frame, stream)
        grid.translate((2.0 + k, 0.0, 3.0), stream)
    s = grid.stats()
    native.synchronize(stream)
    assert grid.stats() == s
    assert s["calls"]["trace"] == 40 and s["calls"]["convolve"] == 20 and s["calls"]["translate"] == 20
    assert all(0.0 < s["last_ms"][k] < 50.0 for k in ("setup", "trace", "shade", "convolve", "translate"))
    assert native.DeviceBuffer._hip.hipStreamDestroy(stream) == 0


@pytest.mark.parametrize("handle", [None, 2])  # the null stream, the thread's own (hipStreamPerThread)
def test_statistics_of_calls_on_implicit_streams(handle):
    ds = native.DeviceScene(scenegen.room_scene(1, num_boxes=4))
    cfg = Config.make((16, 4, 16), step=(1.0, 1.0, 1.0), rays=256)
    grid, frame = native.ProbeGrid(cfg), scenegen.make_frame(1, config=cfg)
    stream = ctypes.c_void_p(handle)
    for k in range(8):
        grid.update(ds, frame, stream)
        grid.translate((2.0 + k, 0.0, 3.0), stream)
    s = grid.stats()
    native.synchronize(stream)
    assert grid.stats() == s
    assert s["calls"]["convolve"] == 8 and s["calls"]["translate"] == 8
