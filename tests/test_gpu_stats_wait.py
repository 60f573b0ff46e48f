"""Reading or resetting a context's statistics waits for the context's own calls, not for
other work on the device."""
import ctypes

import pytest

from anerend_amd import native, scenegen
from anerend_amd.types import Config

pytestmark = pytest.mark.gpu

NOT_READY = 600


@pytest.mark.parametrize("flags", [0, 1])  # of the context's own stream: blocking, non-blocking
def test_statistics_wait_for_their_context_alone(flags):
    ds = native.DeviceScene(scenegen.terrain_scene(9, cells=48, num_instances=200, spread=18.0))
    small = Config.make((16, 4, 16), step=(1.0, 1.0, 1.0), rays=256)
    large = Config.make((32, 16, 32), step=(1.0, 1.0, 1.0), rays=512)
    a, other = native.ProbeGrid(small), native.ProbeGrid(large)
    fa, fo = scenegen.make_frame(1, config=small), scenegen.make_frame(2, config=large)
    hip = native.DeviceBuffer(1) and native.DeviceBuffer._hip
    streams = [ctypes.c_void_p() for _ in range(2)]
    for s, f in zip(streams, (flags, 1)):
        assert hip.hipStreamCreateWithFlags(ctypes.byref(s), f) == 0
    other.update(ds, fo, streams[1])  # allocations and the first grid
    other.update(ds, fo, streams[1])
    a.update(ds, fa, streams[0])
    native.synchronize(streams[0])
    native.synchronize(streams[1])
    for _ in range(400):  # some 0.4 s of work
        other.update(ds, fo, streams[1])
    for k in range(20):
        a.update(ds, fa, streams[0])
        a.trace(ds, fa, streams[0])
        a.translate((2.0 + k, 0.0, 3.0), streams[0])
    s = a.stats()
    busy = hip.hipStreamQuery(streams[1])
    native.synchronize(streams[0])
    assert a.stats() == s  # its own calls were complete
    assert s["calls"]["trace"] == 41 and s["calls"]["convolve"] == 21 and s["calls"]["translate"] == 20
    assert all(0.0 < s["last_ms"][k] < 50.0 for k in ("setup", "trace", "shade", "convolve", "translate"))
    a.reset_stats()
    busy_after = hip.hipStreamQuery(streams[1])
    native.synchronize(streams[1])
    assert busy == NOT_READY and busy_after == NOT_READY
    assert other.stats()["calls"]["convolve"] == 402
    for s in streams:
        assert hip.hipStreamDestroy(s) == 0


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
