"""Screen passes captured into a caller's graph beside direct calls on the same scene and
context.  A graph that holds a sun-grid build writes the grid anew whenever it is replayed,
so a direct call that follows must not take the grid for its own light's."""
import ctypes

import numpy as np
import pytest

from anerend_amd import native, scenegen
from anerend_amd.types import INSTANCE_DTYPE, MATERIAL_DTYPE, Config
from tests.test_oracle_shading import _view_proj

pytestmark = pytest.mark.gpu

CAM = (2.0, 14.0, 18.0)
W, H = 160, 90
DOWN = (0.11, -0.9, 0.07)       # light directions: the grid is in use along this one,
SLANTED = (0.5, -0.9, -0.4)     # and along this one,
ALONG = (1.0, -0.011, 0.013)    # and over its capacity along the strip


def hip(name, *args):
    if native.DeviceBuffer._hip is None:
        native.DeviceBuffer(1).close()
    rc = getattr(native.DeviceBuffer._hip, name)(*args)
    assert rc == 0, f"{name}: {rc}"


class Graph:
    """What `call(stream)` queues, captured; launch() replays it and waits."""

    def __init__(self, call):
        self.stream, graph, self.exec = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_void_p()
        hip("hipStreamCreateWithFlags", ctypes.byref(self.stream), 1)
        hip("hipStreamBeginCapture", self.stream, 1)
        status = call(self.stream)
        rc = native.DeviceBuffer._hip.hipStreamEndCapture(self.stream, ctypes.byref(graph))
        native.check(status)
        assert rc == 0
        hip("hipGraphInstantiate", ctypes.byref(self.exec), graph, None, None, ctypes.c_size_t(0))
        hip("hipGraphDestroy", graph)

    def launch(self):
        hip("hipGraphLaunch", self.exec, self.stream)
        hip("hipStreamSynchronize", self.stream)

    def close(self):
        hip("hipGraphExecDestroy", self.exec)
        hip("hipStreamDestroy", self.stream)


def strip_scene(n=16000):
    """Small triangles over a strip 400 m long, 20 m wide and 1 m high."""
    rng = np.random.default_rng(3)
    p = rng.uniform((-200, 0, -10), (200, 1, 10), (n, 1, 3)) + rng.uniform(-0.5, 0.5, (n, 3, 3))
    p = np.ascontiguousarray(p.reshape(-1, 3), np.float32)
    mb = scenegen._MeshBuilder()
    mesh = mb.add(p, np.tile(np.float32([0, 1, 0]), (len(p), 1)), np.arange(len(p), dtype=np.uint32))
    v, i, m = mb.arrays()
    mats = np.zeros(1, MATERIAL_DTYPE)
    mats["bindless_indices"] = -1
    mats["base_col_fac"] = (0.6, 0.5, 0.4, 1)
    inst = np.array([scenegen.make_instance(mesh, 0, np.eye(3), (1, 1, 1), (0, 0, 0))], INSTANCE_DTYPE)
    return scenegen.Scene(v, i, m, mats, inst)


class Passes:
    """The shadow mask or the mirror reflections of one view, into a device image."""

    def __init__(self, kind, ds, w=W, h=H):
        rng = np.random.default_rng(8)
        self.kind, self.ds, self.w, self.h = kind, ds, w, h
        depth = rng.uniform(0.97, 0.9995, (h, w)).astype(np.float32)
        depth[:6] = 1.0
        normal = rng.normal(size=(h, w, 4)).astype(np.float32)
        self.ivp = _view_proj(CAM, (0.0, 0.0, 0.0))[1].T.ravel().astype(np.float32)
        self.cfg = Config.make((4, 3, 4), step=(4.0, 4.0, 4.0), rays=64)
        self.grid = native.ProbeGrid(self.cfg)
        self.shape = (h, w) if kind == "mask" else (h, w, 4)
        nbytes = 4 * int(np.prod(self.shape))
        self.bufs = [native.DeviceBuffer(depth.nbytes), native.DeviceBuffer(normal.nbytes), native.DeviceBuffer(nbytes)]
        self.bufs[0].upload(depth)
        self.bufs[1].upload(normal)

    def call(self, light, stream, grid=None):
        d, n, out = self.bufs
        if self.kind == "mask":
            light3 = np.array(light, np.float32)
            return native.load().ane_scene_shadow_mask(self.ds.handle, d.ptr, self.w, self.h, native.ptr(self.ivp),
                                                       native.ptr(light3), out.ptr, None, stream)
        frame = scenegen.make_frame(4, camera=CAM, config=self.cfg)
        frame.light_dir[:3] = light
        return native.load().ane_ddgi_mirror_reflections((grid or self.grid).handle, self.ds.handle,
                                                         ctypes.byref(frame), d.ptr, n.ptr, self.w, self.h,
                                                         native.ptr(self.ivp), out.ptr, None, stream)

    def image(self, run):
        self.bufs[2].upload(np.full(self.shape, -7.0, np.float32))  # a pass that writes nothing shows
        run()
        native.synchronize()
        return self.bufs[2].download(np.zeros(self.shape, np.float32))

    def direct(self, light):
        return self.image(lambda: native.check(self.call(light, None)))

    def traversed(self, light):
        """The same image from a scene and context that have no grid."""
        if self.kind == "mask":
            other = Passes("mask", native.DeviceScene(strip_scene()), self.w, self.h)
            return other.direct(light)
        return self.image(lambda: native.check(self.call(light, None, native.ProbeGrid(self.cfg))))


@pytest.mark.parametrize("kind", ["mask", "mirror"])
@pytest.mark.parametrize("other", [ALONG, SLANTED])
def test_direct_calls_after_a_replayed_build(kind, other):
    p = Passes(kind, native.DeviceScene(strip_scene()))
    want, want_other = p.traversed(DOWN), p.traversed(other)
    assert not np.array_equal(want, want_other)
    for _ in range(4):  # traversal, a build, its grid of unknown and of known state
        assert np.array_equal(p.direct(DOWN), want)
    first = Graph(lambda st: p.call(other, st))   # a light seen once: traversed
    second = Graph(lambda st: p.call(other, st))  # seen twice: this graph holds a build
    third = Graph(lambda st: p.call(other, st))   # and this one relies on it
    assert np.array_equal(p.direct(other), want_other)  # the captured build has not run
    for _ in range(3):
        assert np.array_equal(p.image(second.launch), want_other)
        assert np.array_equal(p.image(third.launch), want_other)
        assert np.array_equal(p.direct(other), want_other)
        for _ in range(4):
            assert np.array_equal(p.direct(DOWN), want)
        assert np.array_equal(p.image(second.launch), want_other)
        assert np.array_equal(p.direct(DOWN), want)  # the device holds the other light's grid
        assert np.array_equal(p.image(third.launch), want_other)
        assert np.array_equal(p.image(first.launch), want_other)
    for g in (first, second, third):
        g.close()


@pytest.mark.parametrize("kind", ["mask", "mirror"])
def test_a_pass_of_a_warm_size_is_captured(kind):
    """The grid alone answers the direct calls of the larger size; its capture queues the
    traversal too, in the workspace that those calls prepared."""
    ds = native.DeviceScene(strip_scene())
    small, large = Passes(kind, ds, 32, 24), Passes(kind, ds, 200, 130)
    large.grid = small.grid
    for _ in range(4):
        small.direct(DOWN)
    want = large.traversed(DOWN)
    for _ in range(2):
        assert np.array_equal(large.direct(DOWN), want)
    g = Graph(lambda st: large.call(DOWN, st))
    for _ in range(3):
        assert np.array_equal(large.image(g.launch), want)
        assert np.array_equal(large.direct(DOWN), want)
    g.close()
