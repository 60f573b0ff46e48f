"""A sun that moves with every update whose calls are captured into graphs: builds end once
a grid was found out of use, and a caller's capture never starts them by itself."""
import ctypes

import numpy as np
import pytest

from anerend_amd import native, scenegen
from anerend_amd.types import INSTANCE_DTYPE, MATERIAL_DTYPE, Config
from tests.test_gpu_graph_replays import Graph, strip_scene

pytestmark = pytest.mark.gpu

CFG = Config.make((8, 8, 16), step=(2.0, 2.0, 2.0), rays=640)  # 655,360 rays, over 2.5 a triangle + 600,000


def towers_scene():
    """16,000 small triangles in 160 rows along x: along x over 32 candidates of a ray."""
    rng = np.random.default_rng(5)
    spot = np.repeat(rng.uniform(0, 20, (160, 2)), 100, 0)
    c = np.concatenate([rng.uniform(-200, 200, (16000, 1)), spot], 1)
    p = (c[:, None, :] + rng.uniform(-0.05, 0.05, (16000, 3, 3))).reshape(-1, 3).astype(np.float32)
    mb = scenegen._MeshBuilder()
    mesh = mb.add(p, np.tile(np.float32([0, 1, 0]), (len(p), 1)), np.arange(len(p), dtype=np.uint32))
    v, i, m = mb.arrays()
    mats = np.zeros(1, MATERIAL_DTYPE)
    mats["bindless_indices"] = -1
    mats["base_col_fac"] = (0.6, 0.5, 0.4, 1)
    inst = np.array([scenegen.make_instance(mesh, 0, np.eye(3), (1, 1, 1), (0, 0, 0))], INSTANCE_DTYPE)
    return scenegen.Scene(v, i, m, mats, inst)


def frame(k, along):
    f = scenegen.make_frame(4, camera=(0.5, 12.0, 0.5), config=CFG, iteration=k)
    a = 1e-5 * (k + 1)
    f.light_dir[:] = (1.0, -a, a, 0.0) if along else (0.1 + 0.01 * k, -1.0, 0.2, 0.0)
    return f


def library_graph(grid, ds, f, stream):
    """The request loop's captured update (ane::ddgi_update_graph)."""
    fn = getattr(native.load(), "_ZN3ane17ddgi_update_graphEP12ane_ddgi_ctxPK9ane_scenePK14ane_ddgi_frameP12ihipStream_t")
    fn.restype, fn.argtypes = ctypes.c_int, [ctypes.c_void_p] * 4
    native.check(fn(grid.handle, ds.handle, ctypes.byref(f), stream))


def direct(grid, ds, f, stream):
    grid.update(ds, f, stream)


@pytest.mark.parametrize("update", [direct, library_graph])
@pytest.mark.parametrize("in_use", [True, False])
def test_builds_of_a_moving_sun_end_when_they_are_not_used(update, in_use):
    ds = native.DeviceScene(strip_scene() if in_use else towers_scene())
    a, b = native.ProbeGrid(CFG), native.ProbeGrid(CFG)
    b.set_counting(1)  # every ray traverses
    estimates = []
    for k in range(8):
        f = frame(k, along=not in_use)
        update(a, ds, f, None if update is direct else _stream())
        native.synchronize(None if update is direct else _stream())
        b.update(ds, f)
        (ha, sa), (hb, sb) = a.debug_rays(f), b.debug_rays(f)
        assert np.array_equal(ha, hb) and np.array_equal(sa, sb)
        s = a.stats()
        estimates.append(s["sun_grid_candidates"])  # of the last build that ran
    built = int(np.count_nonzero(np.diff(estimates)))  # each light's estimate is its own
    if in_use:
        assert s["sun_grid_state"] == 1 and built == 7
    else:
        assert s["sun_grid_state"] == 2 and s["sun_grid_candidates"] > 32.0 and built == 1


_made = []


def _stream():
    if not _made:
        _made.append(Graph(lambda st: 0))
    return _made[0].stream


def test_a_callers_capture_of_a_new_direction_traverses():
    """The first update prepared no grid: one captured for another light right after it
    allocates nothing and builds nothing."""
    ds = native.DeviceScene(strip_scene())
    a, b = native.ProbeGrid(CFG), native.ProbeGrid(CFG)
    b.set_counting(1)
    f = [frame(k, along=False) for k in range(2)]
    a.update(ds, f[0])
    native.synchronize()
    g = Graph(lambda st: native.load().ane_ddgi_update(a.handle, ds.handle, ctypes.byref(f[1]), st))
    assert a.stats()["sun_grid_state"] == 0
    b.update(ds, f[0])
    for _ in range(3):
        g.launch()
        b.update(ds, f[1])
        (ha, sa), (hb, sb) = a.debug_rays(f[1]), b.debug_rays(f[1])
        assert np.array_equal(ha, hb) and np.array_equal(sa, sb)
        assert np.array_equal(a.atlas, b.atlas)
    g.close()


@pytest.mark.parametrize("update", [direct, library_graph])
def test_builds_end_beside_a_callers_graph(update):
    """The same over a scene whose grids are refused, in a context that has a build in a
    caller's graph."""
    ds = native.DeviceScene(towers_scene())
    a, b = native.ProbeGrid(CFG), native.ProbeGrid(CFG)
    b.set_counting(1)
    stream = None if update is direct else _stream()
    same, f = native.DeviceScene(towers_scene()), frame(20, along=True)
    a.update(same, f)
    a.update(same, f)  # a first build, over another scene: the grid's buffers
    native.synchronize()
    other = frame(21, along=True)
    graphs = [Graph(lambda st: native.load().ane_ddgi_update(a.handle, ds.handle, ctypes.byref(other), st))
              for _ in range(2)]
    update(a, ds, other, stream)  # its build was captured alone
    native.synchronize(stream)
    graphs[1].launch()
    estimates = []
    for k in range(8):
        f = frame(k, along=True)
        update(a, ds, f, stream)
        native.synchronize(stream)
        estimates.append(a.stats()["sun_grid_candidates"])
    assert np.count_nonzero(np.diff(estimates)) <= 1
    a.atlas = np.zeros(CFG.atlas_shape, np.float32)
    graphs[1].launch()
    b.update(ds, other)
    (ha, sa), (hb, sb) = a.debug_rays(other), b.debug_rays(other)
    assert np.array_equal(ha, hb) and np.array_equal(sa, sb)
    for g in graphs:
        g.close()
