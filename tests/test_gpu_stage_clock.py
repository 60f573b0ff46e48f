"""The stage times of ane_ddgi_stats: counted per call, folded from either stamp set."""
import pytest

from anerend_amd import native, scenegen
from anerend_amd.types import Config

pytestmark = pytest.mark.gpu


# a streaming, a split-ray and a register-tiled convolution
@pytest.mark.parametrize("rays", [256, 704, 33])
def test_stage_clock_counts_and_folds(rays):
    ds = native.DeviceScene(scenegen.room_scene(1, num_boxes=4))
    cfg = Config.make((3, 2, 5), step=(1.0, 1.0, 1.0), rays=rays)
    grid = native.ProbeGrid(cfg)
    frame = scenegen.make_frame(1, config=cfg)
    assert not any(grid.stats()["calls"].values())
    grid.update(ds, frame)
    one = grid.stats()
    assert one["calls"] == dict(setup=1, trace=1, sungrid=0, shade=1, convolve=1, translate=0, shadow=0)
    for k, n in one["calls"].items():
        assert one["mean_ms"][k] == one["last_ms"][k]
        assert (0.0 < one["last_ms"][k] < 50.0) == bool(n)
    sums = dict(one["last_ms"])
    for n in range(2, 6):  # both stamp sets, with and without a sun grid; a read in between folds nothing twice
        grid.update(ds, frame)
        grid.convolve(frame) if n == 3 else None
        grid.translate((float(n), 0.0, 0.0))
        s = grid.stats()
        assert grid.stats() == s
        for k in ("setup", "trace", "shade"):
            sums[k] += s["last_ms"][k]
            assert s["calls"][k] == n
            assert s["mean_ms"][k] * n == pytest.approx(sums[k], rel=1e-4)
    assert s["calls"]["convolve"] == 6 and s["calls"]["translate"] == 4
    assert s["calls"]["sungrid"] == 1 and s["calls"]["shadow"] == 4
    grid.reset_stats()
    r = grid.stats()
    assert not any(r["calls"].values()) and not any(r["mean_ms"].values())
    assert r["last_ms"] == s["last_ms"]
