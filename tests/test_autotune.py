"""The raster autotuner on a stand-in context: one configuration of every tile
size is timed, a knob leaves its default only for a clear gain, settings that
the frame cannot use are skipped, and entries written before a knob was dropped
still apply."""
import json

import pytest

from softlight_amd import api as A
from softlight_amd import autotune

TILES = [(32, 16, 1), (32, 8, 2), (16, 16, 1), (16, 8, 2), (16, 8, 4), (16, 16, 4), (32, 16, 4), (32, 32, 2), (32, 8, 4),
         (32, 8, 8), (8, 8, 2), (64, 64, 1)]


class Ctx:
    """Frame times by knob: the tile's index, then the occupancy cap, then the split."""

    def __init__(self, times):
        self.times, self.knobs, self.tried = times, {"config": 0, "wg": 0, "split": autotune.SPLIT_DEFAULT}, []

    def raster_config(self, cfg=-1):
        cfg = self.knobs["config"] if cfg == -1 else cfg
        return (cfg, TILES[cfg]) if cfg < len(TILES) else (0, TILES[0])

    def set_raster_config(self, cfg):
        self.knobs["config"] = cfg

    def set_raster_occupancy(self, wg):
        self.knobs["wg"] = wg

    def set_raster_split(self, n):
        self.knobs["split"] = n

    def reset_stats(self):
        pass

    def frame(self):
        self.tried.append(dict(self.knobs))
        if self.knobs["config"] == 10:
            raise A.SLError("too many tiles")

    def stats(self):
        ms = self.times(self.knobs)
        return {"frames": 1, "ms_raster": ms, "ms_total": ms}


def test_tile_sizes_once_and_defaults_kept(tmp_path):
    ctx = Ctx(lambda k: {2: 0.5}.get(k["config"], 1.0) * (0.99 if k["wg"] == 4 else 1.0) * (0.99 if k["split"] == 0 else 1.0))
    path = str(tmp_path / "cache.json")
    res = autotune.tune(ctx, ctx.frame, "w", frames=1, path=path)
    assert sorted(res["timings"]["config"]) == [0, 1, 2, 3, 7, 10, 11]
    assert "unsupported" in res["timings"]["config"][10]
    assert (res["config"], res["wg_per_cu"], res["split"]) == (2, 0, autotune.SPLIT_DEFAULT)
    assert ctx.knobs == {"config": 2, "wg": 0, "split": autotune.SPLIT_DEFAULT}
    assert autotune.cached_entry("w", path)["config"] == 2


def test_clear_gains_taken():
    ctx = Ctx(lambda k: (0.5 if k["wg"] == 8 else 1.0) * (0.9 if k["split"] == 256 else 1.0))
    res = autotune.tune(ctx, ctx.frame, "w", frames=1, path=None)
    assert (res["wg_per_cu"], res["split"]) == (8, 256)
    assert res["frame_ms"] == pytest.approx(0.45)


def test_entry_of_an_earlier_cache(tmp_path):
    path = tmp_path / "cache.json"
    path.write_text(json.dumps({"gfx950": {"w": {"config": 6, "tile": [32, 16, 4], "depth_reject": True}}}))
    ctx = Ctx(lambda k: 1.0)
    entry = autotune.cached_entry("w", str(path))
    autotune.apply(ctx, entry)
    assert ctx.knobs == {"config": 6, "wg": 0, "split": autotune.SPLIT_DEFAULT}
    assert "depth_reject" not in autotune.describe(entry)
