"""swe_autotune's result is the setting its fastest trial ran: on a map of one
round of workgroups, whose default lists no tiles, the reported
SWE_TUNE_HEAVY_FIRST mode set again lists what the tuned context lists."""
import numpy as np
import pytest

from simplewinderosion_amd import World, Wind, capi

pytestmark = pytest.mark.gpu


def test_autotune_reports_the_mode_it_timed(statics):
    print("case autotune heavy", flush=True)
    World.SEED, World.settling, Wind.suspension, Wind.maxAge = 4, 0.01, 1e-3, 60
    w = World(640, 640, periodic=True)  # 800 tiles of 16 x 32, every one of them light
    w.upload((np.random.default_rng(1).random((640, 640)) * 0.3).astype(np.float32))
    for _ in range(10):
        r = w.autotune(20000, trial_cycles=2, cache=None)
        w.lib.swe_reset_stats(w.ctx)
        w.erode(20000)
        assert (w.stats()["light_tile_windows"] > 0) == (r["heavy_first"] == 2), r
        assert w.get_tune(capi.SWE_TUNE_HEAVY_FIRST) == r["heavy_first"]
    w.close()
