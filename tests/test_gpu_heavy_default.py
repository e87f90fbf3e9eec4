"""The default of SWE_TUNE_HEAVY_FIRST by a call's load: no lists where one
round of workgroups holds the map, only crowded tiles where the mean load is at
most 1.5 times a light tile's, crowded and light ones above; a mode that is
set is obeyed.  The same bits whichever."""
import numpy as np
import pytest

from simplewinderosion_amd import Batch, World, Wind, capi

pytestmark = pytest.mark.gpu


def _run(total, mode, nx=864):
    """Two terrains of nx x 448 cells: the first holds 1000 particles (every
    tile of it is light), the second the rest."""
    World.SEED, World.settling, Wind.suspension, Wind.maxAge = 4, 0.01, 1e-3, 6
    b = Batch([(nx, 448)] * 2, periodic=True)
    if mode is not None:
        b.set_tune(capi.SWE_TUNE_HEAVY_FIRST, mode)
    for k in range(2):
        b.upload(k, (np.random.default_rng(k).random((nx, 448)) * 0.3).astype(np.float32))
    b.erode([1000, total - 1000])
    out = b.master(0)[0], b.master(1)[0], b.stats()
    b.close()
    return out


@pytest.mark.parametrize("total,light", [(100000, False), (1512 * 384, False), (1512 * 384 + 1, True)])
def test_default_follows_the_load(statics, total, light):
    """2 x 54 x 14 tiles, more than the 1280 of one round"""
    print("case heavy default", total, flush=True)
    za, zb, s = _run(total, None)
    assert (s["light_tile_windows"] > 0) == light
    za2, zb2, s2 = _run(total, 2)
    assert s2["light_tile_windows"] > 0
    assert np.array_equal(za, za2) and np.array_equal(zb, zb2)


def test_one_round_lists_nothing(statics):
    print("case heavy default, one round", flush=True)
    *_, s = _run(1260 * 512, None, nx=720)  # 2 x 45 x 14 tiles
    assert s["light_tile_windows"] == 0 and s["heavy_tile_windows"] == 0
