"""A terrain's seed and wind are data of the captured cycle, not part of it:
changing them between calls replays the graph.  A replay's issue takes the host
a fraction of a capture's (514 launches recorded and instantiated)."""
import time

import numpy as np
import pytest

from simplewinderosion_amd import Batch, World, Wind, capi, glm_normalize

pytestmark = pytest.mark.gpu


def _issue(b, parts, before):
    """median host time of an erode call (it returns before the GPU is done)"""
    out = []
    for i in range(9):
        before(i)
        b.synchronize()
        t = time.perf_counter()
        b.erode(parts)
        out.append(time.perf_counter() - t)
    b.synchronize()
    return sorted(out)[4]


@pytest.mark.parametrize("sizes", [[(64, 64)], [(64, 64), (48, 80)]])
def test_terrain_changes_replay_the_graph(statics, sizes):
    print("case graph terrain", sizes, flush=True)
    World.settling, Wind.suspension = 0.01, 1e-4
    b = Batch(sizes, periodic=True)
    for k, size in enumerate(sizes):
        b.upload(k, np.random.default_rng(k).random(size).astype(np.float32))
        b.set_terrain(k, 7 + k, glm_normalize((1.0, 0.0, 1.0)))
    parts = [500] * len(sizes)
    b.erode(parts, n_cycles=2)
    same = _issue(b, parts, lambda i: None)
    changed = _issue(b, parts, lambda i: b.set_terrain(0, 100 + i, glm_normalize((1.0, 0.0, 0.1 * i))))
    capture = _issue(b, parts, lambda i: b.set_tune(capi.SWE_TUNE_TILE_ORDER, i % 4 + 1))
    print("issue us: same %.0f changed %.0f capture %.0f" % (1e6 * same, 1e6 * changed, 1e6 * capture), flush=True)
    assert changed - same < 0.5 * (capture - same)
    b.close()


def test_one_terrain_with_and_without_its_own_wind(statics):
    """A batch of one terrain equals the map: first with the batch's seed and
    wind, then with its own (which the captured cycle reads from memory)."""
    print("case graph terrain, one", flush=True)
    World.settling, Wind.suspension = 0.01, 1e-3
    World.SEED = 3
    h = np.random.default_rng(4).random((50, 70)).astype(np.float32)
    b = Batch([(50, 70)], periodic=True)
    w = World(50, 70, periodic=True)
    b.upload(0, h)
    w.upload(h)
    for seed in (3, 8, 9, 9):
        if seed != 3:
            World.SEED, Wind.pspeed = seed, glm_normalize((0.3, 0.0, float(seed)))
            b.set_terrain(0, seed, Wind.pspeed)
        b.erode([900], n_cycles=2)
        w.erode(900, n_cycles=2)
        assert np.array_equal(b.master(0)[0], w.master()[0]), seed
    b.close()
    w.close()
