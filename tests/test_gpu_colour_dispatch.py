"""The tile path's class launches (maps of many rounds of tiles, where
colour_fused prefers them to the relax inside the step kernel) give the bits of
the global path, alone, in a batch, and where the particle count moves a map
from one way to the other between cycles."""
import numpy as np
import pytest

from simplewinderosion_amd import Batch, World, Wind, capi

pytestmark = pytest.mark.gpu


def _inputs(nx, ny, layers):
    rng = np.random.default_rng(3)
    return (rng.random((nx, ny)) * 0.4).astype(np.float32), (
        np.full((nx, ny), 0.004, np.float32) if layers == 2 else None)


@pytest.mark.parametrize("nx,ny,periodic,layers,counts", [
    (641, 640, False, 2, [200000]),              # 16 x 16 tiles: 1.6 rounds, 9 classes: class launches
    (642, 639, True, 2, [200000, 9000, 200000]),  # 9 classes; few particles: inside the step kernel
    (640, 641, True, 1, [9000, 200000]),
])
def test_large_maps_equal_the_global_path(statics, nx, ny, periodic, layers, counts):
    print("case colour dispatch", nx, ny, periodic, layers, counts, flush=True)
    World.SEED, World.settling, Wind.suspension, Wind.maxAge = 5, 1.0, 5e-3, 6
    h, s = _inputs(nx, ny, layers)
    out = []
    for path in (2, 1):
        w = World(nx, ny, periodic=periodic, layers=layers, abrasion=1e-3 if layers == 2 else 0.0)
        w.set_path(path)
        w.set_tune(capi.SWE_TUNE_SHAPE, 2)
        w.upload(h, s)
        for n in counts:
            w.erode(n, n_cycles=2)
        out.append(dict(w.download(), z=w.master()[0], sm=w.master()[1], lost=w.audit()["lost"],
                        steps=w.stats()["particle_steps"]))
        w.close()
    for k in out[0]:
        assert np.array_equal(out[0][k], out[1][k]), k


@pytest.mark.parametrize("periodic", [True, False])
def test_large_batch_equals_single_runs(statics, periodic):
    print("case colour dispatch batch", periodic, flush=True)
    World.SEED, World.settling, Wind.suspension, Wind.maxAge = 5, 1.0, 5e-3, 6
    sizes = [(513, 512), (300, 405), (258, 511), (96, 33)]
    parts = [int(0.5 * a * b) for a, b in sizes]
    b = Batch(sizes, periodic=periodic, layers=2, abrasion=1e-3)
    b.set_tune(capi.SWE_TUNE_SHAPE, 2)
    for k, size in enumerate(sizes):
        b.set_terrain(k, 5 + k, Wind.pspeed)
        b.upload(k, *_inputs(*size, 2))
    b.erode(parts, n_cycles=2)
    for k, size in enumerate(sizes):
        World.SEED = 5 + k
        w = World(*size, periodic=periodic, layers=2, abrasion=1e-3)
        w.set_path(1)
        w.upload(*_inputs(*size, 2))
        w.erode(parts[k], n_cycles=2)
        for x, y in zip(b.master(k), w.master()):
            assert np.array_equal(x, y), k
        w.close()
    b.close()
