"""The colour-ordered relax inside the step kernel (k_colour_step) on several
terrains: each terrain's own record, cells and tiles, its classes by its own
sides mod 3, and the halo of the widest of them.  Every terrain equals the same
map eroded alone by the class launches of the global path."""
import numpy as np
import pytest

from simplewinderosion_amd import Batch, World, Wind, capi, glm_normalize

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [
    [(31, 29), (40, 17), (33, 64), (50, 98), (10, 10)],  # residues 1 2, 1 2, 0 1, 2 2, 1 1: the widest halo
    [(48, 96), (30, 33), (3, 3)],                        # all 0: the interior halo
    [(49, 97), (16, 32), (64, 18)],                      # 0 and 1
])
@pytest.mark.parametrize("periodic", [True, False])
@pytest.mark.parametrize("layers", [1, 2])
@pytest.mark.parametrize("shape", [0, 4])
def test_batch_equals_single_runs(statics, sizes, periodic, layers, shape):
    print("case colour batch fused", sizes, periodic, layers, shape, flush=True)
    World.settling, Wind.suspension, Wind.maxAge = 1.0, 5e-3, 40
    rng = np.random.default_rng(5)
    winds = [glm_normalize((np.cos(a), 0.2, np.sin(a))) for a in rng.uniform(0, 6.28, len(sizes))]
    heights = [(rng.random(sz) * 0.4).astype(np.float32) for sz in sizes]
    seds = [np.full(sz, 0.004, np.float32) if layers == 2 else None for sz in sizes]
    parts = [max(4, int(0.6 * a * b)) for a, b in sizes]
    b = Batch(sizes, periodic=periodic, layers=layers, abrasion=1e-3 if layers == 2 else 0.0)
    b.set_tune(capi.SWE_TUNE_SHAPE, shape)
    for k in range(len(sizes)):
        b.set_terrain(k, 100 + k, winds[k])
        b.upload(k, heights[k], seds[k])
    b.erode(parts, n_cycles=2)
    for k, size in enumerate(sizes):
        World.SEED, Wind.pspeed = 100 + k, winds[k]
        w = World(*size, periodic=periodic, layers=layers, abrasion=1e-3 if layers == 2 else 0.0)
        w.set_path(1)
        w.upload(heights[k], seds[k])
        w.erode(parts[k], n_cycles=2)
        zb, sb = b.master(k)
        zw, sw = w.master()
        assert np.array_equal(zb, zw), k
        if layers == 2:
            assert np.array_equal(sb, sw), k
        got, want = b.download(k), w.download()
        for key in ("massflow", "momentum"):
            assert np.array_equal(got[key], want[key]), (k, key)
        assert b.audit(k)["lost"] == w.audit()["lost"], k
        w.close()
    b.close()
