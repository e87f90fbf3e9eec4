"""The colour-ordered relax inside the tile step kernel where its short
conversion of a master (heights below 128 that no transfer carries past 2^15)
does not hold: heights above 128, settling above 1, and a negative threshold,
with which a transfer exceeds half the height difference.  The oracle's bits."""
import numpy as np
import pytest

import oracle as O
from simplewinderosion_amd import World, Wind, capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("periodic,layers", [(True, 1), (False, 1), (True, 2)])
@pytest.mark.parametrize("top,settling,maxdiff", [
    (0.4, 1.0, 0.005), (127.0, 1.0, 0.005), (129.0, 1.0, 0.005), (40000.0, 1.0, 0.005), (-300.0, 1.0, 0.005),
    (0.4, 1.6, 0.005),
    (0.4, 1.0, -0.01), (0.4, 1.0, -1e5), (0.4, 1.0, -1e7),
])
def test_relax_outside_the_short_conversion(statics, top, settling, maxdiff, periodic, layers):
    print("case colour extremes", top, settling, maxdiff, periodic, layers, flush=True)
    nx, ny = 50, 61
    rng = np.random.default_rng(2)
    h = (rng.random((nx, ny)) * top).astype(np.float32)
    s = np.full((nx, ny), 0.02, np.float32) if layers == 2 else None
    World.SEED, World.settling, World.maxdiff = 11, settling, maxdiff
    Wind.suspension, Wind.maxAge = 1e-3, 3
    w = World(nx, ny, periodic=periodic, layers=layers, abrasion=1e-3 if layers == 2 else 0.0)
    w.set_path(2)
    w.upload(h, s)
    st = O.OracleState(nx, ny, h, sediment=s, params=O.params_from(w.params()))
    assert O.load().or_colour_mode(st.p) == 1
    w.erode(900)
    st.erode(900, 1)
    z, sm = w.master()
    assert np.array_equal(z.ravel(), st.zm)
    if layers == 2:
        assert np.array_equal(sm.ravel(), st.sm)
    assert w.stats()["particle_steps"] == st.steps.value
    w.close()
