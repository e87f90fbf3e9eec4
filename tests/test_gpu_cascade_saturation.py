"""World::cascade's transfers at the ends of the fixed point's range: an
amount of 2^31 or more saturates in magnitude, with the sign it is given
after (the giver's loss equals the taker's gain), as the oracle has it."""
import ctypes

import numpy as np
import pytest

import oracle as O
from simplewinderosion_amd import World

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("settling", [0.2, 1.0, 3.0])  # 3: a negative factor at two events
@pytest.mark.parametrize("maxdiff", [-3e38, -4e9, -1e9, 0.005])
@pytest.mark.parametrize("periodic", [False, True])
def test_transfers_saturate_as_the_oracle(statics, settling, maxdiff, periodic):
    print("case cascade saturation", settling, maxdiff, periodic, flush=True)
    nx, ny = 9, 7
    World.settling, World.maxdiff = settling, maxdiff
    rng = np.random.default_rng(6)
    w = World(nx, ny, periodic=periodic)
    w.upload((rng.standard_normal((nx, ny)) * 1.5e9).clip(-2.1e9, 2.1e9).astype(np.float32))
    S = np.ascontiguousarray(w.download()["height"], np.float32)
    op = O.params_from(w.params())
    i64 = ctypes.POINTER(ctypes.c_int64)
    for x, y in ((0, 0), (4, 3), (8, 6), (2, 5), (6, 1)):
        for events in (1, 2, 3):
            nbc, nbf = np.zeros(8, np.int64), np.zeros(8, np.int64)
            n = O.load().or_cascade_cell(S.ravel().ctypes.data_as(ctypes.POINTER(ctypes.c_float)), None, nx, ny,
                                         ctypes.byref(op), x, y, events, nbc.ctypes.data_as(i64),
                                         nbf.ctypes.data_as(i64))
            assert w.debug_cascade(x, y, events) == [(int(nbc[i]), int(nbf[i])) for i in range(n)], (x, y, events)
    w.close()
