"""root_of (csrc/swe_device.hpp): the square root and its reciprocal from
v_rsq_f32 and v_rcp_f32 seeds are the correctly rounded ones for every float,
special values and those past its guarded range included."""
import ctypes

import pytest

from simplewinderosion_amd import World

pytestmark = pytest.mark.gpu


def test_root_of_every_float():
    w = World(3, 3)
    for first in range(0, 1 << 32, 1 << 28):
        print("case root_of from %08x" % first, flush=True)
        n, bad = ctypes.c_uint64(), ctypes.c_uint32()
        assert w.lib.swe_debug_root(w.ctx, first, 1 << 28, ctypes.byref(n), ctypes.byref(bad)) == 0
        assert n.value == 0, "%d differ, the first at %08x" % (n.value, bad.value)
    w.close()
