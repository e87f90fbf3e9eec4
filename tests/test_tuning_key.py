"""The tuning cache's key (tuning.py): a workload's launches, so the
colour-ordered cascade, which runs another kernel with other LDS, has entries of
its own; those of the synchronous cascade keep the keys they had."""
import json

from simplewinderosion_amd import capi, tuning


class _Lib:
    def swe_device_arch(self, ctx, buf, n):
        buf.value = b"gfx950"
        return 0


class _Target:
    lib, ctx, sizes = _Lib(), None, [(64, 48)]

    def __init__(self, **kw):
        self.p = capi.SweParams(window=1, layers=2, track=1, periodic=1, max_age=512, cascade_order=-1, **kw)

    def params(self):
        return self.p

    def _check(self, rc, what):
        assert rc == 0, what


def _key(cascade_order, settling):
    t = _Target(settling=settling)
    t.p.cascade_order = cascade_order
    return tuning._key(t, [100])


def test_colour_order_has_its_own_entries():
    sync = _key(-1, 0.01)
    assert sync == _key(0, 0.25) and "cascade" not in json.loads(sync)
    assert _key(1, 0.01) != sync and _key(-1, 1.0) == _key(1, 0.01)
