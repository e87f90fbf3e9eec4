"""The colour-ordered relax inside the tile step kernel (k_colour_step) gives
the bits of the same cascade run class by class over the whole map (the
global path's launches), where it can go wrong: axes of every residue mod 3
(the classes past 2 and their wider halo), maps smaller than a tile's
region (cells met twice across the wrap), tiles cut by the map's edge, few
and many visited cells, every tile shape, one and two layers."""
import numpy as np
import pytest

from simplewinderosion_amd import World, Wind, capi

pytestmark = pytest.mark.gpu


def _run(path, shape, nx, ny, particles, periodic, layers, seed):
    rng = np.random.default_rng(seed)
    h = (rng.random((nx, ny)) * 0.4).astype(np.float32)
    s = np.full((nx, ny), 0.004, np.float32) if layers == 2 else None
    World.SEED, World.settling, Wind.suspension, Wind.maxAge = seed, 1.0, 5e-3, 40
    w = World(nx, ny, periodic=periodic, layers=layers, abrasion=1e-3 if layers == 2 else 0.0)
    w.set_path(path)
    if shape is not None:
        w.set_tune(capi.SWE_TUNE_SHAPE, shape)
    w.upload(h, s)
    w.erode(particles, n_cycles=2)
    z, sm = w.master()
    out = dict(w.download(), z=z, sm=sm, lost=w.audit()["lost"])
    w.close()
    return out


def _same(a, b):
    for k in a:
        assert np.array_equal(a[k], b[k]), k


@pytest.mark.parametrize("nx,ny,per_cell", [
    (3, 4, 1.0), (5, 5, 1.0), (8, 14, 0.5),     # cells of a region met many times
    (16, 32, 1.0), (17, 33, 0.05), (31, 65, 1.0),
    (48, 96, 0.02), (49, 97, 0.02), (50, 98, 0.02),  # residues 0, 1, 2: few visited cells a tile
    (48, 96, 1.0), (49, 98, 1.0), (50, 97, 1.0),     # many
    (100, 131, 0.3),
])
@pytest.mark.parametrize("periodic,layers", [(True, 2), (False, 1), (True, 1), (False, 2)])
def test_tile_relax_equals_class_launches(statics, nx, ny, per_cell, periodic, layers):
    print("case colour tiles", nx, ny, per_cell, periodic, layers, flush=True)
    n = max(4, int(per_cell * nx * ny))
    _same(_run(2, None, nx, ny, n, periodic, layers, 5), _run(1, None, nx, ny, n, periodic, layers, 5))


@pytest.mark.parametrize("shape", range(5))
@pytest.mark.parametrize("periodic", [True, False])
def test_every_shape(statics, shape, periodic):
    print("case colour tiles shape", shape, periodic, flush=True)
    _same(_run(2, shape, 77, 110, 3000, periodic, 2, 9), _run(1, None, 77, 110, 3000, periodic, 2, 9))
