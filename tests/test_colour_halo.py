"""The halo the tile step kernel loads for the colour-ordered relax
(csrc/swe_step.h, colour_halo) covers every cell the result can depend on:
the dependence set of a cell, run backwards through the colour classes with
every cell visited, on the unrolled periodic map."""
import os
import re

import numpy as np
import pytest

from simplewinderosion_amd import build as B

AX, AY = 12, 40  # half widths of the window the sets are followed in


def _halos():
    text = open(os.path.join(B.CSRC, "swe_step.h")).read()
    return {name: tuple(int(v) for v in re.search(r"%s = \{([^}]*)\}" % name, text).group(1).split(","))
            for name in ("kColourHalo", "kColourHaloSeam", "kColourHaloMax")}


def _classes(x, n, periodic):
    x = x % n if periodic else x
    lim = n - n % 3 if periodic else n
    return np.where(x < lim, x % 3, 3 + x - lim)


def _grow(s):
    for ax in (0, 1):
        t = s.copy()
        lo, hi = [slice(None)] * 2, [slice(None)] * 2
        lo[ax], hi[ax] = slice(1, None), slice(None, -1)
        t[tuple(lo)] |= s[tuple(hi)]
        t[tuple(hi)] |= s[tuple(lo)]
        s = t
    return s


def _extent(px, py, nx, ny, periodic):
    """(-x, +x, -y, +y) reach of the cells that cell (px, py) depends on."""
    c = (_classes(np.arange(px - AX, px + AX + 1), nx, periodic)[:, None] * 5
         + _classes(np.arange(py - AY, py + AY + 1), ny, periodic)[None, :])
    s = np.zeros(c.shape, bool)
    s[AX, AY] = True
    for k in sorted(np.unique(c))[::-1]:
        s |= _grow(_grow(s) & (c == k))
    xs, ys = np.nonzero(s)
    return AX - xs.min(), xs.max() - AX, AY - ys.min(), ys.max() - AY


def _seam(p, n, lo, hi):
    """the cells p - lo .. p + hi meet one of the last n mod 3 cells of a period"""
    return any((p + d) % n >= n - n % 3 for d in range(-lo, hi + 1))


SIZES = [(3, 4), (4, 5), (5, 5), (5, 14), (8, 8), (14, 14), (11, 4), (16, 16), (16, 61), (18, 19), (22, 25), (25, 62),
         (26, 61), (26, 62), (24, 61), (25, 60), (30, 90)]


@pytest.mark.parametrize("nx,ny", SIZES)
def test_halo_covers_the_dependences(nx, ny):
    h = _halos()
    r = (nx % 3, ny % 3)
    if r == (0, 0):
        wide = h["kColourHalo"]
    elif max(r) <= 1 and min(nx, ny) >= 16:
        wide = h["kColourHaloSeam"]
    else:
        wide = h["kColourHaloMax"]
    for px in range(nx):
        for py in range(ny):
            ext = np.array(_extent(px, py, nx, ny, True)) + 1  # a tile also keeps its one-cell halo
            near = (r[0] and _seam(px, nx, wide[0], wide[1])) or (r[1] and _seam(py, ny, wide[2], wide[3]))
            assert np.all(ext <= (wide if near else h["kColourHalo"])), (px, py, ext)


def test_interior_halo_on_a_bounded_map():
    h = _halos()
    for px in range(30, 33):
        for py in range(60, 63):
            assert np.all(np.array(_extent(px, py, 3000, 3000, False)) + 1 <= h["kColourHalo"])
