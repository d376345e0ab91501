"""Tiles of the direction march (host code of the library, no device calls):
every grid it takes has one that its kernel can run."""
import ctypes
import itertools

import numpy as np
import pytest

from gpaw_amd import _lib


def axis_stencil(R):
    """Coefficients and offsets of an axis stencil of radius R."""
    off = [(0, 0, 0)]
    for c in range(3):
        for k in range(1, R + 1):
            for s in (k, -k):
                o = [0, 0, 0]
                o[c] = s
                off.append(tuple(o))
    return [-6.0] + [1.0] * (len(off) - 1), off


def march_tile(coef, off, n, dtype, nin=1, plain=1):
    coef = np.array(coef, float)
    off = np.array(off, np.int32)
    tile = (ctypes.c_int * 4)()
    st = _lib.load().gfd_march_tile(
        len(coef), coef.ctypes.data_as(_lib._dp),
        off.ctypes.data_as(_lib._ip), (ctypes.c_int * 3)(*n), dtype, nin,
        plain, tile)
    return st, list(tile)


@pytest.mark.parametrize('line', [None, 0, 1, 2])
@pytest.mark.parametrize('R', [1, 2, 3, 4])
def test_every_plane_has_a_tile(R, line):
    """Laplacians; gradients, whose halo is along their axis only."""
    coef, off = axis_stencil(R)
    hy, hz = (R if line in (None, c) else 0 for c in (1, 2))
    if line is not None:
        off = [o for o in off if o[line]]
        coef = [1.0] * len(off)
    sides = [s for s in [*range(1, 34), 63, 64, 65, 100, 511, 512, 513,
                         1025, 4099] if s >= R]
    for n1, n2 in itertools.product(sides, sides):
        for n0, nin, dtype, plain in ((R, 1, 0, 1), (40, 1, 1, 1),
                                      (8, 300, 1, 1), (8, 3, 1, 0)):
            st, (tz, ty, xchunk, threads) = march_tile(
                coef, off, (n0, n1, n2), dtype, nin, plain)
            assert st == _lib.GFD_OK, (n0, n1, n2)
            assert 1 <= tz <= n2 and 1 <= ty <= n1 and xchunk >= 1
            assert threads % 64 == 0 and 64 <= threads <= 512
            # one thread per point, four staged points per thread at most
            assert tz * ty <= threads, (n1, n2)
            wz, wy = (hz, hy) if plain else (R, R)
            assert (tz + 2 * wz) * (ty + 2 * wy) <= 4 * threads, (n1, n2)


def test_sides_below_the_radius_are_refused():
    coef, off = axis_stencil(3)
    for n in ((2, 8, 8), (8, 2, 8), (8, 8, 2), (8, 4000, 1)):
        assert march_tile(coef, off, n, 0)[0] == _lib.GFD_ENOTSUP
