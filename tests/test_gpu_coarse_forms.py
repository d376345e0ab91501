"""The nearest-neighbour form of the LDS-resident coarse solve: every
segment length it is built for, levels held by one wave, odd sides, both
boundaries, against the launches per level."""
import numpy as np
import pytest

from gpaw_amd import _lib
from gpaw_amd.grid_descriptor import GridDescriptor
from gpaw_amd.poisson import FDPoissonSolver
from gpu_util import dev, host, say
from helpers import relerr

pytestmark = pytest.mark.gpu

# fine grids; the levels below them hold (in order) one wave with segments
# of 1 and 3 points, then segments of 1, 2, 3, 4, 6 and 10 points
SHAPES = [((8, 8, 8), True), ((18, 8, 10), (True, False, True)),
          ((16, 12, 20), False), ((24, 24, 24), True),
          ((24, 32, 32), (False, True, True)), ((32, 32, 32), True),
          ((24, 40, 40), True), ((40, 40, 40), False)]


def _solver(shape, pbc):
    gd = GridDescriptor(shape, np.array(shape) * 0.35, pbc)
    s = FDPoissonSolver(nn=3)
    s.set_grid_descriptor(gd)
    rho = np.random.default_rng(7).uniform(-1, 1, tuple(gd.n_c))
    if gd.pbc_c.all():
        rho -= rho.mean()
    return s, rho


def _with_lds(on, f):
    lib = _lib.load()
    _lib.check(lib.gfd_set_tuning(b'coarse_lds', on), 'tuning')
    try:
        return f()
    finally:
        lib.gfd_set_tuning(b'coarse_lds', 1)


@pytest.mark.parametrize('shape,pbc', SHAPES)
def test_cycle_matches_launches(shape, pbc):
    """Two FP64 V-cycles.  Some 60 sweeps round about 10 operations each at
    2.2e-16, so the two orders of rounding stay within 60 * 10 * 2.2e-16 =
    1.4e-13 of each other, times 3 for the growth through the levels."""
    res = []
    for on in (1, 0):
        s, rho = _solver(shape, pbc)
        phi = dev(np.zeros_like(rho))

        def cycles():
            for _ in range(2):
                s.iterate2(None, 0, phi, dev(rho))
            return host(phi)
        say('coarse form', shape, pbc, on)
        res.append(_with_lds(on, cycles))
    assert relerr(res[0], res[1]) < 4e-13


@pytest.mark.parametrize('shape,pbc', [((24, 24, 24), True),
                                       ((40, 40, 40), False),
                                       ((48, 48, 48), True)])
def test_mixed_cycles(shape, pbc):
    """The FP32 cycles (Chebyshev on the coarsest level, a 24-plane first
    level): the refinement reaches its residual in as many steps as with a
    launch per sweep (Chebyshev may save some)."""
    steps = []
    for on in (1, 0):
        s, rho = _solver(shape, pbc)
        phi = dev(np.zeros_like(rho))
        say('coarse form, mixed', shape, pbc, on)
        n, rel = _with_lds(on, lambda: s.solve_mixed(
            phi, dev(rho), 1e-10, pre=3, post=3, w0=0.8, coarse_sweeps=16))
        assert rel <= 1e-10
        steps.append(n)
    assert steps[0] <= steps[1] + 1
