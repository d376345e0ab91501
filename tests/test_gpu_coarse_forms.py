"""The nearest-neighbour form of the LDS-resident coarse solve: every
segment length it is built for, levels held by one wave, odd sides, both
boundaries, against the launches per level."""
import numpy as np
import pytest

from gpaw_amd import _lib
from gpaw_amd.grid_descriptor import GridDescriptor
from gpaw_amd.poisson import FDPoissonSolver, PoissonConvergenceError
from gpu_util import dev, host, say
from helpers import relerr

pytestmark = pytest.mark.gpu

# fine grids, and the longest segment of every level below them
SHAPES = [((8, 8, 8), True, [1, 1, 1]), ((18, 8, 10), (True, False, True), [3]),
          ((16, 12, 20), False, [1, 1]), ((24, 24, 24), True, [2, 1, 1]),
          ((24, 32, 32), (False, True, True), [3, 1, 1]),
          ((32, 32, 32), True, [4, 1, 1, 1, 1]),
          ((24, 40, 40), True, [6, 1, 2]), ((40, 40, 40), False, [10, 1, 1])]


def _solver(shape, pbc):
    gd = GridDescriptor(shape, np.array(shape) * 0.35, pbc)
    s = FDPoissonSolver(nn=3)
    s.set_grid_descriptor(gd)
    rho = np.random.default_rng(7).uniform(-1, 1, tuple(gd.n_c))
    if gd.pbc_c.all():
        rho -= rho.mean()
    return s, rho


def _with_lds(on, f, cheb=1):
    """f() with the coarse levels in one workgroup, as many as fit it, or as
    launches per sweep; the blocked half cycles, which would take the larger
    ones, are off both times."""
    lib = _lib.load()
    keys = {b'coarse_lds': on, b'tsmooth': 0, b'coarse_max_points': 14000,
            b'coarse_cheb': cheb}
    for k, v in keys.items():
        _lib.check(lib.gfd_set_tuning(k, v), 'tuning')
    try:
        return f()
    finally:
        for k, v in ((b'coarse_lds', 1), (b'tsmooth', 1),
                     (b'coarse_max_points', 0), (b'coarse_cheb', 1)):
            lib.gfd_set_tuning(k, v)


def _plan(s, which):
    """First level in the workgroup, longest segments of its levels."""
    v = (_lib.ctypes.c_int * 12)()
    n = _lib.load().gfd_poisson_coarse_plan(s._handle(), which, v, 12)
    assert n >= 2 and v[1] == (v[0] >= 0)
    return v[0], list(v[2:n])


@pytest.mark.parametrize('shape,pbc,segments', SHAPES)
def test_cycle_matches_launches(shape, pbc, segments):
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
        assert _plan(s, 0) == ((1, segments) if on else (-1, []))
    assert relerr(res[0], res[1]) < 4e-13


MIXED = [((24, 24, 24), True, [2, 1, 1]), ((40, 40, 40), False, [10, 1, 1]),
         ((48, 48, 48), True, [24, 2, 1, 1])]


@pytest.mark.parametrize('shape,pbc,segments', MIXED)
def test_mixed_cycles(shape, pbc, segments):
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
        assert _plan(s, 1) == ((1, segments) if on else (-1, []))
        steps.append(n)
    assert steps[0] <= steps[1] + 1


@pytest.mark.parametrize('pre,post', [(3, 3), (5, 5)])
@pytest.mark.parametrize('shape,pbc,segments', MIXED)
def test_mixed_steps_match_launches(shape, pbc, segments, pre, post):
    """The solution after two refinement steps, Jacobi on the coarsest level
    both times.  Some 60 sweeps (100 with five each way) round about 10 FP32
    operations each at 6e-8: 100 * 10 * 6e-8 = 6e-5 of the correction, times
    3 for the growth through the levels."""
    out = []
    for on in (1, 0):
        s, rho = _solver(shape, pbc)
        phi = dev(np.zeros_like(rho))
        say('coarse form, mixed steps', shape, pbc, pre, on)

        def steps():
            with pytest.raises(PoissonConvergenceError):
                s.solve_mixed(phi, dev(rho), 1e-30, pre=pre, post=post,
                              w0=0.8, coarse_sweeps=16, max_outer=2)
        _with_lds(on, steps, cheb=0)
        assert _plan(s, 1) == ((1, segments) if on else (-1, []))
        out.append(host(phi))
    assert relerr(out[0], out[1]) < 2e-4


def test_five_sweeps_keep_a_large_first_level():
    """With more sweeps than the blocked half cycles have, the workgroup
    starts at the 24-plane level by default; with fewer they take it."""
    s, rho = _solver((48, 48, 48), True)
    for sweeps, plan in ((5, (1, [24])), (4, (2, [2])), (5, (1, [24]))):
        phi = dev(np.zeros_like(rho))
        s.solve_mixed(phi, dev(rho), 1e-10, pre=sweeps, post=sweeps, w0=0.8,
                      coarse_sweeps=16)
        lc, segments = _plan(s, 1)
        assert (lc, segments[:1]) == plan
