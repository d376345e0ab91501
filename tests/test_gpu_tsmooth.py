"""Blocked half cycles (sweeps, residual and restriction; interpolation and
sweeps, one launch each) against the separate launches: tile remainders,
grids smaller than a tile's halo, both boundaries, every sweep count."""
import numpy as np
import pytest

from gpaw_amd import _lib
from gpaw_amd.batch_poisson import BatchedPoissonSolver
from gpaw_amd.grid_descriptor import GridDescriptor
from gpaw_amd.poisson import FDPoissonSolver, PoissonConvergenceError
from gpu_util import dev, host, kernels_of, say
from helpers import relerr

pytestmark = pytest.mark.gpu


def _tuned(on, f):
    """f() with the blocked half cycles on or off; the LDS-resident coarse
    solve is off, so that every level below the finest takes part."""
    lib = _lib.load()
    _lib.check(lib.gfd_set_tuning(b'tsmooth', on), 'tsmooth')
    _lib.check(lib.gfd_set_tuning(b'coarse_lds', 0), 'coarse_lds')
    try:
        return f()
    finally:
        lib.gfd_set_tuning(b'tsmooth', 1)
        lib.gfd_set_tuning(b'coarse_lds', 1)


def _solver(shape, pbc):
    gd = GridDescriptor(shape, np.array(shape) * 0.35, pbc)
    s = FDPoissonSolver(nn=3)
    s.set_grid_descriptor(gd)
    rho = np.random.default_rng(3).uniform(-1, 1, tuple(gd.n_c))
    if gd.pbc_c.all():
        rho -= rho.mean()
    return s, rho


SHAPES = [((16, 16, 16), True), ((32, 24, 40), False),
          ((48, 32, 24), (True, False, True)), ((40, 56, 72), True),
          ((56, 40, 48), (False, False, True))]


@pytest.mark.parametrize('shape,pbc', SHAPES)
def test_cycle_matches_launches(shape, pbc):
    """Two FP64 V-cycles of the reference schedule (4 sweeps each way).
    Some 60 sweeps round about 10 operations each at 2.2e-16 (1.4e-13),
    times 3 for the growth through the levels."""
    res = []
    for on in (1, 0):
        s, rho = _solver(shape, pbc)
        phi = dev(np.zeros_like(rho))

        def cycles():
            for _ in range(2):
                s.iterate2(None, 0, phi, dev(rho))
            return host(phi)
        say('blocked smoothing', shape, pbc, on)
        res.append(_tuned(on, cycles))
    assert relerr(res[0], res[1]) < 4e-13


@pytest.mark.parametrize('pre,post', [(1, 1), (2, 3), (3, 4), (4, 2)])
@pytest.mark.parametrize('fp64', [False, True])
def test_sweep_counts(pre, post, fp64):
    """The refinement with every number of sweeps, in FP32 and FP64: the
    same solution (residual 1e-10) in as many steps."""
    out = []
    for on in (1, 0):
        s, rho = _solver((40, 32, 48), (True, False, True))
        phi = dev(np.zeros_like(rho))
        say('blocked smoothing', pre, post, fp64, on)
        n, rel = _tuned(on, lambda: s.solve_mixed(
            phi, dev(rho), 1e-10, pre=pre, post=post, w0=0.8,
            coarse_sweeps=24, fp64_inner=fp64, max_outer=200))
        assert rel <= 1e-10
        out.append((n, host(phi)))
    assert abs(out[0][0] - out[1][0]) <= 1
    # the solutions differ by their residuals: 1e-10 times the condition
    # number of this operator (some 1e3) at most
    assert relerr(out[0][1], out[1][1]) < 1e-7


def test_batched():
    """Uneven grids of both boundaries in one launch, and the switch taking
    effect on a solver that has already captured its step: two refinement
    steps by graph replays run the kernels of the setting and equal the eager
    ones bit for bit, and the two settings agree to the FP32 rounding of some
    60 sweeps of 10 operations in each cycle (60 * 10 * 6e-8 = 4e-5, times
    3)."""
    grids = [((24, 32, 40), True), ((40, 24, 16), False), ((16, 16, 16), True),
             ((32, 56, 24), (True, False, True)), ((48, 40, 72), False)]
    gds = [GridDescriptor(n, np.array(n) * 0.35, p) for n, p in grids]
    solver = BatchedPoissonSolver(nn=3)
    solver.set_grid_descriptors(gds)
    rng = np.random.default_rng(4)
    rhos = []
    for gd in gds:
        rho = rng.uniform(-1, 1, tuple(gd.n_c))
        rhos.append(dev(rho - rho.mean() if gd.pbc_c.all() else rho))

    def steps(on, graph):
        lib = _lib.load()
        _lib.check(lib.gfd_set_tuning(b'tsmooth', on), 'tsmooth')
        try:
            phis = [dev(np.zeros(tuple(gd.n_c))) for gd in gds]
            with pytest.raises(PoissonConvergenceError):
                solver.solve_mixed(phis, rhos, 1e-30, max_outer=2,
                                   graph=graph)
            return [host(p) for p in phis]
        finally:
            lib.gfd_set_tuning(b'tsmooth', 1)

    want = {}
    for on in (1, 0, 1):
        say('blocked smoothing, batched', on)
        got, names = kernels_of(lambda: steps(on, True))
        if names:
            assert any('k_tsmooth' in k for k in names) == bool(on)
        want[on] = steps(on, False)
        for a, b in zip(got, want[on]):
            assert (a == b).all()
    for a, b in zip(want[0], want[1]):
        assert relerr(a, b) < 1.2e-4
