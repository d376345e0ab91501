"""One point per thread for few points: every radius on sides as short as
the radius and on ragged ones, both boundaries, apply, Jacobi, residual with
its norm, H psi - eps psi; the largest batch it takes and one grid more."""
import numpy as np
import pytest

import oracle
from gpaw_amd import _lib, bands
from gpaw_amd.fd_operators import Gradient, Laplace
from gpaw_amd.grid_descriptor import GridDescriptor
from gpu_util import dev, host, say
from helpers import rand, relerr

pytestmark = pytest.mark.gpu
TOL = 1e-13


def grid(N, pbc):
    return GridDescriptor(N, np.array(N) * 0.3, pbc)


@pytest.mark.parametrize('nn', [1, 2, 3, 4])
@pytest.mark.parametrize('N,pbc', [((4, 5, 4), True), ((9, 5, 6), False),
                                   ((7, 12, 33), (True, False, True))])
def test_passes(nn, N, pbc):
    rng = np.random.default_rng(nn)
    gd = grid(N, pbc)
    n = tuple(gd.n_c)
    say('point stencil', nn, N, pbc)
    for op in (Laplace(gd, -0.7, nn), Gradient(gd, 1, 1.0, nn)):
        a = rand(rng, (3,) + n)
        out = dev(np.zeros_like(a))
        op.apply(dev(a), out)
        ref = oracle.fd_apply(op.coef_p, op.offset_pc, gd.n_c,
                              gd.neighbor_cd, a)
        assert relerr(host(out), ref) < TOL
    op = Laplace(gd, -0.7, nn)
    f, src = rand(rng, n), rand(rng, n)
    g = dev(f.copy())
    op.relax(2, g, dev(src), 2, 0.6)
    ref = oracle.fd_relax(2, op.coef_p, op.offset_pc, gd.n_c, gd.neighbor_cd,
                          f.copy(), src, 2, 0.6)
    assert relerr(host(g), ref) < TOL
    r, df, ds = dev(np.zeros_like(f)), dev(f), dev(src)
    norm = _lib.ctypes.c_double()
    _lib.check(_lib.load().gfd_operator_residual(
        op._handle(), df.data_ptr(), ds.data_ptr(), r.data_ptr(), 1, None,
        _lib.ctypes.byref(norm), None), 'residual')
    want = oracle.fd_apply(op.coef_p, op.offset_pc, gd.n_c, gd.neighbor_cd,
                           f) - src
    assert relerr(host(r), want) < TOL
    assert abs(norm.value / (want**2).sum() - 1) < 1e-12
    psi, vt, eps = rand(rng, (3,) + n), rand(rng, n), rand(rng, (3,))
    out = dev(np.zeros_like(psi))
    bands.apply_hamiltonian(op, dev(vt), dev(psi), out, eps=dev(eps))
    want = oracle.fd_apply(op.coef_p, op.offset_pc, gd.n_c, gd.neighbor_cd,
                           psi) + (vt - eps[:, None, None, None]) * psi
    assert relerr(host(out), want) < TOL


@pytest.mark.parametrize('count', [9, 10, 14, 15])
def test_either_side_of_the_limit(count):
    """600 000 points are 9.4 grids of 40^3, 900 000 are 14.1: one point per
    thread, the direction march, full rows."""
    rng = np.random.default_rng(2)
    gd = grid((40, 40, 40), True)
    op = Laplace(gd, 1.0, 3)
    a = rand(rng, (count,) + tuple(gd.n_c))
    out = dev(np.zeros_like(a))
    op.apply(dev(a), out)
    ref = oracle.fd_apply(op.coef_p, op.offset_pc, gd.n_c, gd.neighbor_cd, a)
    assert relerr(host(out), ref) < TOL
