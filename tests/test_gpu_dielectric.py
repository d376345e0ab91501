"""The dielectric march (ring of staged planes) at its tile edges against
the oracle: rows of one and several parts, more and fewer staged elements
per thread, x chunks shorter than the ring, every radius, both data types,
Jacobi sweeps."""
import numpy as np
import pytest

import oracle
from gpaw_amd.fd_operators import Gradient, Laplace
from gpaw_amd.grid_descriptor import GridDescriptor
from gpaw_amd.wfd_operators import WeightedFDOperator
from gpu_util import dev, host, say
from helpers import bloch_phases, rand, relerr

pytestmark = pytest.mark.gpu
TOL = 1e-13


def build(N, pbc, nn, dtype):
    gd = GridDescriptor(N, np.array(N) * 0.3, pbc)
    op = WeightedFDOperator([Laplace(gd, 1.0, nn, dtype)] + [
        Gradient(gd, v, 1.0, nn, dtype) for v in range(3)])
    rng = np.random.default_rng(nn)
    w = [rng.uniform(1, 3, tuple(gd.n_c))] + [
        rng.uniform(-1, 1, tuple(gd.n_c)) for _ in range(3)]
    op.set_weights([dev(x) for x in w])
    return gd, op, w, rng


@pytest.mark.parametrize('N,pbc,count', [
    ((6, 5, 7), True, 2), ((13, 9, 65), False, 3),
    ((7, 66, 64), (True, False, True), 1),
    ((31, 12, 129), (False, True, False), 2)])
@pytest.mark.parametrize('nn', [1, 2, 3])
@pytest.mark.parametrize('dtype', [float, complex])
def test_apply(N, pbc, count, nn, dtype):
    gd, op, w, rng = build(N, pbc, nn, dtype)
    a = rand(rng, (count,) + tuple(gd.n_c), dtype)
    ph = bloch_phases(rng, gd.pbc_c) if dtype == complex else None
    out = dev(np.zeros_like(a))
    say('dielectric', N, pbc, nn, dtype)
    op.apply(dev(a), out, ph)
    ref = oracle.wfd_apply(op.coef_ps, op.offset_pcs, np.array(w), gd.n_c,
                           gd.neighbor_cd, a, ph)
    assert relerr(host(out), ref) < TOL


@pytest.mark.parametrize('N,pbc', [((8, 7, 9), True), ((14, 21, 66), False)])
def test_relax(N, pbc):
    gd, op, w, rng = build(N, pbc, 3, float)
    f, src = rand(rng, tuple(gd.n_c)), rand(rng, tuple(gd.n_c))
    g = dev(f.copy())
    say('dielectric relax', N, pbc)
    op.relax(2, g, dev(src), 3, 0.7)
    ref = oracle.wfd_relax(2, op.coef_ps, op.offset_pcs, np.array(w), gd.n_c,
                           gd.neighbor_cd, f.copy(), src, 3, 0.7)
    assert relerr(host(g), ref) < TOL
