"""Tiled K = 2 restriction: coarse sides below, at and past its tiles, all
boundaries, real and complex with Bloch phases, and the narrowing form
(FP64 in, FP32 out) inside the FP32 preconditioner."""
import numpy as np
import pytest

import oracle
from gpaw_amd import _lib
from gpaw_amd.grid_descriptor import GridDescriptor
from gpaw_amd.fd_operators import Laplace
from gpaw_amd.preconditioner import Preconditioner
from gpaw_amd.transformers import Transformer
from gpu_util import dev, host, say
from helpers import bloch_phases, rand, relerr, tspec

pytestmark = pytest.mark.gpu
TOL = 1e-13


@pytest.fixture
def tiled():
    lib = _lib.load()
    lib.gfd_set_tuning(b'xfer_tile', 1)
    yield
    lib.gfd_set_tuning(b'xfer_tile', 0)


@pytest.mark.parametrize('dtype', [float, complex])
@pytest.mark.parametrize('pbc', [True, False, (True, False, True)])
@pytest.mark.parametrize('N', [(4, 6, 8), (8, 16, 64), (10, 18, 66),
                               (6, 8, 136)])
def test_against_oracle(tiled, N, pbc, dtype):
    rng = np.random.default_rng(N[2])
    fine = GridDescriptor(N, np.array(N) * 0.2, pbc)
    t = Transformer(fine, fine.coarsen(), 1, dtype)
    a = rand(rng, (3,) + tuple(fine.n_c), dtype)
    ph = bloch_phases(rng, fine.pbc_c) if dtype == complex else None
    say('tiled restriction', N, pbc, dtype.__name__)
    got = host(t.apply(dev(a), None, ph))
    s = tspec(t)
    ref = oracle.transform(s.interpolate, s.k, s.size_in, s.size_out,
                           s.pad_cd, s.npad_cd, s.skip_cd, s.neighbor_cd, a,
                           ph)
    assert relerr(got, ref) < TOL


class Kpt:
    pass


@pytest.mark.parametrize('dtype', [float, complex])
@pytest.mark.parametrize('pbc', [True, (False, True, True)])
def test_narrowing(dtype, pbc):
    """The FP32 chain with and without the tiles: both restrictions round
    each sum of 27 FP32 values (the same order of terms), so the results
    differ by rounding of the chain at most."""
    rng = np.random.default_rng(5)
    gd = GridDescriptor((24, 20, 72), np.array((24, 20, 72)) * 0.2, pbc)
    p = Preconditioner(gd, Laplace(gd, -0.5, 3, dtype), dtype, block=2,
                       fp32=True)
    kpt = Kpt()
    kpt.phase_cd = bloch_phases(rng, gd.pbc_c)
    res = dev(rand(rng, (2,) + tuple(gd.n_c), dtype))
    say('tiled narrowing restriction', dtype.__name__, pbc)
    lib = _lib.load()
    want = host(p(res, kpt))
    try:
        lib.gfd_set_tuning(b'xfer_tile', 1)
        got = host(p(res, kpt))
    finally:
        lib.gfd_set_tuning(b'xfer_tile', 0)
    assert relerr(got, want) < 1e-6
