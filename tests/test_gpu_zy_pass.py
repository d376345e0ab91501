"""Separable transfers (z and y passes in one launch or in one each, then x):
rows of one, several and ragged column tiles, row tiles with remainders, sides shorter
than the stencil, both directions, all boundaries, real and complex."""
import numpy as np
import pytest

import oracle
from gpaw_amd import _lib
from gpaw_amd.grid_descriptor import GridDescriptor
from gpaw_amd.transformers import Transformer
from gpu_util import dev, host, kernels_of, say
from helpers import bloch_phases, rand, relerr, tspec

pytestmark = pytest.mark.gpu
TOL = 1e-13


@pytest.mark.parametrize('dtype', [float, complex])
@pytest.mark.parametrize('nn', [2, 3, 4])
@pytest.mark.parametrize('N', [(8, 8, 8), (16, 36, 134), (8, 70, 262),
                               (30, 60, 8)])
def test_against_oracle(N, nn, dtype):
    rng = np.random.default_rng(nn)
    for pbc in [True, False, (True, False, True)]:
        fine = GridDescriptor(N, np.array(N) * 0.2, pbc)
        coarse = fine.coarsen()
        for gin, gout in ((fine, coarse), (coarse, fine)):
            try:
                t = Transformer(gin, gout, nn, dtype)
            except ValueError:
                continue
            a = rand(rng, (2,) + tuple(gin.n_c), dtype)
            ph = bloch_phases(rng, gin.pbc_c) if dtype == complex else None
            say('zy pass', N, nn, pbc, gin is coarse, dtype.__name__)
            lib, out = _lib.load(), []
            try:
                for passes in (1, 2):
                    lib.gfd_set_tuning(b'xfer_passes', passes)
                    x = dev(a)
                    y, names = kernels_of(lambda: t.apply(x, None, ph))
                    if names:
                        assert any('k_xfer_zy' in k for k in names) == (
                            passes == 1)
                    out.append(host(y))
            finally:
                lib.gfd_set_tuning(b'xfer_passes', 0)
            got = out[0]
            assert (got == out[1]).all()   # the same 1-D sums
            s = tspec(t)
            ref = oracle.transform(s.interpolate, s.k, s.size_in, s.size_out,
                                   s.pad_cd, s.npad_cd, s.skip_cd,
                                   s.neighbor_cd, a, ph)
            assert relerr(got, ref) < TOL
