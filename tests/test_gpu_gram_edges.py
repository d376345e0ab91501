"""Edges of the band contractions' tiles: band counts around the 16-band
sub-tiles and the 128-band tile, point counts around the 16-point stage and
the two-stage pipeline (one stage, a ragged second or third one)."""
import numpy as np
import pytest

from gpaw_amd import bands
from gpu_util import dev, host, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('nb', [1, 15, 17, 127, 129, 145])
@pytest.mark.parametrize('shape', [(1, 2, 3), (4, 4, 1), (3, 5, 2),
                                   (7, 5, 9)])
def test_overlap_and_rotation_edges(nb, shape):
    """Entries of O(1) data: sums of `npts` (rotation: `nb`) products round
    by at most that many times 2 eps of the sum of their moduli."""
    import torch
    rng = np.random.default_rng(nb)
    npts = int(np.prod(shape))

    def random(*s):
        return rng.uniform(-1, 1, s) + 1j * rng.uniform(-1, 1, s)
    a, b = random(nb, npts), random(nb, npts)
    psi, hpsi = (dev(x.reshape((nb,) + shape)) for x in (a, b))
    say('gram edges', nb, shape)
    eps = 2.0 * np.finfo(float).eps * 2.0
    S = host(bands.overlap(psi, 0.5, True))
    want = 0.5 * a @ a.conj().T
    i, j = np.indices((nb, nb))
    kept = j // 128 <= i // 128           # the lower tiles, whole
    assert np.abs(S - want)[kept].max() < eps * npts
    Hm = host(bands.subspace_matrix(psi, hpsi, 0.5))
    assert np.abs(Hm - 0.5 * a.conj() @ b.T).max() < eps * npts
    # rotation by a lower triangle: orthonormalize with S given through psi
    # needs npts >= nb; the dense rotation takes any Hermitian matrix
    M = random(nb, nb)
    M = M + M.conj().T
    V = dev(M)
    e, out = bands.subspace_diagonalize(V, psi)
    v = host(V)
    assert np.abs(host(out).reshape(nb, npts) - v @ a).max() < \
        eps * nb * np.abs(v).sum(1).max()
    if npts >= 2 * nb:
        out, C = bands.orthonormalize(psi, 0.5)
        o = host(out).reshape(nb, npts)
        want = np.tril(host(C)) @ a
        assert np.abs(o - want).max() < \
            eps * nb * np.abs(np.tril(host(C))).sum(1).max()
    torch.cuda.synchronize()
