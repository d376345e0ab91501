"""Band sums split over several blocks: few bands of many points, ragged
chunks, both data types, and on either side of the lines between split and
unsplit sums."""
import numpy as np
import pytest

from gpaw_amd import bands
from gpaw_amd.rmmdiis import rmm_lambda
from gpu_util import dev, host, kernels_of, say
from helpers import rand

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('dtype', [float, complex])
@pytest.mark.parametrize('nb,n,split', [
    (1, (3, 5, 7), ''), (1, (17, 31, 33), ''), (1, (18, 31, 33), 'fc'),
    (3, (40, 41, 43), 'fc'), (30, (27, 28, 29), 'f'), (30, (34, 34, 35), 'fc'),
    (70, (34, 34, 35), 'f'), (700, (4, 5, 6), '')])
def test_split_sums(dtype, nb, n, split):
    """Sums of m products against numpy, within 2 m eps of the sum of
    their moduli."""
    rng = np.random.default_rng(nb)
    a, b = (rand(rng, (nb,) + n, dtype) for _ in range(2))
    b[0] += 0.5 * a[0]
    say('band split', dtype, nb, n)
    eps = 2 * np.prod(n) * 2.3e-16
    ab = (a.conj() * b).real.sum((1, 2, 3))
    aa = (abs(a)**2).sum((1, 2, 3))
    moduli = abs(a.conj() * b).sum((1, 2, 3))
    da, db = dev(a), dev(b)
    got, names = kernels_of(lambda: host(bands.band_dots(da, db, 0.3)))
    if names:
        assert any('k_band_split' in k for k in names) == (
            ('c' if dtype == complex else 'f') in split)
    assert (abs(got - 0.3 * ab) <= 0.3 * eps * moduli).all()
    lam = host(rmm_lambda(dev(a), dev(b)))
    assert (abs(lam + ab / aa) <= 2 * eps * moduli / aa).all()
    zero = host(rmm_lambda(dev(np.zeros_like(a)), dev(b)))
    assert (zero == 0).all()
