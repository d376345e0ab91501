"""The split of the band contractions over the points (host code of the
library, no device calls): its work space and its choice."""
import math

import pytest

from gpaw_amd import _lib


def cost(nt, K, c):
    rounds = -(-nt * c // 256)
    return rounds * (K / c + 61.0) * (1.0 + 0.06 / rounds)


@pytest.mark.parametrize('K', [1, 63, 64, 500, 13824, 110592, 884736])
def test_work_space_and_choice(K):
    for nt in (*range(1, 40), 78, 100, 136, 255, 256, 257, 528, 1000, 2304,
               2305, 5000):
        c = _lib.load().gfd_gram_chunks(nt, K)
        # nine blocks per CU, or one chunk; four stages of 16 points each
        assert 1 <= c <= max(1, 2304 // nt)
        assert c == 1 or K / c >= 64
        top = max(1, min(2304 // nt, K // 64))
        best = min(cost(nt, K, x) for x in range(1, top + 1))
        assert math.isclose(cost(nt, K, c), best, rel_tol=1e-12)
