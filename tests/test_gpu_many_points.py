"""Labels at the largest call that is written window by window (2^26 points)
and one above it: pairs of points at known places, so that the labels follow
from the numbering alone."""
import numpy as np
import pytest

import dclust

pytestmark = pytest.mark.gpu

LIMIT = 1 << 26


@pytest.mark.parametrize("n", [LIMIT, LIMIT + 1])
def test_pairs_at_the_limit_of_the_windows(devmem, n):
    # input i is point j = (a i + b) mod n; points 2g and 2g + 1 are a pair 0.1
    # apart, pairs are 1 apart, and every fifth "pair" is two lone points
    a, b, side = 38654707, 12345, 8192
    assert np.gcd(a, n) == 1
    back = pow(a, -1, n)
    j = (np.arange(n, dtype=np.int64) * a + b) % n
    g = j >> 1
    gap = np.where(g % 5 == 4, 0.5, 0.1)
    x = np.empty((n, 2))
    x[:, 0] = g % side + (j & 1) * gap
    x[:, 1] = g // side
    del gap
    d_x, d_l = devmem.upload(x), devmem.alloc(4 * n)
    del x
    groups = (n + 1) // 2
    first = np.arange(groups, dtype=np.int64) * 2
    pos = [(k - b) % n * back % n for k in (first, np.minimum(first + 1, n - 1))]
    paired = (np.arange(groups) % 5 != 4) & (first + 1 < n)
    at = np.minimum(*pos)  # the smaller input index of the pair
    mark = np.zeros(n, dtype=np.int32)
    mark[at[paired]] = 1
    rank = np.cumsum(mark, dtype=np.int32)
    want = np.where(paired, rank[at], 0)[g]
    with dclust.Handle(0) as h:
        st = h.run_device(d_x, n, dclust.make_params(2, 0.2, 2, precision=dclust.FP32_GUARD), d_l)
        assert st["n_clusters"] == int(paired.sum())
    lab = devmem.download(np.empty(n, dtype=np.int32), d_l)
    assert np.array_equal(lab, want)
