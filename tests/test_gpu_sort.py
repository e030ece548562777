"""The radix sort's forms (32-, 36- and 64-bit keys), tile sizes and digit
widths: results against the oracle where the key width, the number of
workgroups and the last tile's remainder change."""
import numpy as np
import pytest

import dclust
import oracle

pytestmark = pytest.mark.gpu


def _pairs(n, dim, span, eps, seed):
    # points in groups within eps of each other, spread over a box of `span`
    # cells a side, so that the key width follows from span and dim
    rng = np.random.default_rng(seed)
    c = rng.uniform(0, span - 0.6, (n // 3 + 1, dim))
    x = (c[rng.integers(0, len(c), n)] + rng.uniform(0, 0.6, (n, dim))) * eps / 2
    x[0], x[-1] = 0.0, span * eps / 2
    return x


# one workgroup and its edges; four and five groups of 32 workgroups (128 of 1024
# entries: 131072); the first sizes of 4 and 8 entries a thread
@pytest.mark.parametrize("n", [1, 2, 511, 1024, 1025, 32768, 32769, 65537, 131072, 131073, 1572863, 1572865, 3145729])
def test_sizes(devmem, n):
    eps = 0.5
    x = _pairs(n, 3, 300, eps, n)
    p = dclust.make_params(3, eps, 3, precision=dclust.FP32_GUARD)
    d_x, d_l = devmem.upload(x), devmem.alloc(4 * n)
    ref = oracle.fast_dbscan(x, eps, 3)
    with dclust.Handle(0) as h:
        for _ in range(2):
            st = h.run_device(d_x, n, p, d_l)
            assert st["n_core"] == ref[1].sum()
            assert np.array_equal(devmem.download(np.empty(n, dtype=np.int32), d_l), ref[0])


# key widths around the digit counts and the forms: 9 | 10, 18 | 19, 32 | 33,
# 36 | 37 bits and one of 60
@pytest.mark.parametrize("span,bits", [(6, 9), (8, 10), (60, 18), (68, 19), (1500, 32), (2000, 33),
                                       (3900, 36), (5000, 37), (900000, 60)])
@pytest.mark.parametrize("n", [5000, 70001])
def test_key_widths(devmem, span, bits, n):
    eps = 0.5
    x = _pairs(n, 3, span, eps, span)
    d_x, d_l = devmem.upload(x), devmem.alloc(4 * n)
    p = dclust.make_params(3, eps, 3)
    ref = oracle.fast_dbscan(x, eps, 3)
    with dclust.Handle(0) as h:
        st = h.run_device(d_x, n, p, d_l)
        assert st["key_bits"] == bits
        assert np.array_equal(devmem.download(np.empty(n, dtype=np.int32), d_l), ref[0])
        assert np.array_equal(h.core_flags(n), ref[1])


def test_batch_of_wide_keys(devmem):
    # 33 to 36 bits from the sum of the instances' key spaces
    eps = 0.5
    ns = [4097, 1, 20000, 333]
    xs = [_pairs(n, 3, 1400, eps, n) for n in ns]
    with dclust.Handle(0) as h:
        labels, errs = h.run_batched(xs, [dclust.make_params(3, eps, 3)] * 4)
        assert not np.any(errs) and 32 < h.last_stats["key_bits"] <= 36
    for x, lab in zip(xs, labels):
        assert np.array_equal(lab, oracle.fast_dbscan(x, eps, 3)[0])
