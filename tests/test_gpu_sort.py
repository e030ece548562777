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


# the wider forms at the first sizes of 4 and 8 entries a thread, whose last
# tiles hold one entry: 33 and 36 bits (four of them in the ids), 37 and 60
@pytest.mark.parametrize("span,bits", [(2000, 33), (3900, 36), (5000, 37), (900000, 60)])
@pytest.mark.parametrize("n", [1572865, 3145729])
def test_wide_keys_of_large_calls(devmem, span, bits, n):
    eps = 0.5
    x = _pairs(n, 3, span, eps, span)
    d_x, d_l = devmem.upload(x), devmem.alloc(4 * n)
    ref = oracle.fast_dbscan(x, eps, 3)
    with dclust.Handle(0) as h:
        st = h.run_device(d_x, n, dclust.make_params(3, eps, 3, precision=dclust.FP32_GUARD), d_l)
        assert st["key_bits"] == bits
        assert np.array_equal(devmem.download(np.empty(n, dtype=np.int32), d_l), ref[0])
        assert np.array_equal(h.core_flags(n), ref[1])


@pytest.mark.parametrize("span,lo,hi", [(1400, 33, 36), (4200, 37, 40)])
@pytest.mark.parametrize("n", [1572865, 3145729])
def test_large_batch_of_wide_keys(devmem, span, lo, hi, n):
    eps = 0.5
    ns = np.array([n - 500003, 400000, 3, 100000], dtype=np.int64)
    xs = [_pairs(k, 3, span, eps, k) for k in ns]
    d_x = devmem.upload(np.concatenate([x.ravel() for x in xs]))
    d_l = devmem.alloc(4 * n)
    with dclust.Handle(0) as h:
        assert not np.any(h.run_batched_device(d_x, ns, [dclust.make_params(3, eps, 3)] * 4, d_l))
        assert lo <= h.last_stats["key_bits"] <= hi
    lab = devmem.download(np.empty(n, dtype=np.int32), d_l)
    for x, part in zip(xs, np.split(lab, np.cumsum(ns)[:-1])):
        assert np.array_equal(part, oracle.fast_dbscan(x, eps, 3)[0])


@pytest.mark.parametrize("n", [5000, 70001])
def test_replay_widens_through_the_forms(devmem, n, monkeypatch):
    # a captured run of 32-, 36- or 64-bit keys meets a wider key: the call is
    # run again with the wider form, which then serves the narrower keys too
    monkeypatch.delenv("DCLUST_GRAPH", raising=False)
    x = _pairs(n, 3, 1500, 0.5, 1)
    d_x, d_l = devmem.upload(x), devmem.alloc(4 * n)
    seen = []
    with dclust.Handle(0) as h:
        for eps in (0.5, 0.5, 0.25, 0.25, 0.2, 0.15, 0.15, 0.01, 0.01, 0.2, 0.5):
            devmem.h2d(d_l, np.full(n, -7, dtype=np.int32))
            st = h.run_device(d_x, n, dclust.make_params(3, eps, 3), d_l)
            ref = oracle.fast_dbscan(x, eps, 3)
            assert np.array_equal(devmem.download(np.empty(n, dtype=np.int32), d_l), ref[0])
            assert np.array_equal(h.core_flags(n), ref[1])
            seen.append((st["key_bits"], st["diag"][14]))
    bits = [b for b, _ in seen]
    assert bits[0] <= 32 < bits[2] <= 36 and bits[4] <= 36 < bits[5] <= 45 < bits[7]
    assert [r for _, r in seen] == [0, 1, 0, 1, 1, 0, 1, 0, 1, 1, 1]
