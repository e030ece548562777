"""Labels of large calls, written window by window: sizes around the rule and
where the window width changes, one instance and a batch."""
import numpy as np
import pytest

import dclust
import oracle

pytestmark = pytest.mark.gpu


def _pairs(n, seed):
    rng = np.random.default_rng(seed)
    c = rng.uniform(0, 4 * np.sqrt(n), (n // 3 + 1, 2))
    return c[rng.integers(0, len(c), n)] + rng.uniform(0, 0.3, (n, 2))


@pytest.mark.parametrize("n", [(1 << 21) - 1, 1 << 21, (1 << 22) + 1, (1 << 23) + 1])
def test_one_instance(devmem, n):
    x = _pairs(n, n)
    ref = oracle.fast_dbscan(x, 0.5, 3)[0]
    d_x, d_l = devmem.upload(x), devmem.alloc(4 * n)
    with dclust.Handle(0) as h:
        st = h.run_device(d_x, n, dclust.make_params(2, 0.5, 3, precision=dclust.FP32_GUARD), d_l)
    assert np.array_equal(devmem.download(np.empty(n, dtype=np.int32), d_l), ref)
    assert st["n_noise"] == np.count_nonzero(ref == 0)


def test_batch():
    ns = [1, 1500000, 70001, 640000]
    xs = [_pairs(n, n) for n in ns]
    with dclust.Handle(0) as h:
        labels, errs = h.run_batched(xs, [dclust.make_params(2, 0.5, 3)] * len(ns))
    assert not np.any(errs)
    for x, lab in zip(xs, labels):
        assert np.array_equal(lab, oracle.fast_dbscan(x, 0.5, 3)[0])


# one workgroup ranks the clusters up to 2^19 points: the last size that it
# takes and the first that it does not; a flag in the last bit of the last word
@pytest.mark.parametrize("n", [1 << 19, (1 << 19) + 1, 64 * 1000 - 1])
def test_cluster_ranks(devmem, n):
    x = np.repeat(np.arange((n + 1) // 2, dtype=np.float64), 2)[:n, None] * [1.0, 0.0]
    x = x[np.random.default_rng(n).permutation(n)]
    ref = oracle.fast_dbscan(x, 0.5, 2)[0]
    d_x, d_l = devmem.upload(x), devmem.alloc(4 * n)
    with dclust.Handle(0) as h:
        st = h.run_device(d_x, n, dclust.make_params(2, 0.5, 2), d_l)
    assert np.array_equal(devmem.download(np.empty(n, dtype=np.int32), d_l), ref)
    assert st["n_clusters"] == n // 2


def test_batch_of_many_chunks_and_instances():
    # instances of no point, one point, one chunk and more chunks than the
    # bounding box has stripes
    ns = [200000, 0, 1, 4096, 4097, 33] * 3
    xs = [_pairs(max(n, 1), 7 + n)[:n] for n in ns]
    with dclust.Handle(0) as h:
        labels, errs = h.run_batched(xs, [dclust.make_params(2, 0.5, 3)] * len(ns))
    assert not np.any(errs)
    for x, lab in zip(xs, labels):
        if len(x):
            assert np.array_equal(lab, oracle.fast_dbscan(x, 0.5, 3)[0])
