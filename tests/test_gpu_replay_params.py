"""A captured run is replayed for calls of the same sizes whatever their eps
and minpts; a call that needs a wider key or more columns than the graph holds
runs eagerly, with the same result.  The sizes lie at the edges of the 64-bit
flag words, the 4096-point chunks and the 65536-point rank blocks."""
import numpy as np
import pytest

import dclust
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [dclust.FP64, dclust.FP32_GUARD])
@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("n", [63, 64, 65, 4096, 4097, 65536, 65537])
def test_replay_follows_the_parameters(devmem, prec, dim, n, monkeypatch):
    monkeypatch.delenv("DCLUST_GRAPH", raising=False)
    rng = np.random.default_rng(n + dim)
    c = rng.uniform(0, 1, (max(6, n // 100), dim))
    x = c[rng.integers(0, len(c), n)] + rng.normal(0, 2e-4, (n, dim))
    x[0], x[-1] = 0.0, 1.0
    d_x, d_l = devmem.upload(x), devmem.alloc(4 * n)
    replayed = []
    calls = [(0.05, 4), (0.04, 6), (1e-3, 5), (1.1e-3, 3), (0.05, 2), (1e-3, 8)]
    with dclust.Handle(0) as h:
        for eps, mp in calls:
            devmem.h2d(d_l, np.full(n, -7, dtype=np.int32))
            st = h.run_device(d_x, n, dclust.make_params(dim, eps, mp, precision=prec), d_l)
            replayed.append(st["diag"][14])
            lab = devmem.download(np.empty(n, dtype=np.int32), d_l)
            ref = oracle.fast_dbscan(x, eps, mp)
            assert np.array_equal(lab, ref[0])
            assert np.array_equal(h.core_flags(n), ref[1])
            assert st["n_clusters"] == ref[0].max()
    assert replayed == [0, 1, 0, 1, 1, 1]
