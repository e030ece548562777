"""A captured run is replayed for calls of the same sizes and parameters
whatever buffers they name: each call's labels come from its own input and go
to its own output."""
import numpy as np
import pytest

import dclust
import oracle

pytestmark = pytest.mark.gpu


def _blobs(n, dim, seed):
    rng = np.random.default_rng(seed)
    c = rng.uniform(0, 1, (6, dim))
    return c[rng.integers(0, 6, n)] + rng.normal(0, 0.03, (n, dim))


@pytest.mark.parametrize("prec", [dclust.FP64, dclust.FP32_GUARD])
@pytest.mark.parametrize("dim", [2, 3])
def test_replay_follows_the_buffers(devmem, prec, dim, monkeypatch):
    monkeypatch.delenv("DCLUST_GRAPH", raising=False)
    n, eps, mp = 7001, 0.02, 5
    p = dclust.make_params(dim, eps, mp, precision=prec)
    xs = [_blobs(n, dim, 10 + k) for k in range(4)]
    refs = [oracle.fast_dbscan(x, eps, mp) for x in xs]
    d_x = [devmem.upload(x) for x in xs]
    d_l = [devmem.alloc(4 * n) for _ in xs]
    replayed = []
    with dclust.Handle(0) as h:
        for k in (0, 1, 2, 3, 1, 0):
            # the other outputs must stay as they are
            for j in range(4):
                devmem.h2d(d_l[j], np.full(n, -7 - j, dtype=np.int32))
            st = h.run_device(d_x[k], n, p, d_l[k])
            replayed.append(st["diag"][14])
            for j in range(4):
                lab = devmem.download(np.empty(n, dtype=np.int32), d_l[j])
                assert np.array_equal(lab, refs[k][0] if j == k else np.full(n, -7 - j))
            assert np.array_equal(h.core_flags(n), refs[k][1])
            if st["diag"][14]:
                assert 0 < st["t_core_ms"] < st["t_total_ms"] and st["t_index_ms"] > 0
    assert replayed == [0, 1, 1, 1, 1, 1]


def test_replay_with_guard_band_rechecks(devmem):
    # pairs at eps (1 +- 3e-8) are re-decided from the caller's rows, which
    # differ from call to call
    rng = np.random.default_rng(3)
    eps, m = 1e-3, 400
    p = dclust.make_params(3, eps, 2, precision=dclust.FP32_GUARD)
    with dclust.Handle(0) as h:
        for call in range(4):
            a = np.stack(np.meshgrid(*[np.arange(8)] * 3, indexing="ij"), -1).reshape(-1, 3)[:m] * 0.01
            u = rng.normal(size=(m, 3))
            u /= np.linalg.norm(u, axis=1, keepdims=True)
            b = a + u * eps * (1.0 + rng.uniform(-3e-8, 3e-8, (m, 1)))
            x = np.concatenate([a, b])
            d_x, d_l = devmem.upload(x), devmem.alloc(8 * m)
            st = h.run_device(d_x, 2 * m, p, d_l)
            lab = devmem.download(np.empty(2 * m, dtype=np.int32), d_l)
            ref, _, asym = oracle.fast_dbscan(x, eps, 2)
            assert asym == 0 and np.array_equal(lab, ref)
            assert st["band_rechecks"] >= m and st["diag"][14] == (call > 0)
