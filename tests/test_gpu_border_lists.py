"""The lists of cell pairs across near components: more pairs than a list holds
(lattices, very small calls), and many pairs from few cells."""
import numpy as np
import pytest

import dclust
import oracle

pytestmark = pytest.mark.gpu

PRECS = [dclust.FP64, dclust.FP32_GUARD]


def _check(handle, x, eps, minpts, prec, **kw):
    lab = handle.run(x, eps, minpts, precision=prec, **kw)
    ref, core, asym = oracle.fast_dbscan(x, eps, minpts)
    assert asym == 0
    assert np.array_equal(handle.core_flags(x.shape[0]), core)
    assert np.array_equal(lab, ref), f"{int(np.sum(lab != ref))} labels differ"
    return ref, handle.last_stats


@pytest.mark.parametrize("prec", PRECS)
@pytest.mark.parametrize("dim,side,eps,share", [(2, 130, 1.0, 0.55), (2, 130, 1.5, 0.3),
                                                (3, 26, 1.0, 0.25), (3, 26, 1.5, 0.12),
                                                (3, 40, 2.0, 0.04)])
def test_lattices(handle, prec, dim, side, eps, share):
    # eps near the spacing: cells lie two apart, the near graph has few edges
    # and the pairs are several per point, more than the lists hold
    g = np.stack(np.meshgrid(*[np.arange(side)] * dim, indexing="ij"), -1).reshape(-1, dim)
    rng = np.random.default_rng(side + dim)
    x = g[rng.random(len(g)) < share].astype(np.float64)
    x = x[rng.permutation(len(x))]
    for kw in ({}, {"seeds": 64, "blocks": 16}):
        ref, _ = _check(handle, x, eps, 2, prec, **kw)
        assert ref.max() > 10


@pytest.mark.parametrize("prec", PRECS)
@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("gap", [0.999, 1.001])
@pytest.mark.parametrize("n", [20, 63, 127, 128, 300])
def test_small_calls_with_crowded_cells(handle, prec, dim, gap, n):
    # below 128 points the lists hold nothing; cells of 10 points to more than
    # a wavefront's worth on either side of a gap of one eps
    rng = np.random.default_rng(n + dim)
    eps = 0.1
    a = rng.uniform(0, 0.3 * eps, (n // 2, dim))
    b = rng.uniform(0, 0.3 * eps, (n - n // 2, dim))
    a[:, 0] *= 0.1
    b[:, 0] = (gap + 0.03) * eps + 0.1 * b[:, 0]
    a[0], b[0] = 0.0, 0.0
    a[0, 0], b[0, 0] = 0.03 * eps, (gap + 0.03) * eps  # the nearest pair
    x = np.concatenate([a, b])[rng.permutation(n)]
    ref, _ = _check(handle, x, eps, 5, prec)
    assert ref.max() == (1 if gap < 1 else 2)


@pytest.mark.parametrize("prec", PRECS)
@pytest.mark.parametrize("dim", [2, 3])
def test_pairs_of_few_cells_are_decided_once(handle, prec, dim):
    # two dense sheets just over eps apart: no pair joins, so the number of
    # tests is that of every pair decided once, whatever room the lists have
    # (they grow with the call: 700,000 lone points far away make it ample)
    rng = np.random.default_rng(dim)
    eps, n, m = 0.1, 9000, 700000
    a = rng.uniform(0, 6 * eps, (n, dim))
    a[:, 0] = rng.uniform(0, 0.05 * eps, n)
    b = rng.uniform(0, 6 * eps, (n, dim))
    b[:, 0] = 1.001 * eps + 0.05 * eps + rng.uniform(0, 0.05 * eps, n)
    x = np.concatenate([np.zeros((1, dim)), a, b])
    lone = np.zeros((m, dim))
    lone[:, 0], lone[:, 1] = 20 * eps + 3 * eps * (np.arange(m) % 600), 3 * eps * (np.arange(m) // 600)
    tests = []
    for pts in (x, np.concatenate([x, lone])):
        ref, st = _check(handle, pts, eps, 12, prec)
        assert ref.max() == 2
        tests.append(st["diag"][10])
    assert tests[0] == tests[1]
