"""Near components by union-find (calls without a launch shape) and the
pairs decided across component borders, against the CPU oracle: exact labels
and core flags."""
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


def _snake(n, dim, eps, rng):
    """n points 0.9 eps apart along a path that folds at 300 points per row,
    rows 0.9 eps apart at one end only, with every 977th point left out."""
    i = np.arange(n)
    row, col = i // 300, i % 300
    col = np.where(row % 2 == 0, col, 299 - col)
    x = np.zeros((n, dim))
    x[:, 0] = 5.0 * row
    x[:, -1] = 0.9 * col
    # the step from one row to the next is bridged by four more points
    turns = np.nonzero(i % 300 == 299)[0][:-1]
    bridge = np.repeat(x[turns], 4, axis=0)
    bridge[:, 0] += np.tile([1.0, 2.0, 3.0, 4.0], turns.size)
    x = np.concatenate([np.delete(x, np.arange(976, n, 977), axis=0), bridge]) * eps
    return x[rng.permutation(x.shape[0])]


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("n", [1, 63, 65, 1025, 4097, 20000, 60000])
def test_long_chains_across_runs(handle, dim, n):
    # chains of single-point cells, shorter and longer than the runs of cells
    # one workgroup unites in LDS (4096 to 16384), broken now and then
    x = _snake(n, dim, 0.01, np.random.default_rng(n + dim))
    for kw in ({}, {"seeds": 64, "blocks": 16}):
        ref, st = _check(handle, x, 0.01, 2, dclust.FP32_GUARD, **kw)
        assert st["n_chains"] >= ref.max()
    if n >= 20000:
        assert ref.max() > 10


@pytest.mark.parametrize("prec", PRECS)
@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("gap", [0.8, 0.999, 1.001, 1.3])
def test_heavy_border_pairs(handle, prec, dim, gap):
    # two dense sheets `gap` eps apart (cells of far more than 64 points,
    # some of them not core): joined only through pairs of heavy cells, or
    # not at all
    rng = np.random.default_rng(int(1000 * gap) + dim)
    eps, n = 0.1, 9000
    a = rng.uniform(0, 6 * eps, (n, dim))
    a[:, 0] = rng.uniform(0, 0.05 * eps, n)
    b = rng.uniform(0, 6 * eps, (n, dim))
    b[:, 0] = gap * eps + 0.05 * eps + rng.uniform(0, 0.05 * eps, n)
    lone = np.zeros((40, dim))  # light cells beside them
    lone[:, 0] = np.linspace(-3.0, 4.0, 40) * eps
    lone[:, 1] = 8.0 * eps
    x = np.concatenate([a, b, lone])[rng.permutation(2 * n + 40)]
    ref, st = _check(handle, x, eps, 12, prec)
    assert st["diag"][2] > 0  # heavy cells
    assert ref.max() == (1 if gap < 1 else 2)
