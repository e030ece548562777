"""Column windows and neighbour counts at the sizes where they take another
path, against the CPU oracle: exact labels and core flags in both forms."""
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
    return handle.last_stats


@pytest.mark.parametrize("prec", PRECS)
@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("cells", [1, 2, 3, 5, 40, 4000])
def test_long_columns(handle, prec, dim, cells):
    # a grid of `cells` cells along the last axis and 1 to 6 along the others:
    # columns shorter and longer than a tile of 64 cells and than the 512
    # cells a tile stages, odd and even numbers of cells per block
    rng = np.random.default_rng(cells + dim)
    eps = 0.1
    w = eps / 2 * (1 + 2.0 ** -20)
    for wide in (1, 2, 3, 6):
        n = min(20000, 40 + 3 * cells * wide ** (dim - 1))
        x = rng.uniform(0, 1, (n, dim)) * w * 0.999
        x[:, :-1] *= wide
        x[:, -1] *= cells
        _check(handle, x, eps, 6, prec)


@pytest.mark.parametrize("prec", PRECS)
@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("per_cell,minpts", [(3, 9), (20, 24), (60, 80), (700, 900)])
def test_crowded_and_sparse_windows(handle, prec, dim, per_cell, minpts):
    # a block of cells of `per_cell` points (fewer than minpts: every point is
    # counted), windows below and above 512 candidates and above the 4095
    # points a window's count holds, more neighbours than record slots, beside
    # a sparse half whose windows hold fewer than minpts points
    rng = np.random.default_rng(10 * per_cell + dim)
    eps = 0.1
    side = {2: 12, 3: 5}[dim] if per_cell > 100 else {2: 24, 3: 9}[dim]
    n = per_cell * side ** dim
    x = rng.uniform(0, side * eps / 2, (n, dim))
    x[:, 0] *= 0.5 + rng.uniform(0, 0.5, n)  # thinner towards one side
    sparse = rng.uniform(0, 20 * side * eps, (600, dim))
    sparse[:, 0] += side * eps
    lone = rng.uniform(0, side * eps / 2, (50, dim))  # just outside the block
    lone[:, -1] = side * eps / 2 + rng.uniform(0.2, 1.2, 50) * eps
    x = np.concatenate([x, sparse, lone])
    x = x[rng.permutation(x.shape[0])]
    st = _check(handle, x, eps, minpts, prec)
    if per_cell == 700 and dim == 3:
        assert st["work"][3] > 0  # some points taken by a wavefront each


@pytest.mark.parametrize("prec", PRECS)
def test_mixed_batch_of_small_grids(handle, prec):
    # tiles of 64 cells that hold cells of several instances, of both
    # dimensions, with grids of one to a few columns
    rng = np.random.default_rng(5)
    xs, ps = [], []
    for k in range(60):
        dim = 2 + k % 2
        n = int(rng.integers(1, 200))
        xs.append(rng.uniform(0, rng.uniform(0.05, 2.0), (n, dim)))
        ps.append(dclust.make_params(dim, 0.11, 1 + k % 7, precision=prec))
    labs, errs = handle.run_batched(xs, ps)
    assert not np.any(errs)
    for i, (x, p) in enumerate(zip(xs, ps)):
        ref, _, asym = oracle.fast_dbscan(x, p.eps, p.minpts)
        assert asym == 0 and np.array_equal(labs[i], ref), f"instance {i}"
