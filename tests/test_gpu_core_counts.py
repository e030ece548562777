"""Neighbour counts shared by several lanes: results against the oracle at the
size where the lanes per point change, with records of every length, crowded
windows, pairs at exactly eps and pairs inside the guard band."""
import numpy as np
import pytest

import dclust
import oracle

pytestmark = pytest.mark.gpu


def _check(devmem, x, eps, minpts, prec):
    n = len(x)
    d_x, d_l = devmem.upload(x), devmem.alloc(4 * n)
    ref, core, _ = oracle.fast_dbscan(x, eps, minpts)
    with dclust.Handle(0) as h:
        p = dclust.make_params(x.shape[1], eps, minpts, precision=prec)
        for _ in range(2):
            st = h.run_device(d_x, n, p, d_l)
            assert np.array_equal(h.core_flags(n), core)
            assert np.array_equal(devmem.download(np.empty(n, dtype=np.int32), d_l), ref)
    return st


@pytest.mark.parametrize("prec", [dclust.FP64, dclust.FP32_GUARD])
@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("n", [(1 << 19) - 1, 1 << 19])
def test_size_of_the_rule(devmem, prec, dim, n):
    rng = np.random.default_rng(n + dim)
    c = rng.uniform(0, 1, (n // 40, dim))
    eps = 0.4 * (1.0 / n) ** (1.0 / dim) * 8
    x = c[rng.integers(0, len(c), n)] + rng.normal(0, eps / 3, (n, dim))
    _check(devmem, x, eps, 7, prec)


@pytest.mark.parametrize("prec", [dclust.FP64, dclust.FP32_GUARD])
@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("minpts", [2, 8, 9, 33, 40, 300])
def test_records_and_crowds(devmem, prec, dim, minpts):
    # uniform points around a core that holds more than 512 candidates a window
    rng = np.random.default_rng(minpts)
    x = np.concatenate([rng.uniform(-6, 6, (6000, dim)), rng.normal(0, 0.6, (3000, dim))])
    _check(devmem, x, 0.45 if dim == 2 else 0.8, minpts, prec)


@pytest.mark.parametrize("prec", [dclust.FP64, dclust.FP32_GUARD])
@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("step", [0.25, 0.5, 0.125])
def test_pairs_at_eps(devmem, prec, dim, step):
    # lattices: many pairs at exactly eps, on the edges of the reach of a point
    m = 24 if dim == 3 else 120
    g = np.stack(np.meshgrid(*[np.arange(m)] * dim, indexing="ij"), -1).reshape(-1, dim) * step
    x = g[np.random.default_rng(1).random(len(g)) < 0.4] - 1.0
    full = {2: 13, 3: 33}[dim] if step == 0.25 else 4
    st = _check(devmem, x, 0.5, max(2, full // 2), prec)
    if prec == dclust.FP32_GUARD and step == 0.5:  # (no nearer neighbour makes up for them)
        assert st["band_rechecks"] > 0


@pytest.mark.parametrize("prec", [dclust.FP64, dclust.FP32_GUARD])
@pytest.mark.parametrize("dim,minpts", [(2, 3), (2, 5), (2, 6), (3, 7), (3, 8)])
def test_every_point_at_eps(devmem, prec, dim, minpts):
    # a lattice with eps its spacing: each point's neighbours are all exactly
    # eps away (2 dim of them inside the lattice); beside it a crowd of more
    # than 512 candidates a point, whose points share the same list
    m = 150 if dim == 2 else 30
    g = np.stack(np.meshgrid(*[np.arange(m)] * dim, indexing="ij"), -1).reshape(-1, dim) * 0.5
    rng = np.random.default_rng(dim + minpts)
    x = np.concatenate([g, 200.0 + rng.normal(0, 0.25, (2500, dim))])
    st = _check(devmem, x[rng.permutation(len(x))], 0.5, minpts, prec)
    if prec == dclust.FP32_GUARD:
        assert st["band_rechecks"] > len(g)
