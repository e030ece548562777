"""Data so small or large that eps^2 rounds to zero or infinity, where the
predicate comes down to its box test, and data just inside the ordinary range."""
import numpy as np
import pytest

import dclust
import oracle

pytestmark = pytest.mark.gpu


def _points(kind, dim, rng):
    if kind == "lattice":  # eps 1.5 spacings: the box holds what the ball does not
        g = np.stack(np.meshgrid(*[np.arange(40 if dim == 2 else 12)] * dim, indexing="ij"), -1)
        x = g.reshape(-1, dim).astype(np.float64)
        return x[rng.random(len(x)) < (0.4 if dim == 2 else 0.2)], 1.5
    if kind == "sheets":
        x = rng.uniform(0, 1, (4000, dim))
        x[:, 0] = np.round(x[:, 0] * 6) * 0.101 + rng.uniform(0, 0.002, 4000)
        return x, 0.1
    c = rng.uniform(0, 1, (9, dim))
    return c[rng.integers(0, 9, 3000)] + rng.normal(0, 0.04, (3000, dim)), 0.03


@pytest.mark.parametrize("prec", [dclust.FP64, dclust.FP32_GUARD])
@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("kind", ["lattice", "sheets", "blobs"])
@pytest.mark.parametrize("scale", [1e-290, 1e-170, 1e-145, 1e151, 1e160, 1e290])
def test_eps_whose_square_leaves_the_range(handle, scale, kind, dim, prec):
    x, eps = _points(kind, dim, np.random.default_rng(dim))
    x, eps = x * scale, eps * scale
    for minpts in (2, 6, 20):
        ref, core, asym = oracle.fast_dbscan(x, eps, minpts)
        assert asym == 0
        for kw in ({}, {"seeds": 64, "blocks": 16}):
            lab = handle.run(x, eps, minpts, precision=prec, **kw)
            assert np.array_equal(handle.core_flags(len(x)), core)
            assert np.array_equal(lab, ref)
