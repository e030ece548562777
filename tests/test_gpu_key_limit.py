"""Cells whose sort keys lie above 2^63: the largest accepted grids (2^21 cells
along each of three axes, whose column order pads the keys past the number of
cells), with clusters in the far corner and across the key 2^63."""
import numpy as np
import pytest

import dclust
import oracle

pytestmark = pytest.mark.gpu

EPS = 1.0
W = 0.5 * EPS * (1.0 + 2.0 ** -20)  # cell width
FULL = 1 << 21


def _corner(nk, seed):
    # walks of points 0.3 to 0.9 eps apart near the last cells of axis 0: in
    # the middle and at the end of axis 1, at several places of axis 2
    rng = np.random.default_rng(seed)
    ext = (np.array(nk) - 0.5) * W
    rows = [np.zeros((1, 3)), ext[None]]
    for fy in (0.0, 0.5, 1.0):
        for fz in (0.0, 0.0005, 0.5, 1.0):
            step = rng.uniform(0.3, 0.9, (60, 1)) * EPS
            u = rng.normal(size=(60, 3))
            walk = np.cumsum(step * u / np.linalg.norm(u, axis=1, keepdims=True), axis=0)
            at = np.array([ext[0] - 3.0, fy * ext[1], fz * ext[2]])
            rows.append(np.clip(at + walk, 0.0, ext))
    x = np.concatenate(rows)
    return x[rng.permutation(len(x))]


@pytest.mark.parametrize("prec", [dclust.FP64, dclust.FP32_GUARD])
@pytest.mark.parametrize("nk", [(FULL, FULL, FULL), (FULL, FULL, FULL - 1),
                                (FULL - 1, FULL - 1, FULL - 1)])
def test_keys_above_2_63(handle, nk, prec):
    x = _corner(nk, nk[2] & 7)
    ref, core, asym = oracle.fast_dbscan(x, EPS, 3)
    assert asym == 0 and ref.max() >= 6
    assert np.array_equal(handle.run(x, EPS, 3, precision=prec), ref)
    assert handle.last_stats["key_bits"] == 64
    assert np.array_equal(handle.core_flags(len(x)), core)


def test_batch_with_keys_above_2_63(handle):
    xs = [_corner((FULL, FULL, FULL - 1), 5), np.random.default_rng(6).uniform(0, 20, (500, 3))]
    labels, errs = handle.run_batched(xs, [dclust.make_params(3, EPS, 3)] * 2)
    assert not np.any(errs) and handle.last_stats["key_bits"] == 64
    for x, lab in zip(xs, labels):
        assert np.array_equal(lab, oracle.fast_dbscan(x, EPS, 3)[0])
