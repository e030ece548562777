"""Host entry points: arrays that go through the pinned halves (4 MiB each,
pieces below 1 MiB) and arrays that do not, alone and mixed in one batch,
against the device entry point on the same points."""
import numpy as np
import pytest

import dclust

pytestmark = pytest.mark.gpu

MIB = 1 << 20


def _points(n, dim, seed):
    rng = np.random.default_rng(seed)
    c = rng.uniform(0, 1, (8, dim))
    return c[rng.integers(0, 8, n)] + rng.normal(0, 0.05, (n, dim))


def _device_labels(handle, devmem, x, p):
    d_x, d_l = devmem.upload(x), devmem.alloc(4 * x.shape[0])
    handle.run_device(d_x, x.shape[0], p, d_l)
    return devmem.download(np.empty(x.shape[0], dtype=np.int32), d_l)


@pytest.mark.parametrize("n", [1, 1000, MIB // 24, MIB // 24 + 1, MIB // 4 - 1, MIB // 4,
                               MIB // 4 + 1])
def test_single(handle, devmem, n):
    # points and labels one below, at and one above the size of a staged piece
    x = _points(n, 3, n)
    p = dclust.make_params(3, 0.02, 5, precision=dclust.FP32_GUARD)
    want = _device_labels(handle, devmem, x, p)
    for _ in range(3):  # eager, captured, replayed
        assert np.array_equal(handle.run(x, 0.02, 5, precision=dclust.FP32_GUARD), want)


@pytest.mark.parametrize("sizes", [[40] * 700, [30000] * 12, [MIB // 16, 5, 0, MIB // 16 - 1, 7],
                                   [200000, 3, 100, 150000, 20000, 20000, 1]])
def test_batch(handle, devmem, sizes):
    # many small pieces, pieces that do not fill a half evenly, and small ones
    # between large ones
    xs = [_points(n, 2, i) if n else np.empty((0, 2)) for i, n in enumerate(sizes)]
    ps = [dclust.make_params(2, 0.01, 4, precision=dclust.FP32_GUARD)] * len(xs)
    for _ in range(2):
        labs, errs = handle.run_batched(xs, ps)
        assert not np.any(errs) and [a.shape[0] for a in labs] == sizes
    d_x = devmem.upload(np.concatenate([x.ravel() for x in xs]))
    d_l = devmem.alloc(4 * sum(sizes))
    handle.run_batched_device(d_x, sizes, ps, d_l)
    want = devmem.download(np.empty(sum(sizes), dtype=np.int32), d_l)
    assert np.array_equal(np.concatenate(labs), want)
