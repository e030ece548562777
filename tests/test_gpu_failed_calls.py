"""Calls that fail leave the handle fit for the next ones: what the library
remembers of earlier calls goes with the memory it lay in."""
import numpy as np
import pytest

import dclust
import oracle

pytestmark = pytest.mark.gpu


def _blobs(n, dim, seed):
    rng = np.random.default_rng(seed)
    c = rng.uniform(0, 1, (6, dim))
    return c[rng.integers(0, 6, n)] + rng.normal(0, 0.03, (n, dim))


@pytest.mark.parametrize("replays", [0, 2])
def test_call_after_one_out_of_memory(devmem, replays):
    # 2^47 bytes of collision pairs cannot be had; the next call runs as ever
    x = _blobs(5000, 3, 1)
    n = len(x)
    p = dclust.make_params(3, 0.02, 4)
    huge = dclust.make_params(3, 0.02, 4, seeds=64, blocks=8192, threads=256, extra=2 ** 31 - 1)
    ref = oracle.fast_dbscan(x, 0.02, 4)[0]
    d_x, d_l = devmem.upload(x), devmem.alloc(4 * n)
    with dclust.Handle(0) as h:
        for _ in range(replays):
            h.run_device(d_x, n, p, d_l)
        with pytest.raises(dclust.DclustError) as e:
            h.run_device(d_x, n, huge, d_l)
        assert e.value.code == dclust.E_OOM
        for _ in range(2):
            devmem.h2d(d_l, np.full(n, -7, dtype=np.int32))
            h.run_device(d_x, n, p, d_l)
            assert np.array_equal(devmem.download(np.empty(n, dtype=np.int32), d_l), ref)
