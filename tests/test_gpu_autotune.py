"""What the autotuners give out is no slower path than the zeros they replace:
launch values that a handle wrote for zeros run without seed lists on it where
that is the faster way, and are an explicit shape anywhere else."""
import numpy as np
import pytest

import dclust
import oracle

pytestmark = pytest.mark.gpu

WAVES = 7  # dclust_stats.diag: expansion wavefronts, 0 without seed lists


def _run(h, x, p):
    lab = h.run(x, p.eps, p.minpts, precision=p.precision, seeds=p.seed_list_size,
                blocks=p.blocks, threads=p.block_threads, extra=p.extra_collision)
    assert np.array_equal(lab, oracle.fast_dbscan(x, p.eps, p.minpts)[0])
    return h.last_stats["diag"][WAVES]


def test_tuned_shape_stands_for_zeros(devmem):
    x, info = dclust.synth_config(3, n=150000)
    p = dclust.make_params(3, info["eps"], info["minpts"], precision=dclust.FP32_GUARD)
    d_x = devmem.upload(np.ascontiguousarray(x))
    with dclust.Handle(0) as h, dclust.Handle(0) as other:
        for _ in range(2):  # (the second sweep measures the shape as itself again)
            tuned = h.autotune_device(d_x, [x.shape[0]], [p])[0]
            assert tuned.seed_list_size > 0 and tuned.blocks > 0 and tuned.block_threads > 0
            assert _run(h, x, tuned) == 0
        assert _run(other, x, tuned) > 0
        tuned.seed_list_size = 64  # the caller's own value
        assert _run(h, x, tuned) > 0


def test_filled_shape_stands_for_zeros(devmem):
    x, info = dclust.synth_config(3, n=60000)

    def params(**kw):
        return dclust.make_params(3, info["eps"], info["minpts"], **kw)

    with dclust.Handle(0) as h, dclust.Handle(0) as other:
        p = h.autotune(x.shape[0], params())
        assert p.seed_list_size > 0 and p.extra_collision > 0
        assert _run(h, x, p) == 0
        assert _run(other, x, p) > 0
        assert _run(h, x, h.autotune(x.shape[0], params(seeds=64))) > 0
