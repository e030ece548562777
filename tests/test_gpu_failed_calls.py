"""Calls that fail leave the handle fit for the next ones: what the library
remembers of earlier calls goes with the memory it lay in."""
import ctypes as C

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


def test_batch_after_a_call_out_of_memory(devmem):
    # the instance table and the chunk list of a repeated batch stay on the
    # device; a batch of more instances takes new ones and then finds no memory
    # (2^47 bytes of collision pairs), so the next batch has to bring its own
    xs = [_blobs(n, d, n) for n, d in ((700, 2), (5000, 3), (300, 2))]
    ps = [dclust.make_params(x.shape[1], 0.02, 4) for x in xs]
    ns = np.array([len(x) for x in xs], dtype=np.int64)
    refs = np.concatenate([oracle.fast_dbscan(x, 0.02, 4)[0] for x in xs])
    d_x = devmem.upload(np.concatenate([x.ravel() for x in xs]))
    d_l = devmem.alloc(4 * int(ns.sum()))
    more = np.full(3000, 2, dtype=np.int64)
    d_m, d_ml = devmem.upload(np.zeros(3000 * 2 * 2)), devmem.alloc(4 * 6000)
    huge = [dclust.make_params(2, 0.02, 4, seeds=64, blocks=8192, threads=256,
                               extra=2 ** 31 - 1)] * 3000
    with dclust.Handle(0) as h:
        for fail in (False, False, True, True, False):
            if fail:
                with pytest.raises(dclust.DclustError) as e:
                    h.run_batched_device(d_m, more, huge, d_ml)
                assert e.value.code == dclust.E_OOM
            devmem.h2d(d_l, np.full(int(ns.sum()), -7, dtype=np.int32))
            assert not np.any(h.run_batched_device(d_x, ns, ps, d_l))
            assert np.array_equal(devmem.download(np.empty_like(refs), d_l), refs)


def test_core_flags_after_a_larger_call_that_failed(devmem):
    # the larger call takes new arrays before it finds its bin width too small
    x, big = _blobs(3000, 3, 2), _blobs(200000, 3, 3)
    with dclust.Handle(0) as h:
        h.run(x, 0.02, 4)
        assert np.array_equal(h.core_flags(len(x)), oracle.fast_dbscan(x, 0.02, 4)[1])
        with pytest.raises(dclust.DclustError) as e:
            h.run(big, 0.02, 4, r=10 ** 6)
        assert e.value.code == dclust.E_BINWIDTH
        with pytest.raises(dclust.DclustError) as e:
            h.core_flags(len(x))
        assert e.value.code == dclust.E_PARAM
        h.run(x, 0.02, 4)
        assert np.array_equal(h.core_flags(len(x)), oracle.fast_dbscan(x, 0.02, 4)[1])


@pytest.mark.parametrize("prec", [dclust.FP64, dclust.FP32_GUARD])
def test_failed_replay_writes_nothing(devmem, prec, monkeypatch):
    # a captured run replays for other parameters and other data; when those
    # fail the call, labels and core flags stay as an eager call leaves them
    monkeypatch.delenv("DCLUST_GRAPH", raising=False)
    x = _blobs(7001, 3, 4)
    n = len(x)
    bad = x.copy()
    bad[1234, 1] = np.nan
    ref, core, _ = oracle.fast_dbscan(x, 0.02, 4)
    d_x, d_bad, d_l = devmem.upload(x), devmem.upload(bad), devmem.alloc(4 * n)

    def params(eps=0.02, r=0):
        return dclust.make_params(3, eps, 4, r=r, precision=prec)

    with dclust.Handle(0) as h:
        for _ in range(3):
            st = h.run_device(d_x, n, params(), d_l)
        assert st["diag"][14] == 1
        devmem.h2d(d_l, np.full(n, -7, dtype=np.int32))
        for buf, p, code in ((d_x, params(r=10 ** 6), dclust.E_BINWIDTH),
                             (d_bad, params(), dclust.E_PARAM),
                             (d_x, params(eps=1e-13), dclust.E_PARAM),
                             (d_x, params(eps=1e-9), dclust.E_CAPACITY)):
            with pytest.raises(dclust.DclustError) as e:
                h.run_device(buf, n, p, d_l)
            assert e.value.code == code
            assert np.all(devmem.download(np.empty(n, dtype=np.int32), d_l) == -7)
            assert np.array_equal(h.core_flags(n), core)
        st = h.run_device(d_x, n, params(), d_l)
        assert np.array_equal(devmem.download(np.empty(n, dtype=np.int32), d_l), ref)


@pytest.mark.parametrize("errors_wanted", [False, True])
def test_failed_replay_of_a_batch(devmem, errors_wanted, monkeypatch):
    # without inst_err one bad instance fails the whole call; with it the
    # others are clustered
    monkeypatch.delenv("DCLUST_GRAPH", raising=False)
    xs = [_blobs(900, 2, 5), _blobs(1100, 3, 6)]
    ns = np.array([len(x) for x in xs], dtype=np.int64)
    tot = int(ns.sum())
    refs = [oracle.fast_dbscan(x, 0.02, 4)[0] for x in xs]
    bad = [xs[0], np.where(np.arange(1100)[:, None] == 7, np.inf, xs[1])]
    d_x = devmem.upload(np.concatenate([x.ravel() for x in xs]))
    d_bad = devmem.upload(np.concatenate([x.ravel() for x in bad]))
    d_l = devmem.alloc(4 * tot)
    parr = (dclust.Params * 2)(*[dclust.make_params(x.shape[1], 0.02, 4) for x in xs])
    errs, st = np.zeros(2, dtype=np.int32), dclust.Stats()

    with dclust.Handle(0) as h:
        def call(buf):
            devmem.h2d(d_l, np.full(tot, -7, dtype=np.int32))
            rc = dclust._lib().dclust_run_batched_device(
                h._h, 2, C.c_void_p(buf), ns.ctypes.data, parr, C.c_void_p(d_l),
                errs.ctypes.data if errors_wanted else None, C.byref(st))
            return rc, devmem.download(np.empty(tot, dtype=np.int32), d_l)

        for k in range(3):
            rc, lab = call(d_x)
            assert rc == 0 and np.array_equal(lab, np.concatenate(refs))
        assert st.diag[14] == 1
        rc, lab = call(d_bad)
        assert rc == dclust.E_PARAM
        if errors_wanted:
            assert errs.tolist() == [0, dclust.E_PARAM]
            assert np.array_equal(lab[:900], refs[0])
        else:
            assert np.all(lab == -7)
        rc, lab = call(d_x)
        assert rc == 0 and np.array_equal(lab, np.concatenate(refs)) and st.diag[14] == 1
