"""Performance cases: the clustering calls that programs make of this library.

Every case goes through the Python binding of the C ABI (Handle.run,
run_device, run_device_noalloc, run_batched, run_batched_device, core_flags)
on synthetic Gaussian-blob data of the shapes the benchmark configurations
name.  How a case's call is made ("entry"):

  resident      a handle and its device buffers that stay: a service clusters
                the same buffers again and again as their contents change
  fresh         one handle for the whole process, and every data set in
                buffers of its own
  noalloc       the entry point for serving loops that may not allocate
  host          host arrays in, host labels out, one handle for the process
                (the reference program's own use: one data set read from a
                file)
  batch         many independent instances in one call, device resident
  batch_host    the same from host arrays

Sizes and parameters of the listed cases are the benchmark configurations'
(2-D 10 k and 1 M points, 3-D 4 M and 32 M points, batches of 200 to 200,000
points each) and generic ones between them.
"""
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "fast-cuda-gpu-dbscan_amd"))
import dclust  # noqa: E402


def _blobs(name, entry, dim, n, precision, minpts, **kw):
    """One data set: `blobs` Gaussian blobs with sigmas in [sigma_lo,
    sigma_hi] (times `box`) and sizes by a Zipf law, a share of uniform noise,
    in [0, box]^dim; eps is given, or found from the number of neighbours a
    typical clustered point shall have."""
    case = {"name": name, "entry": entry, "dim": dim, "n": n, "precision": precision,
            "minpts": minpts, "blobs": 64, "sigma_lo": 0.005, "sigma_hi": 0.03, "zipf": 1.1,
            "noise": 0.05, "filaments": 0.0, "box": 1.0, "eps": 0.0, "neighbours": 30.0, "r": 0,
            "seeds": 0, "core": False}
    case.update(kw)
    return case


def _batch(name, entry, count, lo, hi, precision):
    """`count` instances of 2 or 3 dimensions, sizes log-uniform in [lo, hi],
    each a mixture of 2 to 32 blobs with 5 % noise and its own eps (0.5 to 2
    times a typical 10th-neighbour distance) and minpts (4, 8 or 16)."""
    return {"name": name, "entry": entry, "count": count, "lo": lo, "hi": hi,
            "precision": precision}


def listed():
    return [
        # the smallest ordinary call: the reference's own program on a 2-D
        # file of 10,000 points (latency of one call, transfers included)
        _blobs("host_2d_10k_f64", "host", 2, 10_000, "fp64", 4, blobs=8, sigma_lo=0.015,
               sigma_hi=0.015, zipf=0.0, noise=0.1, box=100.0, eps=1.0, r=5),
        # a serving loop over frames of a 3-D sensor: no allocation allowed
        _blobs("noalloc_3d_100k_f32", "noalloc", 3, 100_000, "fp32", 10, neighbours=25.0),
        # host arrays of ordinary size, core flags wanted as well
        _blobs("host_3d_300k_f32", "host", 3, 300_000, "fp32", 10, neighbours=30.0, core=True),
        # a program that clusters one new tensor after another, odd size
        _blobs("fresh_3d_613757_f32", "fresh", 3, 613_757, "fp32", 8, neighbours=20.0),
        # crowded neighbourhoods and a high minpts, plain FP64
        _blobs("resident_3d_262147_dense_f64", "resident", 3, 262_147, "fp64", 30,
               neighbours=120.0, blobs=32),
        # 2-D, one million points (geographic data): the plain FP64 form
        _blobs("resident_2d_1m_f64", "resident", 2, 1_000_000, "fp64", 4, sigma_lo=0.002,
               sigma_hi=0.02, zipf=1.2, eps=0.002),
        # the same scale in new buffers each time, FP32 with guard band
        _blobs("fresh_2d_1500001_f32", "fresh", 2, 1_500_001, "fp32", 8, sigma_lo=0.002,
               sigma_hi=0.02, zipf=1.2, neighbours=40.0),
        # 3-D, four million points (the headline size), both forms
        _blobs("resident_3d_4m_f32", "resident", 3, 4_000_000, "fp32", 10, blobs=128,
               noise=0.03, eps=0.001425),
        _blobs("resident_3d_4m_f64", "resident", 3, 4_000_000, "fp64", 10, blobs=128,
               noise=0.03, eps=0.001425),
        # the largest: 32 million points in very dense blobs and thin
        # filaments, seed lists of 64 cells
        _blobs("resident_3d_32m_dense_f32", "resident", 3, 32_000_000, "fp32", 20, blobs=16,
               sigma_lo=0.002, sigma_hi=0.002, zipf=0.0, noise=0.01, filaments=0.08, eps=0.001,
               seeds=64),
        # many uneven independent instances in one call
        _batch("batch_256_f32", "batch", 256, 200, 200_000, "fp32"),
        # many tiny instances from host arrays
        _batch("batch_host_400_tiny_f64", "batch_host", 400, 50, 2_000, "fp64"),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    precision = rng.choice(["fp32", "fp64"])
    entry = rng.choice(["resident", "resident", "resident", "fresh", "fresh", "host", "noalloc",
                        "batch", "batch_host"])
    if entry == "batch":
        case = _batch("", entry, _log_uniform(rng, 8, 256), 200, 200_000, precision)
    elif entry == "batch_host":
        case = _batch("", entry, _log_uniform(rng, 8, 400), 50, 2_000, precision)
    else:
        dim = rng.choice([2, 3, 3])
        most = {"resident": 16_000_000, "fresh": 4_000_000, "host": 1_000_000,
                "noalloc": 150_000}[entry]
        lo = rng.uniform(0.002, 0.02)
        case = _blobs("", entry, dim, _log_uniform(rng, 1_000, most), precision,
                      rng.choice([4, 8, 10, 16, 20, 30]), blobs=_log_uniform(rng, 4, 256),
                      sigma_lo=round(lo, 5), sigma_hi=round(lo * rng.uniform(1.0, 6.0), 5),
                      zipf=round(rng.uniform(0.0, 1.3), 3), noise=round(rng.uniform(0.0, 0.2), 3),
                      neighbours=round(math.exp(rng.uniform(math.log(6.0), math.log(150.0))), 2),
                      core=entry == "host" and rng.random() < 0.5)
    del case["name"]
    return case


# ------------------------------------------------------------------ inputs --
_BALL = {2: math.pi, 3: 4.0 * math.pi / 3.0}


def _weighted_median(values, weights):
    order = np.argsort(values)
    c = np.cumsum(np.asarray(weights, dtype=np.float64)[order])
    return float(np.asarray(values)[order][np.searchsorted(c, 0.5 * c[-1])])


def _typical_eps(counts, sigmas, dim, neighbours):
    """Radius of the ball that holds `neighbours` points at the mean density
    around a point of a blob, for the blob of the median point."""
    counts = np.maximum(np.asarray(counts, dtype=np.float64), 1.0)
    vol = np.prod(2.0 * math.sqrt(math.pi) * sigmas[:, :dim], axis=1)
    radius = (neighbours * vol / (counts * _BALL[dim])) ** (1.0 / dim)
    return _weighted_median(radius, counts)


def _points(dim, n, k, sigma_lo, sigma_hi, zipf, noise, filaments, rng, gen, device):
    """n shuffled rows in [0, 1]^dim on the device, the blobs' sizes and
    sigmas.  `rng` makes the mixture, `gen` its points."""
    centres = rng.uniform(0.1, 0.9, (k, dim)) if filaments else rng.uniform(0.0, 1.0, (k, dim))
    sig = rng.uniform(sigma_lo, sigma_hi, (k, dim)) if dim == 2 else \
        np.repeat(rng.uniform(sigma_lo, sigma_hi, (k, 1)), dim, axis=1)
    n_noise = int(round(noise * n))
    n_fil = int(round(filaments * n))
    weights = np.arange(1, k + 1, dtype=np.float64) ** -zipf
    share = np.floor((n - n_noise - n_fil) * weights / weights.sum()).astype(np.int64)
    share[: n - n_noise - n_fil - int(share.sum())] += 1
    who = torch.repeat_interleave(torch.arange(k, device=device),
                                  torch.from_numpy(share).to(device))

    def normal(*shape):
        return torch.randn(shape, generator=gen, device=device, dtype=torch.float64)

    def uniform(*shape):
        return torch.rand(shape, generator=gen, device=device, dtype=torch.float64)

    x = torch.empty((n, dim), device=device, dtype=torch.float64)
    m = who.numel()
    z = normal(m, dim) * torch.from_numpy(sig).to(device)[who]
    if dim == 2:  # anisotropic blobs lie at any angle
        a = torch.from_numpy(rng.uniform(0.0, math.pi, k)).to(device)[who]
        z = torch.stack([a.cos() * z[:, 0] - a.sin() * z[:, 1],
                         a.sin() * z[:, 0] + a.cos() * z[:, 1]], dim=1)
    x[:m] = torch.from_numpy(centres).to(device)[who] + z
    if n_fil:  # two random cubic curves with a little jitter
        for part, at in ((n_fil // 2, m), (n_fil - n_fil // 2, m + n_fil // 2)):
            p = torch.from_numpy(rng.uniform(0.1, 0.9, (4, dim))).to(device)
            t = uniform(part, 1)
            u = 1.0 - t
            x[at:at + part] = (u ** 3 * p[0] + 3 * u * u * t * p[1] + 3 * u * t * t * p[2] +
                               t ** 3 * p[3] + 1e-4 * normal(part, dim))
    x[n - n_noise:] = uniform(n_noise, dim)
    x = x.abs()
    x = torch.where(x > 1.0, (2.0 - x).abs(), x)  # reflected into the box
    return x[torch.randperm(n, generator=gen, device=device)], share, sig


_handle = None


def _process_handle():
    """The one handle of a program that keeps a single one."""
    global _handle
    if _handle is None:
        _handle = dclust.Handle(0)
    return _handle


def _batch_plan(case):
    """(dimension, points) of each instance: the case's, whatever the data."""
    rng = np.random.default_rng([case["count"], case["lo"], case["hi"]])
    dims = rng.integers(2, 4, case["count"])
    sizes = np.exp(rng.uniform(math.log(case["lo"]), math.log(case["hi"]), case["count"]))
    return [(int(d), int(round(n))) for d, n in zip(dims, sizes)]


def _prepare_batch(case, rng, gen):
    on_host = case["entry"] == "batch_host"
    device = "cpu" if on_host else "cuda"
    rows, ns, params = [], [], []
    for dim, n in _batch_plan(case):
        k = int(rng.integers(2, 33))
        x, share, sig = _points(dim, n, k, 0.005, 0.05, 0.0, 0.05, 0.0, rng, gen, device)
        eps = float(rng.uniform(0.5, 2.0)) * _typical_eps(share, sig, dim, 10.0)
        rows.append(x)
        ns.append(n)
        params.append(dclust.make_params(dim, eps, int(rng.choice([4, 8, 16])),
                                         precision=case["precision"]))
    if on_host:
        return {"entry": "batch_host", "handle": _process_handle(), "params": params,
                "x": [np.ascontiguousarray(x.numpy()) for x in rows]}
    return {"entry": "batch", "handle": dclust.Handle(0), "params": params,
            "x": torch.cat([x.reshape(-1) for x in rows]), "ns": np.array(ns, dtype=np.int64),
            "labels": torch.empty(sum(ns), device="cuda", dtype=torch.int32)}


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    on_host = case["entry"] == "batch_host"
    gen = torch.Generator(device="cpu" if on_host else "cuda")
    gen.manual_seed(int(seed))
    if case["entry"] in ("batch", "batch_host"):
        state = _prepare_batch(case, rng, gen)
        torch.cuda.synchronize()
        return state
    dim, n = case["dim"], case["n"]
    x, share, sig = _points(dim, n, case["blobs"], case["sigma_lo"], case["sigma_hi"],
                            case["zipf"], case["noise"], case["filaments"], rng, gen, "cuda")
    x = (x * case["box"]).contiguous()
    eps = case["eps"] or case["box"] * _typical_eps(share, sig, dim, case["neighbours"])
    state = {"entry": case["entry"], "n": n, "eps": eps, "minpts": case["minpts"],
             "precision": case["precision"], "r": case["r"], "core": case["core"],
             "handle": dclust.Handle(0) if case["entry"] == "resident" else _process_handle(),
             "params": dclust.make_params(dim, eps, case["minpts"], r=case["r"],
                                          seeds=case["seeds"], precision=case["precision"])}
    if case["entry"] == "host":
        state["x"] = x.cpu().numpy()
    else:
        state["x"] = x
        state["labels"] = torch.empty(n, device="cuda", dtype=torch.int32)
    torch.cuda.synchronize()  # the library works on a stream of its own
    return state


# --------------------------------------------------------------------- run --
def run(state):
    h, x, entry = state["handle"], state["x"], state["entry"]
    if entry == "host":
        precision = dclust.FP32_GUARD if state["precision"] == "fp32" else dclust.FP64
        labels = h.run(x, state["eps"], state["minpts"], r=state["r"], precision=precision)
        return (labels, h.core_flags(state["n"])) if state["core"] else labels
    if entry == "batch_host":
        labels, errors = h.run_batched(x, state["params"])
        return np.concatenate(labels), errors
    if entry == "batch":
        errors = h.run_batched_device(x.data_ptr(), state["ns"], state["params"],
                                      state["labels"].data_ptr())
        return state["labels"], errors
    call = h.run_device_noalloc if entry == "noalloc" else h.run_device
    call(x.data_ptr(), state["n"], state["params"], state["labels"].data_ptr())
    return state["labels"]


def work(case):
    """Each coordinate read once, each label written once (and each core flag
    where asked for); one distance test per point."""
    if "count" in case:
        sets, flag = _batch_plan(case), 0
    else:
        sets, flag = [(case["dim"], case["n"])], 1 if case["core"] else 0
    return {"bytes": sum(n * (8.0 * dim + 4.0 + flag) for dim, n in sets),
            "flops": sum(n * 3.0 * dim for dim, n in sets)}
