"""The work whose speed is tracked: k-Shape fits, assignments, shape
extraction and the primitives, called as a program that keeps its series in
torch tensors on the GPU calls them.

listed() names the cases and says what each stands for, draw() gives one more
of the same ranges, prepare() makes the device inputs, run() is one pass
through the public entry points (timesc.Context, timesc.Batch, the C ABI of
include/timesc.h), exact() the same result in 64-bit torch, work() the bytes
and operations no implementation can do without.
"""
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PACKAGE = os.path.join(ROOT, "times-c_amd")
if PACKAGE not in sys.path:
    sys.path.insert(0, PACKAGE)

import timesc  # noqa: E402  (after torch, so that both share one HIP runtime)

_ctx = None
_batch = None


def _context():
    """The one context of the program, with the launch shapes measured for
    this GPU loaded, as bench.py does."""
    global _ctx
    if _ctx is None:
        timesc.tune_load(os.path.join(PACKAGE, "tune_mi355x.txt"))
        _ctx = timesc.Context(0)
    return _ctx


def _workers():
    """The one pool of the program, of the benchmark's eight workers."""
    global _batch
    if _batch is None:
        _context()
        _batch = timesc.Batch(0, workers=8)
    return _batch


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # the smallest job of the benchmark: launches and waits count
        {"name": "fit_small", "kind": "fit", "n": 512, "m": 128, "k": 4, "sigma": 0.3,
         "max_iter": 10, "least_iters": 3},
        # the benchmark's headline job: a large data set, noise that keeps
        # labels moving for all ten iterations
        {"name": "fit_large", "kind": "fit", "n": 100000, "m": 512, "k": 16, "sigma": 0.5,
         "max_iter": 10, "least_iters": 10},
        # many independent uneven jobs at once (one per sensor, shop, patient)
        {"name": "batch", "kind": "batch", "jobs": 64, "mix": 1, "max_iter": 10, "least_iters": 3},
        # one refinement step of a program with its own loop: labels known,
        # shifts left to the call
        {"name": "extract", "kind": "extract", "n": 20000, "m": 512, "k": 16, "sigma": 0.4,
         "given_shift": False},
        # a serving query: a few new series against a fitted model
        {"name": "assign_query", "kind": "assign", "n": 96, "m": 256, "k": 24, "sigma": 0.3,
         "dmat": False},
        # labelling a whole archive of short series
        {"name": "assign_short", "kind": "assign", "n": 200000, "m": 96, "k": 32, "sigma": 0.4,
         "dmat": False},
        # labelling a year of daily values per series
        {"name": "assign_daily", "kind": "assign", "n": 30000, "m": 365, "k": 12, "sigma": 0.4,
         "dmat": False},
        # long series (the length of the long single-job configuration)
        {"name": "assign_long", "kind": "assign", "n": 3000, "m": 2709, "k": 8, "sigma": 0.3,
         "dmat": False},
        # all distances, for a program that ranks or thresholds them
        {"name": "distances", "kind": "assign", "n": 8000, "m": 1000, "k": 20, "sigma": 0.4,
         "dmat": True},
        # whole correlation sequences of some series with some patterns
        {"name": "ncc", "kind": "ncc", "n": 700, "m": 301, "k": 12, "sigma": 0.4},
        # a copy of one cluster's members aligned to its centroid
        {"name": "align", "kind": "align", "n": 12000, "m": 700, "k": 1, "sigma": 0.3},
        # freshly loaded series made comparable, an odd length
        {"name": "znorm", "kind": "znorm", "n": 60000, "m": 365, "k": 1, "sigma": 0.4},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["fit", "fit", "batch", "extract", "assign", "assign", "assign", "assign",
                       "ncc", "align", "znorm"])
    if kind == "batch":
        return {"kind": "batch", "jobs": rng.randint(32, 56), "mix": rng.randint(2, 1 << 20),
                "max_iter": 10, "least_iters": 3}
    m = _log_int(rng, 24, 3000)
    c = {"kind": kind, "m": m, "k": 1, "sigma": round(rng.uniform(0.25, 0.5), 2)}
    if kind == "fit":
        c["m"] = m = _log_int(rng, 48, 1500)
        c["k"] = k = rng.randint(2, 24)
        c["n"] = min(_log_int(rng, 300, 60000), 400_000_000 // (m * k))
        c["max_iter"], c["least_iters"] = 10, 3
    elif kind == "extract":
        c["m"] = m = _log_int(rng, 48, 1500)
        c["k"] = k = rng.randint(2, 24)
        c["n"] = min(_log_int(rng, 300, 40000), 160_000_000 // (m * k))
        c["given_shift"] = rng.random() < 0.5
    elif kind == "assign":
        c["k"] = k = rng.randint(2, 64)
        c["n"] = min(_log_int(rng, 1, 200000), 600_000_000 // (m * k))
        c["dmat"] = rng.random() < 0.3
        if c["dmat"]:
            c["n"] = min(c["n"], 160_000_000 // (m * k))
    elif kind == "ncc":
        c["k"] = k = rng.randint(1, 32)
        c["n"] = min(_log_int(rng, 4, 4000), 4_000_000 // (m * k) + 1)
    elif kind == "align":
        c["n"] = min(_log_int(rng, 50, 50000), 9_000_000 // m)
    else:
        c["n"] = min(_log_int(rng, 50, 200000), 24_000_000 // m)
    return c


# ------------------------------------------------------------------ the inputs
def _series(g, n, m, classes, sigma):
    """Series of the benchmark's distribution, made on the GPU: per class
    three sines and a bump, each series a scaled, circularly shifted, offset
    copy of its prototype with noise.  Returns (series, class of each)."""
    d = torch.device("cuda")

    def u(*shape):
        return torch.rand(*shape, generator=g, device=d, dtype=torch.float64)

    t = torch.arange(m, device=d, dtype=torch.float64)
    f = torch.randint(1, 9, (classes, 3, 1), generator=g, device=d).double()
    amp = torch.randn(classes, 3, 1, generator=g, device=d, dtype=torch.float64)
    proto = (amp * torch.sin(2 * math.pi * (f * t / m + u(classes, 3, 1)))).sum(1)
    proto += torch.exp(-((t - m * u(classes, 1)) ** 2) / (2 * (m / 20) ** 2))
    y = torch.randint(0, classes, (n,), generator=g, device=d)
    reach = m // 10
    s = torch.randint(-reach, reach + 1, (n, 1), generator=g, device=d)
    at = (torch.arange(m, device=d)[None, :] - s) % m + y[:, None] * m
    x = proto.float().reshape(-1)[at]
    del at
    x *= (0.5 + 1.5 * u(n, 1)).float()
    x += torch.randn(n, 1, generator=g, device=d)
    x += sigma * torch.randn(n, m, generator=g, device=d)
    return x, y.int()


def _zscore(x, ddof=0):
    x = x.double()
    x = x - x.mean(1, keepdim=True)
    sd = (x.square().sum(1, keepdim=True) / (x.shape[1] - ddof)).sqrt()
    return torch.nan_to_num(x / sd)


def _centroids(g, x, y, k):
    """Centroids as an earlier fit leaves them: one per class, the mean of a
    few members' copies shifted onto the first, z-normalized."""
    n, m = x.shape
    c = torch.empty(k, m, device=x.device, dtype=torch.float64)
    F = _fft_size(m)
    for j in range(k):
        rows = torch.nonzero(y == j)[:24, 0]
        if rows.numel() == 0:
            rows = torch.randint(0, n, (1,), generator=g, device=x.device)
        z = _zscore(x[rows])
        c[j] = _roll_zero(z, _lags(z, z[:1], F)[0][:, 0]).mean(0)
    return _zscore(c, 1).float()


def _wrap(t):
    """A torch tensor as the engine's device array (torch keeps the memory)."""
    return timesc.DeviceArray(_context(), t.data_ptr(), tuple(t.shape),
                              {torch.float32: np.float32, torch.int32: np.int32}[t.dtype])


def _inputs(case, seed):
    g = torch.Generator(device="cuda").manual_seed(int(seed) * 1000003 + 17)
    kind = case["kind"]
    if kind == "batch":
        rng = np.random.default_rng(case["mix"])  # the jobs' sizes, as the benchmark draws them
        jobs = []
        for i in range(case["jobs"]):
            n = int(rng.integers(100, 5001))
            m = int(round(math.exp(rng.uniform(math.log(64), math.log(2048)))))
            k = int(rng.integers(2, 33))
            x, _ = _series(g, n, m, k, 0.3)
            jobs.append((_zscore(x).float(), k, int(seed) * 1000 + i))
        return {"jobs": jobs}
    n, m, k = case["n"], case["m"], case["k"]
    x, y = _series(g, n, m, max(k, 1), case["sigma"])
    s = {}
    if kind == "znorm":
        s["x"] = x
        return s
    s["x"] = _zscore(x).float()
    if kind == "fit":
        s["seed"] = int(seed) + 1
        return s
    # at least a few members of each class to make the centroids from
    few, fy = _series(g, 24 * k, m, k, case["sigma"]) if n < 24 * k else (s["x"], y)
    s["c"] = _centroids(g, few, fy, k)
    if kind == "extract":
        # most series where they belong, some still elsewhere
        other = torch.randint(0, k, (n,), generator=g, device="cuda", dtype=torch.int32)
        stray = torch.rand(n, generator=g, device="cuda") < 0.1
        s["label"] = torch.where(stray, other, y).contiguous()
        if case["given_shift"]:
            own = _own_lag(s["x"], s["c"], s["label"])
            s["shift"] = own.int().contiguous()
    return s


def prepare(case, seed):
    s = _inputs(case, seed)
    kind = case["kind"]
    s["case"] = case
    d = torch.device("cuda")
    if kind == "batch":
        s["specs"] = [{"d": _wrap(x), "k": k, "seed": sd, "max_iter": case["max_iter"]}
                      for x, k, sd in s["jobs"]]
        _workers()
    else:
        n, m, k = case["n"], case["m"], case["k"]
        if kind == "assign":
            s["label"] = torch.empty(n, dtype=torch.int32, device=d)
            s["dist"] = torch.empty(n, dtype=torch.float32, device=d)
            s["shift"] = torch.empty(n, dtype=torch.int32, device=d)
            s["dmat"] = torch.empty(n, k, device=d) if case["dmat"] else None
        elif kind == "ncc":
            s["out"] = torch.empty(n, k, 2 * m - 1, device=d)
        elif kind == "align":
            s["work"] = torch.empty_like(s["x"])
        elif kind == "extract":
            s["new"] = torch.empty_like(s["c"])
        _context()
    torch.cuda.synchronize()  # the engine's stream is its own
    return s


def run(s):
    case, ctx = s["case"], _context()
    kind = case["kind"]
    if kind == "fit":
        r = ctx.fit(_wrap(s["x"]), case["k"], max_iter=case["max_iter"], seed=s["seed"])
        return {"labels": r["labels"], "centroids": r["centroids"],
                "iterations": r["stats"]["iterations"]}
    if kind == "batch":
        res = _workers().run(s["specs"], grouped=True)
        return {"labels": np.concatenate([r["labels"] for r in res]),
                "centroids": np.concatenate([r["centroids"].ravel() for r in res]),
                "iterations": np.array([r["stats"]["iterations"] for r in res])}
    n, m, k = case["n"], case["m"], case["k"]
    if kind == "assign":
        timesc.check(ctx.lib.tcx_assign(
            ctx.h, s["x"].data_ptr(), s["c"].data_ptr(), n, m, k, s["label"].data_ptr(),
            s["dist"].data_ptr(), s["shift"].data_ptr(),
            None if s["dmat"] is None else s["dmat"].data_ptr()))
        return {"label": s["label"], "dist": s["dist"], "shift": s["shift"], "dmat": s["dmat"]}
    if kind == "ncc":
        timesc.check(ctx.lib.tcx_ncc(ctx.h, s["x"].data_ptr(), s["c"].data_ptr(),
                                     s["out"].data_ptr(), n, k, m))
        return s["out"]
    if kind == "align":  # in place, and the program keeps its series
        s["work"].copy_(s["x"])
        torch.cuda.current_stream().synchronize()  # the engine's stream is its own
        ctx.sbd_align(_wrap(s["work"]), _wrap(s["c"]))
        return s["work"]
    if kind == "extract":  # old centroids in, new ones out, and the old are kept
        s["new"].copy_(s["c"])
        torch.cuda.current_stream().synchronize()
        filled = ctx.extract_shape(_wrap(s["label"]), _wrap(s["x"]),
                                   _wrap(s["shift"]) if "shift" in s else None, _wrap(s["new"]))
        return {"centroids": s["new"], "filled": filled}
    ctx.znorm(_wrap(s["x"]), ddof=0)  # in place
    return s["x"]


# ------------------------------------------------------------ 64-bit results
def _fft_size(m):
    return 1 << (2 * m - 1).bit_length()


def _ncc64(x, c, F):
    """Normalized correlations [n, k, 2m-1] of the rows of x with those of c."""
    m = x.shape[1]
    x, c = x.double(), c.double()
    p = torch.fft.rfft(x, F)[:, None] * torch.fft.rfft(c, F).conj()[None]
    cc = torch.fft.irfft(p, F)
    cc = torch.cat([cc[..., F - (m - 1):], cc[..., :m]], -1)
    den = x.norm(dim=1)[:, None] * c.norm(dim=1)[None]
    return torch.where(den[..., None] > 0, cc / den.clamp_min(1e-300)[..., None], 0.0)


def _chunks(n, F, k):
    step = max(1, (1 << 26) // (F * k))
    return [(a, min(a + step, n)) for a in range(0, n, step)]


def _lags(x, c, F):
    """(lag of the largest correlation, its value), [n, k] each."""
    lag = torch.empty(x.shape[0], c.shape[0], dtype=torch.int64, device=x.device)
    val = torch.empty(x.shape[0], c.shape[0], dtype=torch.float64, device=x.device)
    for a, b in _chunks(x.shape[0], F, c.shape[0]):
        v, at = _ncc64(x[a:b], c, F).max(-1)
        val[a:b], lag[a:b] = v, at - (x.shape[1] - 1)
    return lag, val


def _own_lag(x, c, label):
    lag, _ = _lags(x, c, _fft_size(x.shape[1]))
    return lag.gather(1, label.long()[:, None])[:, 0]


def _roll_zero(x, lag):
    """out[t] = x[t - lag], zeros outside."""
    m = x.shape[1]
    src = torch.arange(m, device=x.device)[None] - lag[:, None]
    return torch.where((src >= 0) & (src < m), x.gather(1, src.clamp(0, m - 1)), 0.0)


_MASK = (1 << 64) - 1


def _mix(z):
    z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & _MASK
    z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & _MASK
    return z ^ (z >> 31)


def _power_start(cluster, m):
    """The documented start vector of seed 0, iteration 0."""
    h = _mix(0x9E3779B97F4A7C15)
    h = _mix(h ^ ((0xD1B54A32D192ED03 * (cluster + 1)) & _MASK))
    return np.array([(_mix(h ^ ((0x8CB92BA72F3D8DD7 * (i + 1)) & _MASK)) >> 11) * 2.0 ** -53
                     for i in range(m)])


def _extract64(s, k):
    x, c, label = s["x"], s["c"], s["label"].long()
    m = x.shape[1]
    lag = s["shift"].long() if "shift" in s else _own_lag(x, c, label)
    out = torch.zeros(k, m, dtype=torch.float64, device=x.device)
    for j in range(k):
        rows = torch.nonzero(label == j)[:, 0]
        if rows.numel() == 0:
            continue
        a = _roll_zero(x[rows].double(), lag[rows])
        y = _zscore(a, 1)
        y = y - y.mean(1, keepdim=True)
        p = y.T @ y
        v = torch.from_numpy(_power_start(j, m)).to(x.device)
        left = min(m, 1000)
        while left:  # p^left v
            if left & 1:
                v = p @ v
                v = v / v.norm()
            left >>= 1
            if left:
                p = p @ p
                p = p / p.norm()
        if (a[0] - v).norm() >= (a[0] + v).norm():
            v = -v
        out[j] = _zscore(v[None], 1)[0]
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind in ("fit", "batch"):  # a fit's steps depend on the labels on the way
        return None
    s = _inputs(case, seed)
    F = _fft_size(case["m"])
    if kind == "znorm":
        return _zscore(s["x"])
    if kind == "assign":
        _, v = _lags(s["x"], s["c"], F)
        return {"label": None, "dist": (1 - v).min(1)[0], "shift": None,
                "dmat": 1 - v if case["dmat"] else None}
    if kind == "ncc":
        out = torch.empty(case["n"], case["k"], 2 * case["m"] - 1, dtype=torch.float64,
                          device="cuda")
        for a, b in _chunks(case["n"], F, case["k"]):
            out[a:b] = _ncc64(s["x"][a:b], s["c"], F)
        return out
    if kind == "align":
        return _roll_zero(s["x"].double(), _lags(s["x"], s["c"], F)[0][:, 0])
    return {"centroids": _extract64(s, case["k"]), "filled": None}


# -------------------------------------------------------- what it cannot do without
def _fit_work(n, m, k, iters):
    """The series read once, labels and centroids written once; one forward
    transform of each series, then per iteration one inverse transform of
    each (its own centroid's correlation) and the upper triangle of S."""
    F = _fft_size(m)
    t = 2.5 * F * math.log2(F)
    return {"bytes": 4 * n * m + 4 * n + 4 * k * m,
            "flops": n * t + iters * (n * (t + 3 * F + 2 * m) + n * m * (m + 1.0))}


def work(case):
    kind = case["kind"]
    if kind == "batch":  # the mean job: n 2550, m 570, k 17
        w = _fit_work(2550, 570, 17, case["least_iters"])
        return {q: v * case["jobs"] for q, v in w.items()}
    n, m, k = case["n"], case["m"], case["k"]
    F = _fft_size(m)
    t = 2.5 * F * math.log2(F)  # one real transform of length F
    one = t + 3 * F + 2 * m     # one correlation from two spectra, and its maximum
    if kind == "fit":
        return _fit_work(n, m, k, case["least_iters"])
    if kind == "znorm":
        return {"bytes": 8 * n * m, "flops": 6 * n * m}
    if kind == "align":
        return {"bytes": 8 * n * m + 4 * m, "flops": (n + 1) * t + n * one}
    if kind == "ncc":
        return {"bytes": 4 * (n + k) * m + 4 * n * k * (2 * m - 1),
                "flops": (n + k) * t + n * k * one}
    if kind == "extract":
        aligned = 0 if case["given_shift"] else (n + k) * t + n * one
        return {"bytes": 4 * n * m + 4 * n + 8 * k * m,
                "flops": aligned + n * m * (m + 1.0) + 6 * n * m}
    pairs = n * k if case["dmat"] else n  # without all distances: the nearest one's
    return {"bytes": 4 * (n + k) * m + 12 * n + (4 * n * k if case["dmat"] else 0),
            "flops": (n + k) * t + pairs * one}
