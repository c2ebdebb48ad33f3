"""The work whose speed counts: one call of each family of the package, over the sizes that its users bring.

A case is a dict of plain values. ``kind`` names the family and the other entries its sizes and options:

* ``rolling``      move_* over the last axis of (rows, n);
* ``rolling0``     move_* over the first axis of (n, d1, d2), the layout of (time, latitude, longitude) arrays;
* ``ewm``          move_exp_nan* over the last axis, with a Python-float alpha;
* ``group``        group_nan* of (rows, n) by one label vector;
* ``fill``         ffill / bfill over the last axis;
* ``reduce``       plain reductions, over the first axis of (n, d1, d2) or over the last of (rows, n);
* ``factorize``    sorted factorisation of a label column;
* ``matrix``       correlation / covariance matrices of (batch, vars, obs);
* ``move_matrix``  moving and exponential matrices of (obs, vars);
* ``ragged``       move_mean and group_nanmean of many series of uneven lengths in one launch.

Inputs live on the GPU. Sizes follow the configurations that the benchmark measures, and generic ones.
"""

from __future__ import annotations

import math

import numpy as np
import torch

import numbagg_amd as nb
from numbagg_amd import ragged

DEV = "cuda"
_DT = {"f32": torch.float32, "f64": torch.float64, "i32": torch.int32, "i64": torch.int64}
_SIZE = {"f32": 4, "f64": 8, "i32": 4, "i64": 8}
PAIR_FUNCS = ("move_cov", "move_corr", "move_exp_nancov", "move_exp_nancorr")


def listed():
    return [
        # the smallest ordinary call: 100 short float64 series, a 20-step mean; launch and host time
        {"name": "rolling_small", "kind": "rolling", "func": "move_mean", "dtype": "f64", "rows": 100, "n": 10_000,
         "window": 20, "min_count": 20, "data": "normal", "p_nan": 0.1},
        # long windows over long price-like walks, two inputs: a correlation screen
        {"name": "rolling_corr", "kind": "rolling", "func": "move_corr", "dtype": "f32", "rows": 256, "n": 2_000_000,
         "window": 1000, "min_count": 500, "data": "walk", "p_nan": 0.02},
        # ten years of daily maps (time first, odd sizes), a 30-day mean along time
        {"name": "rolling_time_first", "kind": "rolling0", "func": "move_mean", "dtype": "f32", "n": 3653, "d1": 181,
         "d2": 360, "window": 30, "min_count": 15, "data": "normal", "p_nan": 0.05},
        # exponentially weighted volatility of many long series
        {"name": "ewm_var", "kind": "ewm", "func": "move_exp_nanvar", "dtype": "f32", "rows": 256, "n": 2_000_000,
         "alpha": 0.01, "data": "walk", "p_nan": 0.02},
        # one long float64 series: no rows to spread over the chip
        {"name": "ewm_one_series", "kind": "ewm", "func": "move_exp_nanmean", "dtype": "f64", "rows": 1,
         "n": 10_000_000, "alpha": 0.1, "data": "normal", "p_nan": 0.1},
        # variance per group of a wide table, 1000 groups
        {"name": "group_var", "kind": "group", "func": "group_nanvar", "dtype": "f32", "rows": 64, "n": 4_000_000,
         "labels": 1000, "label_dtype": "i32", "skew": "uniform", "p_nan": 0.05},
        # gaps filled in a large array of sensor series, runs of missing values
        {"name": "fill_large", "kind": "fill", "func": "ffill", "dtype": "f32", "rows": 1024, "n": 1_000_000,
         "limit": 0},
        # the time variance of each map cell (reduction over the first axis)
        {"name": "reduce_time_first", "kind": "reduce", "func": "nanvar", "dtype": "f32", "axis": 0, "n": 3653,
         "d1": 181, "d2": 360, "p_nan": 0.05},
        # a column of 16M keys with 1000 distinct ones turned into group codes
        {"name": "factorize", "kind": "factorize", "dtype": "i64", "n": 16_000_000, "uniques": 1000},
        # many small correlation matrices
        {"name": "matrix_batch", "kind": "matrix", "func": "nancorrmatrix", "dtype": "f32", "batch": 30_000, "nv": 5,
         "obs": 1000, "p_nan": 0.02},
        # the rolling correlation matrix of 32 series
        {"name": "move_matrix", "kind": "move_matrix", "func": "move_corrmatrix", "dtype": "f32", "obs": 200_000,
         "nv": 32, "window": 20, "alpha": 0.0, "p_nan": 0.02},
        # a serving batch: 2000 series of 100 to 1M values, each smoothed and grouped by its own labels
        {"name": "ragged", "kind": "ragged", "series": 2000, "window": 50},
    ]


# --------------------------------------------------------------------------
# more cases of the same ranges
# --------------------------------------------------------------------------
def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["rolling", "rolling0", "ewm", "group", "fill", "reduce", "factorize", "matrix", "move_matrix",
                       "ragged"])
    dtype = rng.choice(["f32", "f32", "f64"])
    half = 1 if dtype == "f32" else 2
    if kind == "rolling":
        rows = _log(rng, 1, 512)
        n = max(1000, _log(rng, 1e5, 4e8 / half) // rows)
        window = _log(rng, 5, 1000)
        func = rng.choice(["move_sum", "move_mean", "move_std", "move_var", "move_cov", "move_corr"])
        return {"kind": kind, "func": func, "dtype": dtype, "rows": rows, "n": n, "window": window,
                "min_count": max(2, window // 2), "data": rng.choice(["walk", "normal"]), "p_nan": 0.02}
    if kind == "rolling0":
        d1, d2 = _log(rng, 20, 400), _log(rng, 20, 400)
        n = min(_log(rng, 200, 8000), int(2.3e8 / half) // (d1 * d2))
        window = _log(rng, 5, 100)
        func = rng.choice(["move_sum", "move_mean", "move_std", "move_corr"])
        return {"kind": kind, "func": func, "dtype": dtype, "n": n, "d1": d1, "d2": d2, "window": window,
                "min_count": max(2, window // 2), "data": "normal", "p_nan": 0.05}
    if kind == "ewm":
        rows = _log(rng, 1, 512)
        n = max(1000, _log(rng, 1e5, 3e8 / half) // rows)
        func = "move_exp_nan" + rng.choice(["mean", "mean", "sum", "var", "std", "cov", "corr", "count"])
        return {"kind": kind, "func": func, "dtype": dtype, "rows": rows, "n": n,
                "alpha": rng.choice([0.01, 0.05, 0.1, 0.5]), "data": rng.choice(["walk", "normal"]), "p_nan": 0.05}
    if kind == "group":
        rows = _log(rng, 1, 128)
        n = max(1000, _log(rng, 1e5, 2.5e8 / half) // rows)
        func = "group_nan" + rng.choice(["sum", "mean", "var", "std", "count", "argmax", "first", "min"])
        return {"kind": kind, "func": func, "dtype": dtype, "rows": rows, "n": n, "labels": _log(rng, 5, 20_000),
                "label_dtype": rng.choice(["i32", "i64"]), "skew": rng.choice(["uniform", "zipf"]), "p_nan": 0.05}
    if kind == "fill":
        rows = _log(rng, 1, 1024)
        n = max(1000, _log(rng, 1e5, 8e8 / half) // rows)
        return {"kind": kind, "func": rng.choice(["ffill", "bfill"]), "dtype": dtype, "rows": rows, "n": n,
                "limit": rng.choice([0, 16])}
    if kind == "reduce":
        func = rng.choice(["nansum", "nanmean", "nanvar", "nanstd", "nanmax", "nancount"])
        case = {"kind": kind, "func": func, "dtype": dtype, "axis": rng.choice([0, 0, -1])}
        if case["axis"] == 0:
            case["d1"], case["d2"] = _log(rng, 20, 400), _log(rng, 20, 400)
            case["n"] = min(_log(rng, 200, 20_000), int(4e8 / half) // (case["d1"] * case["d2"]))
        else:
            case["d1"], case["d2"] = _log(rng, 1, 512), 1
            case["n"] = max(1000, _log(rng, 1e5, 5e8 / half) // case["d1"])
        return dict(case, p_nan=0.05)
    if kind == "factorize":
        return {"kind": kind, "dtype": rng.choice(["i64", "i64", "i32", "f64"]), "n": _log(rng, 1e5, 3e7),
                "uniques": _log(rng, 10, 50_000)}
    if kind == "matrix":
        nv = _log(rng, 3, 128)
        obs = _log(rng, 100, 100_000)
        size = min(_log(rng, 1e5, 1.5e8 / half), int(5e10 / (6 * (nv + 1))))
        return {"kind": kind, "func": rng.choice(["nancorrmatrix", "nancovmatrix"]), "dtype": dtype,
                "batch": max(1, min(30_000, size // (nv * obs))), "nv": nv, "obs": obs, "p_nan": 0.02}
    if kind == "move_matrix":
        nv = _log(rng, 3, 48)
        obs = max(500, min(_log(rng, 1000, 400_000), int(2e8 / half) // (nv * nv)))
        func = rng.choice(["move_corrmatrix", "move_covmatrix", "move_exp_nancorrmatrix", "move_exp_nancovmatrix"])
        return {"kind": kind, "func": func, "dtype": dtype, "obs": obs, "nv": nv, "window": _log(rng, 10, 200),
                "alpha": rng.choice([0.05, 0.1, 0.5]), "p_nan": 0.02}
    return {"kind": kind, "series": _log(rng, 50, 2000), "window": _log(rng, 10, 100)}


# --------------------------------------------------------------------------
# inputs
# --------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _chunks(rows, n, most=1 << 25):
    step = max(1, most // max(1, n))
    return [(r, min(rows, r + step)) for r in range(0, rows, step)]


def _values(g, rows, n, dtype, data, p_nan):
    """(rows, n): N(0, 1), or random walks about 1e4, with missing values."""
    out = torch.empty((rows, n), dtype=_DT[dtype], device=DEV)
    for r0, r1 in _chunks(rows, n):
        if data == "walk":
            v = torch.randn((r1 - r0, n), generator=g, device=DEV, dtype=torch.float64)
            v = torch.cumsum(v, dim=1).add_(1e4).to(_DT[dtype])
        else:
            v = torch.randn((r1 - r0, n), generator=g, device=DEV, dtype=_DT[dtype])
        v.masked_fill_(torch.rand((r1 - r0, n), generator=g, device=DEV) < p_nan, math.nan)
        out[r0:r1] = v
    return out


def _with_runs(g, rows, n, dtype, mean_nan=50.0, mean_valid=116.7):
    """N(0, 1) values whose missing ones come in runs of geometric length (30% of all)."""
    out = torch.empty((rows, n), dtype=_DT[dtype], device=DEV)
    k = int(n / (mean_nan + mean_valid) * 1.3) + 64
    for r0, r1 in _chunks(rows, n):
        m = r1 - r0
        u = torch.rand((m, k, 2), generator=g, device=DEV, dtype=torch.float64)
        rate = torch.tensor([math.log(1 - 1 / mean_valid), math.log(1 - 1 / mean_nan)], device=DEV)
        ends = torch.cumsum((torch.log(u) / rate).floor_().long().add_(1).reshape(m, 2 * k), dim=1)
        ends -= (torch.rand((m, 1), generator=g, device=DEV) * (mean_nan + mean_valid)).long()
        ends.clamp_(0, n)
        delta = torch.zeros((m, n + 1), dtype=torch.int16, device=DEV)
        one = torch.ones((m, k), dtype=torch.int16, device=DEV)
        delta.scatter_add_(1, ends[:, 0::2], one)
        delta.scatter_add_(1, ends[:, 1::2], -one)
        v = torch.randn((m, n), generator=g, device=DEV, dtype=_DT[dtype])
        v.masked_fill_(torch.cumsum(delta[:, :n], dim=1, dtype=torch.int16) > 0, math.nan)
        out[r0:r1] = v
    return out


def _zipf_labels(g, count, k, s=1.1):
    """`count` labels below `k` (a number, or one per value), the first ones the most frequent."""
    u = torch.rand(count, generator=g, device=DEV, dtype=torch.float64)
    kf = k.double() if isinstance(k, torch.Tensor) else float(k)
    a = s - 1.0
    lab = torch.floor((1.0 - u * (1.0 - kf ** -a)) ** (-1.0 / a)).long() - 1
    return torch.minimum(lab, k - 1) if isinstance(k, torch.Tensor) else lab.clamp_(max=k - 1)


def _pair(case):
    return case["func"] in PAIR_FUNCS


def _ragged_shape(case):
    s = case["series"]
    rng = np.random.default_rng(s)
    lengths = np.round(np.exp(rng.uniform(np.log(100), np.log(1e6), s))).astype(np.int64)
    ks = np.round(np.exp(rng.uniform(np.log(10), np.log(1e5), s))).astype(np.int64)
    return lengths, ks


def _inputs(case, seed):
    g, kind = _gen(seed), case["kind"]
    if kind in ("rolling", "ewm"):
        return [_values(g, case["rows"], case["n"], case["dtype"], case["data"], case["p_nan"])
                for _ in range(1 + _pair(case))]
    if kind == "rolling0":
        return [_values(g, case["n"], case["d1"] * case["d2"], case["dtype"], case["data"], case["p_nan"])
                .view(case["n"], case["d1"], case["d2"]) for _ in range(1 + _pair(case))]
    if kind == "group":
        v = _values(g, case["rows"], case["n"], case["dtype"], "normal", case["p_nan"])
        if case["skew"] == "zipf":
            lab = _zipf_labels(g, case["n"], case["labels"])
        else:
            lab = torch.randint(0, case["labels"], (case["n"],), generator=g, device=DEV)
        return [v, lab.to(_DT[case["label_dtype"]])]
    if kind == "fill":
        return [_with_runs(g, case["rows"], case["n"], case["dtype"])]
    if kind == "reduce":
        if case["axis"] == 0:
            x = _values(g, case["n"], case["d1"] * case["d2"], case["dtype"], "normal", case["p_nan"])
            return [x.view(case["n"], case["d1"], case["d2"])]
        return [_values(g, case["d1"], case["n"], case["dtype"], "normal", case["p_nan"])]
    if kind == "factorize":
        keys = torch.randint(0, case["uniques"], (case["n"],), generator=g, device=DEV) * 7919 - 500_000
        return [keys.to(_DT[case["dtype"]])]
    if kind == "matrix":
        x = _values(g, case["batch"] * case["nv"], case["obs"], case["dtype"], "normal", case["p_nan"])
        return [x.view(case["batch"], case["nv"], case["obs"])]
    if kind == "move_matrix":
        return [_values(g, case["obs"], case["nv"], case["dtype"], "normal", case["p_nan"])]
    lengths, ks = _ragged_shape(case)
    total = int(lengths.sum())
    values = _values(g, 1, total, "f32", "normal", 0.05).view(-1)
    labels = torch.empty(total, dtype=torch.int32, device=DEV)
    offs = np.concatenate([[0], np.cumsum(lengths)])
    for s0 in range(0, case["series"], 500):
        s1 = min(case["series"], s0 + 500)
        k = torch.repeat_interleave(torch.from_numpy(ks[s0:s1]).to(DEV), torch.from_numpy(lengths[s0:s1]).to(DEV))
        labels[int(offs[s0]):int(offs[s1])] = _zipf_labels(g, k.numel(), k).to(torch.int32)
    return [values, labels]


def prepare(case, seed):
    x = _inputs(case, seed)
    kind = case["kind"]
    if kind in ("rolling", "rolling0"):
        kw = {"window": case["window"], "min_count": case["min_count"], "axis": -1 if kind == "rolling" else 0}
    elif kind == "ewm":
        kw = {"alpha": case["alpha"]}
    elif kind == "group":
        kw = {"num_labels": case["labels"], "axis": -1}
    elif kind == "fill":
        kw = {"limit": case["limit"] or None}
    elif kind == "reduce":
        kw = {"axis": case["axis"]}
    elif kind == "factorize":
        kw = {"sort": True}
    elif kind == "matrix":
        kw = {}
    elif kind == "move_matrix":
        kw = {"alpha": case["alpha"]} if "exp" in case["func"] else {"window": case["window"],
                                                                    "min_count": case["window"] // 2}
    else:
        lengths, ks = _ragged_shape(case)
        plan = ragged.RaggedMoveMeanGroupMean(lengths, ks, window=case["window"], strategy="lds", lds_labels=4096)
        return {"call": plan, "x": x, "kw": {}}
    return {"call": getattr(nb, case["func"] if kind != "factorize" else "factorize"), "x": x, "kw": kw}


def run(state):
    return state["call"](*state["x"], **state["kw"])


def work(case):
    kind = case["kind"]
    if kind == "ragged":
        lengths, ks = _ragged_shape(case)
        return {"bytes": 12.0 * lengths.sum() + 4.0 * ks.sum(), "flops": 2.0 * lengths.sum()}
    es = _SIZE[case["dtype"]]
    if kind in ("rolling", "rolling0", "ewm"):
        elems = case["rows"] * case["n"] if kind != "rolling0" else case["n"] * case["d1"] * case["d2"]
        out = 8 if kind == "ewm" else es  # a Python-float alpha makes the output float64
        return {"bytes": elems * (es * (1 + _pair(case)) + out), "flops": elems * 4.0 * (1 + 2 * _pair(case))}
    if kind == "group":
        elems = case["rows"] * case["n"]
        return {"bytes": elems * es + case["n"] * _SIZE[case["label_dtype"]] + case["rows"] * case["labels"] * es,
                "flops": elems * 2.0}
    if kind == "fill":
        return {"bytes": case["rows"] * case["n"] * 2 * es, "flops": 0.0}
    if kind == "reduce":
        cells = case["d1"] * case["d2"]
        return {"bytes": cells * (case["n"] * es + 8), "flops": 3.0 * cells * case["n"]}
    if kind == "factorize":
        return {"bytes": case["n"] * (es + 8) + case["uniques"] * es, "flops": 0.0}
    if kind == "matrix":
        pairs = case["nv"] * (case["nv"] + 1) // 2
        products = 6 if "corr" in case["func"] else 4
        return {"bytes": case["batch"] * case["nv"] * (case["obs"] + case["nv"]) * es,
                "flops": 2.0 * products * pairs * case["obs"] * case["batch"]}
    out = 8 if "exp" in case["func"] else es
    pairs = case["nv"] * (case["nv"] + 1) // 2
    return {"bytes": case["obs"] * case["nv"] * (es + case["nv"] * out), "flops": 12.0 * case["obs"] * pairs}


# --------------------------------------------------------------------------
# the same in 64 bits, in plain torch
# --------------------------------------------------------------------------
def _window_sum(x, w):
    """Sums of the last `w` entries along the last axis, added up from the two blocks of length `w` that a window
    meets (the tail of one, the head of the next), so that nothing is subtracted."""
    rows, n = x.shape
    w = int(w)
    blocks = (n + w - 1) // w + 1
    p = torch.zeros((rows, blocks * w), dtype=torch.float64, device=x.device)
    p[:, w:w + n] = x
    b = p.view(rows, blocks, w)
    head = torch.cumsum(b, dim=2).view(rows, -1)
    tail = torch.flip(torch.cumsum(torch.flip(b, (2,)), dim=2), (2,)).reshape(rows, -1)
    tail.view(rows, blocks, w)[:, :, 0] = 0  # a window that is one whole block is its head alone
    return head[:, w:w + n] + tail[:, 1:n + 1]


def _decayed_sum(x, d):
    """s[i] = d s[i - 1] + x[i] along the last axis, by doubling."""
    s, k, f = x.clone(), 1, float(d)
    while k < x.shape[-1] and f > 1e-40:
        s[..., k:] += f * s[..., :-k].clone()
        k, f = 2 * k, f * f
    return s


def _masked(xs):
    """The valid mask of all arrays, and each array in float64 about its row's mean with 0 where that is not valid."""
    ok = ~torch.isnan(xs[0])
    for x in xs[1:]:
        ok = ok & ~torch.isnan(x)
    out = []
    for x in xs:
        y = torch.where(ok, x.double(), torch.zeros((), dtype=torch.float64, device=x.device))
        level = y.sum(dim=-1, keepdim=True) / ok.sum(dim=-1, keepdim=True).clamp(min=1)
        out.append((torch.where(ok, y - level, torch.zeros_like(y)), level))
    return ok, out


def _nan_where(v, bad):
    return v.masked_fill_(bad, math.nan)


def _moment(func, total, w, ys):
    """A statistic from sums: `total` sums the last axis, `w` holds the summed weights, `ys` the shifted values with
    their levels; and w - 1 for an unbiased one."""
    (y, level), z = ys[0], ys[-1][0]
    if func.endswith("sum"):
        return total(y) + level * w
    s = total(y)
    if func.endswith("mean"):
        return s / w + level
    t = total(z) if z is not y else s
    c = total(y * z) - s * t / w
    if func.endswith("corr"):
        return c / torch.sqrt((total(y * y) - s * s / w) * (total(z * z) - t * t / w))
    return c


def _exact_rolling(func, xs, window, min_count):
    ok, ys = _masked(xs)
    cnt = _window_sum(ok.double(), window).round_()
    v = _moment(func, lambda a: _window_sum(a, window), cnt, ys)
    if func[5:] in ("var", "std", "cov"):
        v = v / (cnt - 1)
    if func == "move_std":
        v = torch.sqrt(v)
    least = {"move_sum": min_count, "move_mean": max(1, min_count), "move_corr": max(1, min_count)}
    return _nan_where(v, cnt < least.get(func, max(2, min_count)))


def _exact_ewm(func, xs, alpha):
    d = 1.0 - alpha
    ok, ys = _masked(xs)
    w = _decayed_sum(ok.double(), d)
    if func.endswith("count"):
        return w
    seen = torch.cumsum(ok, dim=-1)
    v = _moment(func, lambda a: _decayed_sum(a, d), w, ys)
    if func.endswith("mean") or func.endswith("sum"):
        return _nan_where(v, seen < 1)
    if not func.endswith("corr"):
        v = v / w / (1.0 - _decayed_sum(ok.double(), d * d) / (w * w))
    if func.endswith("std"):
        v = torch.sqrt(v)
    return _nan_where(v, seen < 2)


def _by_rows(fn, xs, most=1 << 24):
    rows, n = xs[0].shape
    out = torch.empty((rows, n), dtype=torch.float64, device=DEV)
    for r0, r1 in _chunks(rows, n, most):
        out[r0:r1] = fn([x[r0:r1] for x in xs])
    return out


def _exact_group(case, v, lab):
    func, k = case["func"][9:], case["labels"]
    if func not in ("sum", "mean", "var", "std", "count"):
        return None
    order = torch.argsort(lab, stable=True)
    sizes = torch.bincount(lab, minlength=k)
    out = torch.empty((case["rows"], k), dtype=torch.float64, device=DEV)
    zero = torch.zeros((), dtype=torch.float64, device=DEV)

    def total(a):
        return torch.segment_reduce(a, "sum", lengths=sizes, axis=0, unsafe=True)

    for r in range(case["rows"]):
        x = v[r, order].double()
        ok = ~torch.isnan(x)
        x = torch.where(ok, x, zero)
        cnt, s = total(ok.double()), total(x)
        if func == "count":
            out[r] = cnt
        elif func == "sum":
            out[r] = s
        elif func == "mean":
            out[r] = _nan_where(s / cnt, cnt < 1)
        else:
            dev = torch.where(ok, x - torch.repeat_interleave(s / cnt, sizes), zero)
            var = _nan_where(total(dev * dev) / (cnt - 1), cnt < 2)
            out[r] = torch.sqrt(var) if func == "std" else var
    return out


def _exact_fill(case, x):
    if case["func"] == "bfill":
        return torch.flip(_exact_fill(dict(case, func="ffill"), torch.flip(x, (1,))), (1,))
    out = torch.empty(x.shape, dtype=torch.float64, device=DEV)
    at = torch.arange(x.shape[1], device=DEV)
    limit = case["limit"] or x.shape[1]
    for r0, r1 in _chunks(*x.shape):
        part = x[r0:r1]
        last = torch.cummax(torch.where(torch.isnan(part), -1, at), dim=1).values
        v = torch.gather(part, 1, last.clamp(min=0)).double()
        out[r0:r1] = _nan_where(v, (last < 0) | (at - last > limit))
    return out


def _exact_reduce(case, x):
    dim, func = (0 if case["axis"] == 0 else 1), case["func"]
    if func in ("nancount", "nanmax"):  # whole numbers; a copied value
        return None
    parts = []
    y = x.reshape(case["n"], -1) if dim == 0 else x
    for c0, c1 in _chunks(y.shape[1 - dim], y.shape[dim]):
        v = (y[:, c0:c1] if dim == 0 else y[c0:c1]).double()
        ok = ~torch.isnan(v)
        cnt = ok.sum(dim=dim).double()
        v = v.nan_to_num_(nan=0.0)
        s = v.sum(dim=dim)
        if func == "nansum":
            parts.append(s)
            continue
        mean = s / cnt
        if func == "nanmean":
            parts.append(mean)
            continue
        dev = torch.where(ok, v - mean.unsqueeze(dim), torch.zeros_like(v))
        var = (dev * dev).sum(dim=dim) / (cnt - 1)
        parts.append(torch.sqrt(var) if func == "nanstd" else var)
    r = torch.cat(parts)
    return r.view(case["d1"], case["d2"]) if dim == 0 else r


def _exact_matrix(case, x):
    nv, corr = case["nv"], "corr" in case["func"]
    out = torch.empty((case["batch"], nv, nv), dtype=torch.float64, device=DEV)
    for b0, b1 in _chunks(case["batch"], nv * case["obs"]):
        v = x[b0:b1].double()
        ok = ~torch.isnan(v)
        m = ok.double()
        y = v.nan_to_num_(nan=0.0)
        y = (y - y.sum(dim=2, keepdim=True) / m.sum(dim=2, keepdim=True)) * m
        mt, yt = m.transpose(1, 2).contiguous(), y.transpose(1, 2).contiguous()
        n, p, si = torch.matmul(m, mt), torch.matmul(y, yt), torch.matmul(y, mt)
        sj = si.transpose(1, 2)
        c = p - si * sj / n
        if corr:
            q = torch.matmul(y * y, mt)
            c = c / torch.sqrt((q - si * si / n) * (q.transpose(1, 2) - sj * sj / n))
            out[b0:b1] = _nan_where(c, n < 2)
        else:
            out[b0:b1] = _nan_where(c / (n - 1), n < 2)
    return out


def _exact_move_matrix(case, x):
    cols = x.t().contiguous()
    nv = case["nv"]
    out = torch.empty((case["obs"], nv, nv), dtype=torch.float64, device=DEV)
    name = case["func"].replace("matrix", "")
    for i in range(nv):
        xs = [cols[i:i + 1].expand(nv, -1), cols]
        if "exp" in name:
            v = _exact_ewm(name, xs, case["alpha"])
        else:
            v = _exact_rolling(name, xs, case["window"], max(2, case["window"] // 2))
        out[:, i] = v.t()
    return out


def _exact_ragged(case, values, labels):
    lengths, ks = _ragged_shape(case)
    w = case["window"]
    ln = torch.from_numpy(lengths).to(DEV)
    start = torch.repeat_interleave(torch.cumsum(ln, 0) - ln, ln)
    pos = torch.arange(values.numel(), device=DEV) - start
    ok = ~torch.isnan(values)
    v = values.double().nan_to_num_(nan=0.0)
    s, c = v.clone(), ok.to(torch.int32)
    for k in range(1, w):
        inside = pos[k:] >= k
        s[k:] += v[:-k] * inside
        c[k:] += ok[:-k] & inside
    moved = _nan_where(s / w, c < w)
    kt = torch.from_numpy(ks).to(DEV)
    flat = torch.repeat_interleave(torch.cumsum(kt, 0) - kt, ln) + labels
    gs = torch.zeros(int(ks.sum()), dtype=torch.float64, device=DEV).index_add_(0, flat, v)
    gc = torch.zeros_like(gs).index_add_(0, flat, ok.double())
    return moved, _nan_where(gs / gc, gc < 1)


def exact(case, seed):
    kind = case["kind"]
    if kind == "factorize":  # whole numbers and copied keys
        return None
    x = _inputs(case, seed)
    if kind == "rolling":
        return _by_rows(lambda a: _exact_rolling(case["func"], a, case["window"], case["min_count"]), x)
    if kind == "rolling0":
        rows = [a.view(case["n"], -1).t().contiguous() for a in x]
        r = _by_rows(lambda a: _exact_rolling(case["func"], a, case["window"], case["min_count"]), rows)
        return r.t().reshape(x[0].shape)
    if kind == "ewm":
        return _by_rows(lambda a: _exact_ewm(case["func"], a, case["alpha"]), x)
    if kind == "group":
        return _exact_group(case, *x)
    if kind == "fill":
        return _exact_fill(case, *x)
    if kind == "reduce":
        return _exact_reduce(case, *x)
    if kind == "matrix":
        return _exact_matrix(case, *x)
    if kind == "move_matrix":
        return _exact_move_matrix(case, *x)
    return _exact_ragged(case, *x)
