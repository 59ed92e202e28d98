"""The measured workloads of the batch-indicator path.

Every case is one enqueue of a public entry point on inputs that are already
in device memory, as a program that keeps its market data on the GPU calls it:
one-series parameter sweeps (ALMA, EMA, RSI, ADX, Bollinger Bands, weighted
moving averages), packed requests of many lengths, time-major panels of many
series (the fused EMA + RSI + ATR launch, the rolling-window indicators) and
the double-ALMA crossover backtest.  Sizes are those of the repository's own
benchmark and tests.
"""
import ctypes
import functools
import math
import random

import numpy as np
import torch

import vectorta_amd as vta

P = ctypes.c_void_p


def listed():
    return [
        # one indicator on one chart: 100,000 closes, the default ALMA(9, 0.85, 6)
        {"name": "alma_single_100k", "op": "alma", "kernel": "auto", "bars": 100_000,
         "first": 9, "last": 9, "step": 1, "offsets": 1, "sigmas": 1},
        # the headline sweep: 25 periods x 10 offsets x 5 sigmas over 200,000 bars
        {"name": "alma_sweep_200k_x1250", "op": "alma", "kernel": "mfma", "bars": 200_000,
         "first": 10, "last": 250, "step": 10, "offsets": 10, "sigmas": 5},
        # a served ALMA request as a client leaves it: automatic kernel, ragged length
        {"name": "alma_auto_41117_x370", "op": "alma", "kernel": "auto", "bars": 41_117,
         "first": 5, "last": 41, "step": 1, "offsets": 10, "sigmas": 1},
        # EMA of every period on one long series
        {"name": "ema_200k_x1250", "op": "ema", "bars": 200_000, "first": 2, "combos": 1250},
        # a small interactive RSI request, bound by latency and launches
        {"name": "rsi_10007_x33", "op": "rsi", "bars": 10_007, "first": 2, "combos": 33},
        # ADX of every period on one long series (three inputs, two smoothing stages)
        {"name": "adx_200k_x1250", "op": "adx", "bars": 200_000, "first": 2, "combos": 1250},
        # forty queued RSI requests of uneven lengths and grids served together
        {"name": "rsi_pack_40", "op": "pack", "kind": "rsi", "jobs": 40, "shortest": 1_000,
         "longest": 50_000, "grid": 128, "mix": 31},
        # Bollinger Bands over 100 periods x 5 widths, three outputs
        {"name": "bb_60k_x500", "op": "bb", "bars": 60_000, "first": 5, "periods": 100,
         "widths": 5},
        # weighted moving average of every period on one long series
        {"name": "wma_200k_x1250", "op": "fir", "kind": "wma", "bars": 200_000, "first": 2,
         "combos": 1250},
        # end-of-day refresh of a universe: 4,096 tickers of uneven history, right-aligned
        {"name": "ohlc_4096x50000", "op": "ohlc", "series": 4096, "rows": 50_000,
         "shortest": 2_000, "ema": 20, "rsi": 14, "atr": 14, "mix": 3},
        # rolling windows over a panel with price jumps: bands, percentile and deviation
        {"name": "panel_1024x50000", "op": "panel", "series": 1024, "rows": 50_000, "band": 20,
         "rank": 100, "percent": 70.0, "mad": 64},
        # the crossover backtest: 220 fast x 265 slow periods over 200,000 bars
        {"name": "cross_58300_x200k", "op": "cross", "bars": 200_000, "fast": 5, "nfast": 220,
         "slow": 30, "nslow": 265},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: any of the listed entry points, sizes from a single
    request up to the listed ones, odd lengths included."""
    op = rng.choice(["alma", "alma", "ema", "rsi", "adx", "pack", "bb", "fir", "ohlc", "panel",
                     "cross"])
    if op == "alma":
        first = rng.randint(2, 40)
        return {"op": op, "kernel": rng.choice(["auto", "mfma", "mfma_f16x3", "fp32"]),
                "bars": _log(rng, 1_000, 200_000), "first": first,
                "last": first + rng.randint(0, 200), "step": rng.randint(3, 20),
                "offsets": rng.randint(1, 10), "sigmas": rng.randint(1, 3)}
    if op in ("ema", "rsi", "adx"):
        return {"op": op, "bars": _log(rng, 3_000, 200_000), "first": rng.randint(2, 9),
                "combos": _log(rng, 1, 1250)}
    if op == "pack":
        return {"op": op, "kind": rng.choice(["ema", "rsi", "adx"]), "jobs": rng.randint(2, 60),
                "shortest": 1_000, "longest": _log(rng, 2_000, 50_000), "grid": _log(rng, 2, 128),
                "mix": rng.randint(0, 9_999)}
    if op == "bb":
        return {"op": op, "bars": _log(rng, 1_000, 80_000), "first": rng.randint(2, 20),
                "periods": _log(rng, 1, 150), "widths": rng.randint(1, 5)}
    if op == "fir":
        return {"op": op, "kind": rng.choice(["sma", "wma", "swma"]),
                "bars": _log(rng, 3_000, 200_000), "first": rng.randint(2, 9),
                "combos": _log(rng, 1, 1250)}
    if op == "ohlc":
        return {"op": op, "series": _log(rng, 16, 4096), "rows": _log(rng, 3_000, 50_000),
                "shortest": 1_000, "ema": rng.randint(5, 50), "rsi": rng.randint(5, 30),
                "atr": rng.randint(5, 30), "mix": rng.randint(0, 9_999)}
    if op == "panel":
        return {"op": op, "series": _log(rng, 16, 1024), "rows": _log(rng, 2_000, 50_000),
                "band": rng.randint(5, 60), "rank": rng.randint(5, 128),
                "percent": float(rng.choice([5, 25, 50, 70, 90, 100])), "mad": rng.randint(4, 64)}
    fast = rng.randint(2, 40)
    return {"op": "cross", "bars": _log(rng, 2_000, 200_000), "fast": fast,
            "nfast": _log(rng, 4, 200), "slow": fast + rng.randint(1, 40),
            "nslow": _log(rng, 4, 200)}


# ------------------------------------------------------------------ inputs

@functools.lru_cache(maxsize=1)
def _handles():
    """The context (and with it the stream) a program keeps for its lifetime."""
    return vta.CudaAlma(0)


class _Buf:
    """A torch tensor as the device buffer argument of the enqueue-only calls."""

    def __init__(self, t):
        self.t, self.ptr, self.nbytes = t, t.data_ptr(), t.numel() * t.element_size()


def _walk(rows, cols, sd, seed):
    """Geometric random walks from 100, f32 [rows, cols]; the log returns are
    summed as integers, so the values follow from the seed alone."""
    g = torch.Generator(device="cuda").manual_seed(seed * 64)
    r = torch.randn(rows, cols, generator=g, device="cuda", dtype=torch.float32).double()
    r = (r * (sd * 2.0 ** 40)).round_().long()
    r[0] = 0
    return (torch.cumsum(r, 0).double() * 2.0 ** -40).exp_().mul_(100.0).float()


def _high_low(close, seed):
    """high / low = close (1 +/- |N(0, 0.005)|)."""
    g = torch.Generator(device="cuda").manual_seed(seed * 64 + 63)
    up = torch.randn(close.shape, generator=g, device="cuda").abs_().mul_(0.005)
    dn = torch.randn(close.shape, generator=g, device="cuda").abs_().mul_(0.005)
    return close * (1 + up), close * (1 - dn)


def _grid(case):
    """The ALMA sweep's axes; offsets over 0.05 .. 0.95, sigmas 2, 4, ..."""
    no, ns = case["offsets"], case["sigmas"]
    off = (0.05, 0.95, 0.9 / (no - 1)) if no > 1 else (0.85, 0.85, 0.0)
    sig = (2.0, 2.0 * ns, 2.0) if ns > 1 else (6.0, 6.0, 0.0)
    return vta.AlmaBatchRange(period=(case["first"], case["last"], case["step"]), offset=off,
                              sigma=sig)


def _alma_params(case):
    return [(c.period, c.offset, c.sigma) for c in vta.expand_grid(_grid(case))]


def _jobs(case):
    """Lengths and period tables of the packed requests."""
    r = random.Random(case["mix"])
    out = []
    for _ in range(case["jobs"]):
        n = _log(r, case["shortest"], case["longest"])
        c = min(_log(r, 1, case["grid"]), n // 4 - 4)
        out.append((n, [2 + 2 * i for i in range(max(1, min(c, n // 8)))]))
    return out


def _lengths(case):
    """Bars of history of each ticker, log-uniform; the first has them all."""
    r = random.Random(case["mix"])
    n = [min(case["rows"], _log(r, case["shortest"], case["rows"])) for _ in range(case["series"])]
    n[0] = case["rows"]
    return n


def _starts(case):
    return torch.tensor([case["rows"] - n for n in _lengths(case)], device="cuda")


def _ohlc_inputs(case, seed):
    c = _walk(case["rows"], case["series"], 0.01, seed)
    h, lo = _high_low(c, seed)
    gap = torch.arange(case["rows"], device="cuda")[:, None] < _starts(case)[None, :]
    for a in (c, h, lo):
        a.masked_fill_(gap, float("nan"))
    return c, h, lo


def _panel_input(case, seed):
    """Random walks with 1% of the bars moved by five standard deviations."""
    p = _walk(case["rows"], case["series"], 0.01, seed)
    g = torch.Generator(device="cuda").manual_seed(seed * 64 + 62)
    u = torch.rand(p.shape, generator=g, device="cuda")
    return torch.where(u < 0.005, p * 0.95, torch.where(u > 0.995, p * 1.05, p))


def _series(case, seed):
    """close, high, low of one series."""
    c = _walk(case["bars"], 1, 0.015, seed)
    h, lo = _high_low(c, seed)
    return c[:, 0], h[:, 0].contiguous(), lo[:, 0].contiguous()


def _periods(case):
    return torch.arange(case["first"], case["first"] + case["combos"], dtype=torch.int32,
                        device="cuda")


def _empty(*shape):
    return torch.empty(*shape, dtype=torch.float32, device="cuda")


def _ptr(t):
    return P(t.data_ptr())


def _ok(status):
    if status:
        raise vta.VtaError(status, "enqueue failed")


# ------------------------------------------------------------------ the cases

def prepare(case, seed):
    h = _handles()
    s = {"op": case["op"], "case": case, "h": h, "lib": vta.lib(), "ctx": h.ctx}
    op = case["op"]
    if op == "alma":
        s["x"] = _series(case, seed)[0]
        s["plan"] = h.sweep_plan(_grid(case), case["bars"], kernel=case["kernel"])
        s["out"] = _empty(s["plan"].n_combos, case["bars"])
    elif op in ("ema", "rsi", "adx"):
        s["x"], s["high"], s["low"] = _series(case, seed)
        s["periods"] = _periods(case)
        s["out"] = _empty(case["combos"], case["bars"])
        if op == "ema":
            s["ema"] = vta.CudaEma.__new__(vta.CudaEma)    # EMA on the shared context
            s["ema"].ctx = h.ctx
            s["bufs"] = [_Buf(s[k]) for k in ("x", "periods", "out")]
    elif op == "pack":
        s["out"], s["in"], jobs = [], [], []
        walks = _walk(case["longest"], case["jobs"], 0.01, seed).T.contiguous()
        for k, (n, periods) in enumerate(_jobs(case)):
            c = walks[k, :n].clone()
            hi, lo = _high_low(c, seed + k)
            p = torch.tensor(periods, dtype=torch.int32, device="cuda")
            out = _empty(len(periods), n)
            job = {"close": _Buf(c), "periods": _Buf(p), "out": _Buf(out), "series_len": n,
                   "first_valid": 0, "n_combos": len(periods), "max_period": max(periods)}
            if case["kind"] == "adx":
                job["high"], job["low"] = _Buf(hi), _Buf(lo)
            jobs.append(job)
            s["in"].append((c, hi, lo, p))
            s["out"].append(out)
        torch.cuda.synchronize()
        s["pack"] = vta.RecPack(h.ctx, case["kind"], jobs)
    elif op == "bb":
        s["x"] = _series(case, seed)[0]
        n, w = case["periods"], case["widths"]
        p = torch.arange(case["first"], case["first"] + n, dtype=torch.int32, device="cuda")
        s["periods"] = p.repeat_interleave(w)
        s["up"] = (1.0 + 0.5 * torch.arange(w, device="cuda", dtype=torch.float64)).repeat(n)
        s["dn"] = torch.full((n * w,), 2.0, device="cuda", dtype=torch.float64)
        s["out"] = [_empty(n * w, case["bars"]) for _ in range(3)]
    elif op == "fir":
        s["x"] = _series(case, seed)[0]
        s["periods"] = _periods(case)
        s["warms"] = s["periods"] - 1
        s["out"] = _empty(case["combos"], case["bars"])
    elif op == "ohlc":
        s["c"], s["high"], s["low"] = _ohlc_inputs(case, seed)
        n = case["series"]
        s["meta"] = [torch.empty(n, dtype=torch.int32, device="cuda") for _ in range(3)]
        s["out"] = [_empty(case["rows"], n) for _ in range(3)]
        torch.cuda.synchronize()
        _ok(s["lib"].vta_many_series_prepare(h.ctx.handle, _ptr(s["c"]), _ptr(s["high"]),
                                             _ptr(s["low"]), n, case["rows"], 3,
                                             *map(_ptr, s["meta"])))
    elif op == "panel":
        s["x"] = _panel_input(case, seed)
        n = case["series"]
        s["meta"] = [torch.empty(n, dtype=torch.int32, device="cuda") for _ in range(2)]
        s["out"] = [_empty(case["rows"], n) for _ in range(5)]
        torch.cuda.synchronize()
        _ok(s["lib"].vta_many_series_prepare(h.ctx.handle, _ptr(s["x"]), None, None, n,
                                             case["rows"], 4, _ptr(s["meta"][0]), None,
                                             _ptr(s["meta"][1])))
        s["bb"] = vta.CudaBollingerBands.__new__(vta.CudaBollingerBands)
        s["bb"].ctx = h.ctx
        s["bufs"] = [_Buf(t) for t in [s["x"]] + s["meta"] + s["out"][:3]]
    else:
        x = _series(case, seed)[0].cpu().numpy()
        one = dict(offset=(0.85, 0.85, 0.0), sigma=(6.0, 6.0, 0.0))
        s["plan"] = vta.DoubleAlmaPlan(
            h.ctx, x,
            vta.AlmaBatchRange(period=(case["fast"], case["fast"] + case["nfast"] - 1, 1), **one),
            vta.AlmaBatchRange(period=(case["slow"], case["slow"] + case["nslow"] - 1, 1), **one))
    torch.cuda.synchronize()
    return s


def run(s):
    """One pass: enqueue the call; the crossover also reads its statistics,
    which are the whole result of a backtest."""
    op, case, lib, ctx = s["op"], s["case"], s["lib"], s["ctx"]
    if op == "alma":
        s["plan"].launch(s["x"].data_ptr(), 0, s["out"].data_ptr())
    elif op == "ema":
        x, p, out = s["bufs"]
        s["ema"].ema_batch_device(x, p, None, case["bars"], 0, case["combos"], out)
    elif op == "rsi":
        _ok(lib.vta_rsi_batch_device(ctx.handle, _ptr(s["x"]), _ptr(s["periods"]),
                                     case["first"] + case["combos"] - 1, case["bars"], 0,
                                     case["combos"], _ptr(s["out"])))
    elif op == "adx":
        _ok(lib.vta_adx_batch_device(ctx.handle, _ptr(s["high"]), _ptr(s["low"]), _ptr(s["x"]),
                                     _ptr(s["periods"]), case["first"] + case["combos"] - 1,
                                     case["bars"], 0, case["combos"], _ptr(s["out"])))
    elif op == "pack":
        s["pack"].launch()
    elif op == "bb":
        n = case["periods"] * case["widths"]
        _ok(lib.vta_bollinger_bands_batch_device(
            ctx.handle, _ptr(s["x"]), case["bars"], 0, case["bars"], _ptr(s["periods"]),
            _ptr(s["up"]), _ptr(s["dn"]), n, case["first"] + case["periods"] - 1,
            *map(_ptr, s["out"])))
    elif op == "fir":
        last = case["first"] + case["combos"] - 1
        if case["kind"] == "swma":
            _ok(lib.vta_swma_batch_device(ctx.handle, _ptr(s["x"]), _ptr(s["periods"]),
                                          _ptr(s["warms"]), case["bars"], case["combos"], last,
                                          _ptr(s["out"])))
        else:
            fn = lib.vta_sma_batch_device if case["kind"] == "sma" else lib.vta_wma_batch_device
            _ok(fn(ctx.handle, _ptr(s["x"]), _ptr(s["periods"]), case["bars"], case["combos"], 0,
                   last, _ptr(s["out"])))
    elif op == "ohlc":
        _ok(lib.vta_ema_rsi_atr_many_series_device(
            ctx.handle, _ptr(s["c"]), _ptr(s["high"]), _ptr(s["low"]), case["series"],
            case["rows"], case["ema"], case["rsi"], case["atr"], *map(_ptr, s["meta"]),
            *map(_ptr, s["out"])))
    elif op == "panel":
        s["bb"].bollinger_bands_many_series_one_param_device(
            *s["bufs"][:3], case["series"], case["rows"], case["band"], 2.0, 2.0, *s["bufs"][3:])
        _ok(lib.vta_pnr_many_series_one_param_device(
            ctx.handle, _ptr(s["x"]), _ptr(s["meta"][0]), case["series"], case["rows"],
            case["rank"], case["percent"], _ptr(s["out"][3])))
        _ok(lib.vta_medium_ad_many_series_one_param_device(
            ctx.handle, _ptr(s["x"]), _ptr(s["meta"][0]), case["series"], case["rows"],
            case["mad"], _ptr(s["out"][4])))
    else:
        s["plan"].launch()
        stats, pnl = s["plan"].results()
        return {"stats": stats, "pnl": pnl}
    return s["out"]


def work(case):
    """Inputs read once, outputs written once; operations of the definition
    (a multiply-add per tap or state, a compare per window element moved)."""
    op = case["op"]
    if op == "alma":
        ps, t = [p for p, _, _ in _alma_params(case)], case["bars"]
        return {"bytes": 4 * (t + len(ps) * t + sum(ps)),
                "flops": 2 * sum(p * (t - p + 1) for p in ps)}
    if op in ("ema", "rsi", "adx", "fir"):
        n = case["combos"] * case["bars"]
        return {"bytes": 4 * (n + (3 if op == "adx" else 1) * case["bars"] + case["combos"]),
                "flops": {"ema": 3, "rsi": 9, "adx": 14, "fir": 4}[op] * n}
    if op == "pack":
        each = {"ema": 3, "rsi": 9, "adx": 14}[case["kind"]]
        nin = 3 if case["kind"] == "adx" else 1
        n = sum(t * len(p) for t, p in _jobs(case))
        return {"bytes": 4 * (n + sum(nin * t + len(p) for t, p in _jobs(case))),
                "flops": each * n}
    if op == "bb":
        n = case["periods"] * case["widths"] * case["bars"]
        return {"bytes": 4 * (3 * n + case["bars"]) + 20 * case["periods"] * case["widths"],
                "flops": 8 * n + 8 * case["periods"] * case["bars"]}
    if op == "ohlc":
        n, valid = case["series"] * case["rows"], sum(_lengths(case))
        return {"bytes": 12 * (n + valid), "flops": 20 * valid}
    if op == "panel":
        n = case["series"] * case["rows"]
        # every window indicator reads the panel; log2(w) compares per bar replace an element
        ops = 16 + 2 * math.log2(case["rank"] + 1) + 4 * math.log2(case["mad"] + 1)
        return {"bytes": 4 * n * (3 + 5), "flops": int(ops * n)}
    pairs, t = case["nfast"] * case["nslow"], case["bars"]
    lo, hi = case["fast"], case["slow"] + case["nslow"] - 1
    rows = set(range(lo, lo + case["nfast"])) | set(range(case["slow"], hi + 1))
    return {"bytes": 4 * t + 40 * pairs, "flops": 2 * t * (sum(rows) + pairs)}


# Relative 2-norm errors measured against 64 bits, times about four: ALMA up to
# 1.3e-7 (its largest element errors are the split products', 3e-6), RSI and
# ADX (a ratio formed in f32) 5.5e-8, f64 sums rounded to f32 2.5e-8.  The
# crossover's statistics are whole numbers and exactly summed differences.
def tolerance(case):
    op = case["op"]
    if op == "alma":
        return {"rel": 5e-7, "max": 1e-5}
    if op in ("rsi", "adx", "pack", "ohlc"):
        return {"rel": 2.2e-7, "max": 1.6e-6}
    if op == "cross":
        return {"rel": 1e-12, "max": 1e-11, "differ": 0.0}
    return {"rel": 1e-7, "max": 5e-7}


# ------------------------------------------------------------------ 64-bit results

NAN = float("nan")


def _windowed(x, weights, periods):
    """[C, T]: dot of the last p bars with each row of weights [C, W]
    (right-aligned, oldest bar first); NaN before bar p - 1."""
    w, n = weights.shape[1], x.numel()
    xp = torch.cat([torch.zeros(w - 1, dtype=torch.float64, device=x.device), x.double()])
    out = torch.empty(weights.shape[0], n, dtype=torch.float64, device=x.device)
    wt = weights.T.contiguous()
    for a in range(0, n, 16384):
        b = min(n, a + 16384)
        out[:, a:b] = (xp[a:b + w - 1].unfold(0, w, 1).contiguous() @ wt).T
    t = torch.arange(n, device=x.device)
    return out.masked_fill_(t[None, :] < periods[:, None] - 1, NAN)


def _right(rows):
    """Weight lists of uneven length as one right-aligned matrix on the GPU."""
    w = np.zeros((len(rows), max(len(r) for r in rows)))
    for i, r in enumerate(rows):
        w[i, w.shape[1] - len(r):] = r
    return torch.from_numpy(w).cuda()


def _alma_rows(x, params):
    rows = []
    for p, offset, sigma in params:
        d = np.arange(p) - offset * (p - 1)
        w = np.exp(-(d * d) / (2.0 * (p / sigma) ** 2))
        rows.append(w / w.sum())
    return _windowed(x, _right(rows), torch.tensor([len(r) for r in rows], device="cuda"))


def _fir_rows(kind, p):
    if kind == "sma":
        w = np.ones(p)
    elif kind == "wma":
        w = np.arange(1.0, p + 1)
    else:
        a = (p + 1) // 2 if p % 2 else p // 2
        w = np.convolve(np.ones(a), np.ones(p + 1 - a))
    return w / w.sum()


def _smooth(f, beta, at, seed):
    """y of [N, T] with y[at] = seed and y[t] = beta y[t-1] + f[t] after; the
    bars before `at` are NaN.  Blocks of 512 bars side by side, then their carries."""
    n, t = f.shape
    pos = torch.arange(t, device=f.device)[None, :]
    y = f.masked_fill(pos < at[:, None], 0.0)
    ok = at < t
    y[ok, at[ok]] = seed[ok]
    blocks = -(-t // 512)
    y = torch.nn.functional.pad(y, (0, blocks * 512 - t)).view(n, blocks, 512)
    b = beta[:, None]
    for i in range(1, 512):
        y[:, :, i] += b * y[:, :, i - 1]
    decay = beta[:, None] ** torch.arange(1, 513, dtype=torch.float64, device=f.device)
    for k in range(1, blocks):
        y[:, k] += decay * y[:, k - 1, -1:]
    return y.view(n, -1)[:, :t].masked_fill(pos < at[:, None], NAN)


def _at(a, idx):
    return a.gather(1, idx.clamp(0, a.shape[1] - 1)[:, None])[:, 0]


def _ema(x, first, p):
    """Rows x [N, T] (zero before `first`): running mean of p bars, then smoothing."""
    pos = torch.arange(x.shape[1], device=x.device)[None, :]
    count = (pos - first[:, None] + 1).double()
    mean = x.cumsum(1) / count
    alpha = 2.0 / (p.double() + 1.0)
    at = first + p - 1
    y = _smooth(alpha[:, None] * x, 1.0 - alpha, at, _at(mean, at))
    return torch.where(pos < at[:, None], mean, y).masked_fill_(pos < first[:, None], NAN)


def _wilder(f, first, p):
    """Mean of p terms ending at first + p - 1, then Wilder smoothing; f is zero before `first`."""
    at = first + p - 1
    seed = _at(f.cumsum(1), at) / p
    return _smooth(f / p[:, None], 1.0 - 1.0 / p.double(), at, seed)


def _rsi(x, first, p):
    pos = torch.arange(x.shape[1], device=x.device)[None, :]
    d = torch.diff(x, dim=1, prepend=x[:, :1]).masked_fill(pos <= first[:, None], 0.0)
    g = _wilder(d.clamp(min=0), first + 1, p)
    lo = _wilder((-d).clamp(min=0), first + 1, p)
    return torch.where(g + lo == 0, 50.0, 100.0 * g / (g + lo))


def _true_range(h, lo, c):
    pc = torch.cat([c[:, :1], c[:, :-1]], 1)
    return torch.maximum(torch.maximum(h - lo, (h - pc).abs()), (lo - pc).abs())


def _adx(h, lo, c, p):
    """Rows [1, T] of one series, all p; sums from bar 1, DX from bar p, ADX from 2p - 1."""
    up = torch.diff(h, dim=1, prepend=h[:, :1])
    dn = -torch.diff(lo, dim=1, prepend=lo[:, :1])
    pdm = torch.where((up > dn) & (up > 0), up, 0.0)
    mdm = torch.where((dn > up) & (dn > 0), dn, 0.0)
    omr, n, t = 1.0 - 1.0 / p.double(), p.shape[0], h.shape[1]
    pos = torch.arange(t, device=h.device)[None, :]
    plus = _smooth(pdm.expand(n, -1), omr, p, _at(pdm.cumsum(1).expand(n, -1), p))
    minus = _smooth(mdm.expand(n, -1), omr, p, _at(mdm.cumsum(1).expand(n, -1), p))
    dx = torch.where(plus + minus == 0, 0.0, 100.0 * (plus - minus).abs() / (plus + minus))
    del plus, minus
    dx.masked_fill_(pos < p[:, None], 0.0)
    at = 2 * p - 1
    return _smooth(dx / p[:, None], omr, at, _at(dx.cumsum(1), at) / p)


def _recurrence(kind, close, high, low, periods):
    p, zero = periods.long(), torch.zeros_like(periods, dtype=torch.long)
    c, h, lo = (a.double()[None, :] for a in (close, high, low))
    if kind == "ema":
        return _ema(c.expand(len(p), -1), zero, p)
    return _rsi(c, zero, p) if kind == "rsi" else _adx(h, lo, c, p)


def _sliding(x, w):
    """(first row, windows [rows, series, w]) pieces of a panel."""
    for a in range(w - 1, x.shape[0], 512):
        b = min(x.shape[0], a + 512)
        yield a, b, x[a - w + 1:b].unfold(0, w, 1)


def _panel(case, x):
    out = [torch.full(x.shape, NAN, dtype=torch.float64, device="cuda") for _ in range(5)]
    for a, b, w in _sliding(x, case["band"]):
        w = w.double()
        m = w.mean(2)
        sd = (w - m[:, :, None]).square().mean(2).sqrt()
        out[0][a:b], out[1][a:b], out[2][a:b] = m + 2 * sd, m, m - 2 * sd
    k = max(0, min(case["rank"], math.floor(case["percent"] * 0.01 * case["rank"] + 0.5)) - 1)
    for a, b, w in _sliding(x, case["rank"]):
        out[3][a:b] = w.sort(2)[0][:, :, k].double()
    n = case["mad"]
    mid = lambda s: s[:, :, n // 2] if n % 2 else 0.5 * (s[:, :, n // 2 - 1] + s[:, :, n // 2])
    for a, b, w in _sliding(x, n):
        m = mid(w.sort(2)[0].double())
        out[4][a:b] = mid((w.double() - m[:, :, None]).abs().sort(2)[0])
    return out


def _cross(case, seed):
    x = _series(case, seed)[0]
    lo, hi = case["fast"], case["slow"] + case["nslow"] - 1
    rows = _alma_rows(x, [(p, 0.85, 6.0) for p in range(lo, hi + 1)])
    slow = rows[case["slow"] - lo:]
    sp = torch.arange(case["slow"], hi + 1, device="cuda")
    move = torch.diff(x.double(), append=x[-1:].double())
    pos = torch.arange(x.numel(), device="cuda")[None, :]
    pnl = []
    for p in range(lo, lo + case["nfast"]):
        d = torch.sign(rows[p - lo][None, :] - slow)
        d.masked_fill_(pos < sp.clamp(min=p)[:, None] - 1, 0.0)
        d[sp == p] = 0.0
        pnl.append(d @ move)
    return {"stats": None, "pnl": torch.cat(pnl)}


def exact(case, seed):
    op = case["op"]
    if op == "alma":
        return _alma_rows(_series(case, seed)[0], _alma_params(case))
    if op in ("ema", "rsi", "adx"):
        return _recurrence(op, *_series(case, seed), _periods(case))
    if op == "pack":
        walks = _walk(case["longest"], case["jobs"], 0.01, seed).T.contiguous()
        out = []
        for k, (n, periods) in enumerate(_jobs(case)):
            c = walks[k, :n].clone()
            out.append(_recurrence(case["kind"], c, *_high_low(c, seed + k),
                                   torch.tensor(periods, device="cuda")))
        return out
    if op == "bb":
        x, f, n = _series(case, seed)[0], case["first"], case["periods"]
        p = torch.arange(f, f + n, device="cuda")
        box = _right([np.full(q, 1.0 / q) for q in range(f, f + n)])
        # squares about the level of each 4,096-bar stretch, so that little cancels
        m, sd = _windowed(x, box, p), torch.empty(n, x.numel(), dtype=torch.float64, device="cuda")
        halo = box.shape[1] - 1
        for a in range(0, x.numel(), 4096):
            lo, b = max(0, a - halo), min(x.numel(), a + 4096)
            y = x[lo:b].double() - x[a].double()
            my, sq = _windowed(y, box, p), _windowed(y * y, box, p)
            sd[:, a:b] = (sq - my * my).clamp(min=0).sqrt()[:, a - lo:]
        w = case["widths"]
        up = (1.0 + 0.5 * torch.arange(w, device="cuda", dtype=torch.float64)).repeat(n)
        m, sd = m.repeat_interleave(w, 0), sd.repeat_interleave(w, 0)
        return [m + up[:, None] * sd, m, m - 2.0 * sd]
    if op == "fir":
        ps = range(case["first"], case["first"] + case["combos"])
        return _windowed(_series(case, seed)[0], _right([_fir_rows(case["kind"], p) for p in ps]),
                         torch.tensor(list(ps), device="cuda"))
    if op == "ohlc":
        c, h, lo = (a.T.double().contiguous().nan_to_num_(0.0) for a in _ohlc_inputs(case, seed))
        first = _starts(case)
        full = lambda v: torch.full_like(first, v)
        tr = _true_range(h, lo, c)
        tr.scatter_(1, first[:, None], (h - lo).gather(1, first[:, None]))
        del h, lo
        atr = _wilder(tr, first, full(case["atr"])).T
        del tr
        ema = _ema(c, first, full(case["ema"])).T
        return [ema, _rsi(c, first, full(case["rsi"])).T, atr]
    if op == "panel":
        return _panel(case, _panel_input(case, seed))
    return _cross(case, seed)
