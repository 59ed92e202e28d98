"""SMA / WMA / SWMA / SMMA / Wilders parity on the GPU (batch, enqueue-only
batch, many-series, many-series enqueue-only).

Bar: NaN warm-up prefixes and the non-finite rules bit-exact (NaN masks and
infinities equal); values within 1e-5 relative of the f64 oracle on the same
f32 inputs.  The reference's own GPU tests (tests/{sma,wma,swma,smma,wilders}
_cuda.rs) are also replayed with their data, sweeps and tolerances (absolute,
against the CPU on the unrounded f64 data).
"""
import ctypes

import numpy as np
import pytest

import oracle as O
import vectorta_amd as vta
from vectorta_amd import datagen
from vectorta_amd._lib import check
from tests.conftest import require_gpu
from tests.helpers import max_rel_err, nan_mask_equal

pytestmark = pytest.mark.gpu

NAMES = ("sma", "wma", "swma", "smma", "wilders")


@pytest.fixture(scope="module")
def ops():
    require_gpu()
    return {"sma": vta.CudaSma(0), "wma": vta.CudaWma(0), "swma": vta.CudaSwma(0),
            "smma": vta.CudaSmma(0), "wilders": vta.CudaWilders(0)}


def _check(g, ref, what, bound=1e-5):
    nan_mask_equal(g, ref)
    r = np.asarray(ref, dtype=np.float64)
    inf = np.isinf(r)
    assert (np.asarray(g, dtype=np.float64)[inf] == r[inf]).all(), f"{what}: infinities differ"
    err = max_rel_err(g, ref)
    print(f"{what}: max rel err {err:.3e}")
    assert err <= bound, (what, err)


def _batch_oracle(name, x, periods):
    """The reference's batch rows: prefix-sum rows for SMA; the running-sum
    kernels for the others (the WMA prefix row loses ~eps*len^2/p^2 on long
    series, so long WMA series are checked against the running sums)."""
    xd = x.astype(np.float64)
    f = {"sma": O.sma_batch_row, "wma": O.wma, "swma": O.swma, "smma": O.smma,
         "wilders": O.wilders}[name]
    return np.stack([f(xd, p) for p in periods])


def _batch(ops, name, x, period):
    return getattr(ops[name], f"{name}_batch_dev")(x, period).to_host()


@pytest.mark.parametrize("name,period", [("sma", (1, 64, 9)), ("wma", (2, 64, 9)),
                                         ("swma", (1, 64, 9)), ("smma", (1, 64, 9)),
                                         ("wilders", (1, 64, 9))])
def test_batch_small(ops, name, period):
    x = datagen.gbm_close(5_000, 0.01, seed=201)
    x[:9] = np.nan
    ps = ops[name].expand_grid(period)
    _check(_batch(ops, name, x, period), _batch_oracle(name, x, ps), f"{name} batch")
    if name == "wma":   # small series: the reference's batch prefix rows too
        _check(_batch(ops, name, x, period),
               np.stack([O.wma_batch_row(x.astype(np.float64), p) for p in ps]), "wma prefix")


@pytest.mark.parametrize("name", NAMES)
def test_batch_long_series_many_tiles(ops, name):
    """300k bars, periods up to 900: many 1024-bar tiles, several combo groups,
    the recurrences' chunked burn-in."""
    x = datagen.gbm_close(300_000, 0.01, seed=202)
    x[:3] = np.nan
    period = (2, 900, 47)
    ps = ops[name].expand_grid(period)
    assert len(ps) > 16
    _check(_batch(ops, name, x, period), _batch_oracle(name, x, ps), f"{name} long batch")


@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf])
def test_batch_nonfinite_rules(ops, bad):
    """A non-finite bar after first_valid: window sums then NaN (SMA), NaN
    from the bar on (WMA batch), [z, z+a) running sums then NaN (SWMA), the
    recurrences' sequential values; the p <= 2 SWMA forms stay window-only."""
    x = datagen.gbm_close(6_000, 0.01, seed=203)
    x[:5] = np.nan
    x[3_000] = bad
    xd = x.astype(np.float64)
    for name, period in (("sma", (1, 40, 13)), ("swma", (1, 40, 13)), ("smma", (1, 40, 13)),
                         ("wilders", (1, 40, 13))):
        ps = ops[name].expand_grid(period)
        _check(_batch(ops, name, x, period), _batch_oracle(name, x, ps), f"{name} {bad}")
    ps = ops["wma"].expand_grid((2, 40, 13))
    ref = np.stack([O.wma_batch_row(xd, p) for p in ps])
    ref[:, 3_000:] = np.nan        # the batch prefix rows: NaN from the bar on
    _check(_batch(ops, "wma", x, (2, 40, 13)), ref, f"wma {bad}")


@pytest.mark.parametrize("name", NAMES)
def test_many_series(ops, name):
    rng = np.random.default_rng(204)
    rows, cols = 6_000, 70
    tm = (100 + np.cumsum(rng.normal(0, 1, (rows, cols)), axis=0)).astype(np.float32)
    lead = rng.integers(0, 400, size=cols)
    for s in range(cols):
        tm[:lead[s], s] = np.nan
    if name != "wilders":
        tm[2_500, 5] = np.nan
        tm[4_000, 6] = np.inf
    # SWMA: periods up to 80 take the LDS ring of recent bars, 120 the cache
    for p in ((2, 9, 33, 120) if name == "wma" else (1, 2, 9, 33, 120)):
        g = getattr(ops[name], {"sma": "sma_multi_series_one_param_time_major_dev",
                                "wma": "wma_multi_series_one_param_time_major_dev",
                                "swma": "swma_multi_series_one_param_time_major_dev",
                                "smma": "smma_multi_series_one_param_time_major_dev",
                                "wilders": "wilders_many_series_one_param_time_major_dev"}[name])(
            tm, cols, rows, p).to_host()
        ref, st = O.ma_many(name, tm.astype(np.float64), p)
        assert (st == 0).all()
        _check(g, ref, f"{name} many-series p={p}")


@pytest.mark.parametrize("n,longest", [(1_025, 255), (3_001, 1_023), (9_000, 1_700),
                                       (70_001, 90)])
def test_device_batch_prefix_runs_and_replays(ops, n, longest):
    """A thread's run of staged bars from one to past the eight it keeps in
    registers, one to all of the 64 searchers for the first non-finite bar, and
    a captured call replayed over other data in the same buffer: a bar that is
    not finite, none, and one elsewhere, each against the oracle."""
    lead = 3
    for name, p0 in (("sma", 1), ("wma", 2), ("swma", 1)):
        op = ops[name]
        ps = np.unique(np.linspace(p0, longest, 9).astype(np.int32))
        base = datagen.gbm_close(n, 0.01, seed=n)
        base[:lead] = np.nan
        d_x, d_p = op.ctx.to_device(base), op.ctx.to_device(ps)
        d_w = op.ctx.to_device((lead + ps - 1).astype(np.int32))
        d_o = op.ctx.alloc(ps.size * n * 4)

        def call():
            if name == "swma":
                op.swma_batch_device(d_x, d_p, d_w, n, ps.size, int(ps.max()), d_o)
            else:
                getattr(op, f"{name}_batch_device")(d_x, d_p, n, ps.size, lead, int(ps.max()), d_o)
        call()
        op.synchronize()
        op.ctx.begin_capture()
        call()
        graph = op.ctx.end_capture()
        for bad in (None, n - 1, None, n // 2, lead + 1):
            x = base.copy()
            if bad is not None:
                x[bad] = np.nan
            check(vta.lib().vta_memcpy_htod(op.ctx.handle, ctypes.c_void_p(d_x.ptr),
                                            x.ctypes.data_as(ctypes.c_void_p), x.nbytes))
            graph.launch()
            op.synchronize()
            got = d_o.copy_to_host(np.float32).reshape(ps.size, n)
            _check(got, _batch_oracle(name, x, ps), f"{name} n={n} bad={bad}")
        graph.destroy()
        for b in (d_x, d_p, d_w, d_o):
            b.free()


def test_device_entry_points(ops):
    """Enqueue-only forms on device-resident inputs, with the reference
    wrappers' argument lists, equal the host-input forms."""
    x = datagen.gbm_close(20_000, 0.01, seed=205)
    x[:4] = np.nan
    x[12_000] = np.nan
    ctx = ops["sma"].ctx
    for name, period in (("sma", (3, 50, 7)), ("wma", (2, 50, 7)), ("swma", (1, 50, 7))):
        op = ops[name]
        ps = np.asarray(op.expand_grid(period), dtype=np.int32)
        host = getattr(op, f"{name}_batch_dev")(x, period).to_host()
        d_x = op.ctx.to_device(x)
        d_p = op.ctx.to_device(ps)
        d_o = op.ctx.alloc(ps.size * x.size * 4)
        if name == "swma":
            # swma_wrapper.rs:663: warm indices first_valid + p - 1, no first_valid
            d_w = op.ctx.to_device((4 + ps - 1).astype(np.int32))
            op.swma_batch_device(d_x, d_p, d_w, x.size, ps.size, int(ps.max()), d_o)
        else:
            getattr(op, f"{name}_batch_device")(d_x, d_p, x.size, ps.size, 4, int(ps.max()), d_o)
        op.synchronize()
        dev = d_o.copy_to_host(np.float32).reshape(ps.size, x.size)
        assert np.array_equal(host.view(np.uint32), dev.view(np.uint32)), name
    y = x.copy()
    y[12_000] = 1.0
    for name, period in (("smma", (1, 50, 7)), ("wilders", (1, 50, 7))):
        op = ops[name]
        ps = np.asarray(op.expand_grid(period), dtype=np.int32)
        host = getattr(op, f"{name}_batch_dev")(y, period).to_host()
        d_x = op.ctx.to_device(y)
        d_p = op.ctx.to_device(ps)
        d_w = op.ctx.to_device((4 + ps - 1).astype(np.int32))
        d_o = op.ctx.alloc(ps.size * y.size * 4)
        if name == "smma":
            op.smma_batch_device(d_x, d_p, d_w, 4, y.size, ps.size, d_o)
        else:
            op.wilders_batch_device(d_x, d_p, None, d_w, y.size, 4, ps.size, d_o)
        op.synchronize()
        dev = d_o.copy_to_host(np.float32).reshape(ps.size, y.size)
        assert np.array_equal(host.view(np.uint32), dev.view(np.uint32)), name
        if name == "wilders":
            # the reference host code's f32 alphas 1/p: within the bound of the oracle
            d_a = op.ctx.to_device((1.0 / ps.astype(np.float32)).astype(np.float32))
            op.wilders_batch_device(d_x, d_p, d_a, d_w, y.size, 4, ps.size, d_o)
            op.synchronize()
            dev = d_o.copy_to_host(np.float32).reshape(ps.size, y.size)
            _check(dev, np.stack([O.wilders(y.astype(np.float64), int(p)) for p in ps]),
                   "wilders f32 alphas")
    # many-series device forms (first non-finite bar found on the device)
    rng = np.random.default_rng(206)
    rows, cols = 3_000, 40
    tm = (50 + np.cumsum(rng.normal(0, 1, (rows, cols)), axis=0)).astype(np.float32)
    tm[:17, 3] = np.nan
    tm[1_000, 4] = np.nan
    d_tm = ctx.to_device(tm)
    fv = np.argmax(~np.isnan(tm), axis=0).astype(np.int32)
    d_fv = ctx.to_device(fv)
    for name in ("sma", "wma", "swma"):
        op = ops[name]
        host = getattr(op, f"{name}_multi_series_one_param_time_major_dev")(
            tm, cols, rows, 12).to_host()
        d_o = ctx.alloc(rows * cols * 4)
        if name == "sma":
            op.sma_many_series_one_param_device(d_tm, d_fv, cols, rows, 12, d_o)
        elif name == "wma":
            op.wma_multi_series_one_param_time_major_device(d_tm, 12, cols, rows, d_fv, d_o)
        else:
            op.swma_multi_series_one_param_device(d_tm, None, 12, cols, rows, d_fv, d_o)
        op.synchronize()
        dev = d_o.copy_to_host(np.float32).reshape(rows, cols)
        assert np.array_equal(host.view(np.uint32), dev.view(np.uint32)), name
    tmc = np.abs(tm) + 1.0                       # SMMA / Wilders: clean, finite series
    tmc[:17, 3] = np.nan
    d_tmc = ctx.to_device(tmc)
    for name in ("smma", "wilders"):
        op = ops[name]
        d_o = ctx.alloc(rows * cols * 4)
        if name == "smma":
            op.smma_multi_series_one_param_device(d_tmc, 12, cols, rows, d_fv, d_o)
        else:
            op.wilders_many_series_one_param_device(d_tmc, d_fv, 12, np.float32(1.0 / 12.0),
                                                    cols, rows, d_o)
        op.synchronize()
        dev = d_o.copy_to_host(np.float32).reshape(rows, cols)
        ref = O.ma_many(name, tmc.astype(np.float64), 12)[0]
        _check(dev, ref, f"{name} many-series device")
    # SMA's device-input forms that allocate their output (sma_wrapper.rs:830, 982)
    op = ops["sma"]
    ps = [3, 10, 44]
    got = op.sma_batch_dev_from_device(ctx.to_device(x), x.size, ps, 4).to_host()
    host = op.sma_batch_dev(x, (3, 44, 41)).to_host()
    assert np.array_equal(got[[0, 2]].view(np.uint32), host.view(np.uint32))
    _check(got, np.stack([O.sma_batch_row(x.astype(np.float64), p) for p in ps]), "sma")
    got = op.sma_multi_series_one_param_time_major_dev_from_device(d_tm, d_fv, cols, rows,
                                                                   12).to_host()
    host = op.sma_multi_series_one_param_time_major_dev(tm, cols, rows, 12).to_host()
    assert np.array_equal(got.view(np.uint32), host.view(np.uint32))


def test_warm_index_mismatch_reported_at_synchronize(ops):
    """Warm indices other than first_valid + period - 1 (the reference host
    code's values) are an InvalidInput that the next synchronize reports once;
    consistent ones report nothing."""
    x = datagen.gbm_close(5_000, 0.01, seed=208)
    x[:4] = np.nan
    for name in ("smma", "wilders", "swma"):
        op = ops[name]
        ctx = op.ctx
        ctx.synchronize()
        ps = np.array([5, 9, 14], dtype=np.int32)
        d_x, d_p = ctx.to_device(x), ctx.to_device(ps)
        d_o = ctx.alloc(ps.size * x.size * 4)
        bad = (4 + ps - 1).astype(np.int32)
        bad[1] += 1
        d_bad = ctx.to_device(bad)
        if name == "smma":
            op.smma_batch_device(d_x, d_p, d_bad, 4, x.size, ps.size, d_o)
        elif name == "wilders":
            op.wilders_batch_device(d_x, d_p, None, d_bad, x.size, 4, ps.size, d_o)
        else:
            op.swma_batch_device(d_x, d_p, d_bad, x.size, ps.size, int(ps.max()), d_o)
        with pytest.raises(vta.VtaError) as e:
            op.synchronize()
        assert e.value.kind == "InvalidInput" and "warm index" in str(e.value)
        op.synchronize()                             # reported once, then clear
    # SWMA: a warm index implying a first_valid past the longest period's room
    op = ops["swma"]
    ps = np.array([5, 9], dtype=np.int32)
    far = (x.size - 3 + ps - 1).astype(np.int32)
    d_o = op.ctx.alloc(ps.size * x.size * 4)
    op.swma_batch_device(op.ctx.to_device(x), op.ctx.to_device(ps), op.ctx.to_device(far),
                         x.size, ps.size, 9, d_o)
    with pytest.raises(vta.VtaError):
        op.synchronize()
    assert np.isnan(d_o.copy_to_host(np.float32)).all()


@pytest.mark.parametrize("T", [1, 2_047, 2_048, 2_049, 2_100_001, 5_000_003])
def test_first_non_finite_bar_wherever_it_lies(ops, T):
    """The device form's search (2,048 bars per block, at most 1,024 blocks, which
    then go round) against the host form's own, bit for bit: at the edges of its
    blocks, threads and rounds, before first_valid, and nowhere."""
    op, p = ops["sma"], min(3, T)
    x = datagen.gbm_close(T, 0.001, seed=211)
    fv = 5 if T > 8 else 0
    x[:fv] = np.nan
    d_x, d_p, d_o = op.ctx.to_device(x), op.ctx.to_device(np.int32([p])), op.ctx.alloc(T * 4)
    spots = {None, fv + p, 255, 256, 2_047, 2_048, 2_303, 4_095, 2_097_151, 2_097_152, 2_099_000,
             4_194_304, T - 2, T - 1}
    for bad in [b for b in spots if b is None or fv + p <= b < T]:
        y = x.copy()
        if bad is not None:
            y[bad] = np.inf
            y[-1] = np.nan
        check(vta.lib().vta_memcpy_htod(op.ctx.handle, ctypes.c_void_p(d_x.ptr),
                                    y.ctypes.data_as(ctypes.c_void_p), y.nbytes))
        op.sma_batch_device(d_x, d_p, T, 1, fv, p, d_o)
        op.synchronize()
        want = op.sma_batch_dev(y, (p, p, 0)).to_host()[0]
        assert np.array_equal(d_o.copy_to_host(np.uint32), want.view(np.uint32)), (T, bad)


def test_more_combos_than_sixteen_per_workgroup_reach(ops):
    """1,100,000 combos: more rows of workgroups than the grid's y takes (65,536)
    at the 16 combos per workgroup of a long SMA batch."""
    op, T, C = ops["sma"], 64, 1_100_000
    x = datagen.gbm_close(T, 0.01, seed=210)
    ps = (np.arange(C) % 40 + 1).astype(np.int32)
    d_o = op.ctx.alloc(C * T * 4)
    op.sma_batch_device(op.ctx.to_device(x), op.ctx.to_device(ps), T, C, 0, 40, d_o)
    op.synchronize()
    got = d_o.copy_to_host(np.uint32).reshape(C, T)
    d_o.free()
    want = op.sma_batch_dev(x, (1, 40, 1)).to_host().view(np.uint32)
    assert np.array_equal(got[:C // 40 * 40].reshape(-1, 40, T),
                          np.broadcast_to(want, (C // 40, 40, T)))


def _ref_data(n, lead, fa, fb):
    d = np.full(n, np.nan)
    i = np.arange(lead, n, dtype=np.float64)
    d[lead:] = np.sin(i * fa) + fb * i
    return d


@pytest.mark.parametrize("name,n,lead,fa,fb,period,tol", [
    ("sma", 4096, 5, 0.001, 0.0002, (5, 45, 5), 1e-5),        # tests/sma_cuda.rs:30-80
    ("wma", 4096, 4, 0.002, 0.0002, (4, 128, 2), 1e-5),       # tests/wma_cuda.rs:30-80
    ("swma", 4096, 10, 0.0013, 0.0005, (5, 160, 5), 2e-4),    # tests/swma_cuda.rs:30-75
    ("smma", 4096, 12, 0.0017, 0.0003, (5, 140, 5), 2.5e-4),  # tests/smma_cuda.rs:30-75
    ("wilders", 4096, 4, 0.0015, 0.0002, (5, 48, 3), 1e-5),   # tests/wilders_cuda.rs:30-75
])
def test_reference_gpu_tests_replayed(ops, name, n, lead, fa, fb, period, tol):
    data = _ref_data(n, lead, fa, fb)
    g = _batch(ops, name, data.astype(np.float32), period).astype(np.float64)
    ps = ops[name].expand_grid(period)
    f = {"sma": O.sma_batch_row, "wma": O.wma_batch_row, "swma": O.swma, "smma": O.smma,
         "wilders": O.wilders}[name]
    cpu = np.stack([f(data, p) for p in ps])
    nan_mask_equal(g, cpu)
    m = np.isfinite(cpu)
    assert np.max(np.abs(g[m] - cpu[m])) <= tol


def test_errors(ops):
    x = datagen.gbm_close(100, 0.01, seed=207)
    with pytest.raises(vta.VtaError):
        ops["wma"].wma_batch_dev(x, (1, 5, 1))            # WMA needs period > 1
    with pytest.raises(vta.VtaError):
        ops["sma"].sma_batch_dev(x, (0, 0, 0))
    with pytest.raises(vta.VtaError):
        ops["swma"].swma_batch_dev(x, (101, 101, 0))      # period > len
    y = x.copy()
    y[:60] = np.nan
    with pytest.raises(vta.VtaError):
        ops["smma"].smma_batch_dev(y, (41, 41, 0))        # not enough valid data
    z = x.copy()
    z[5] = np.inf
    with pytest.raises(vta.VtaError):
        ops["wilders"].wilders_batch_dev(z, (3, 8, 1))    # non-finite in the warm window
    with pytest.raises(vta.VtaError):
        ops["sma"].sma_batch_dev(np.full(10, np.nan, np.float32), (2, 2, 0))
