"""GPU parity of the moving-window kernels.

Bars (against the long-double exact oracle; NaN masks must be identical):
  float32 sum/mean/var/std: <= 1 float32 ULP of the exact value;
  float32 cov/corr: <= 2 ULP, or <= 1e-6 of the window's scale;
  float64 mean (the (100, 10000) window-20 config): <= 1e-12 relative;
  float64 sum: <= 1e-12 of sum|x| in the window; var/std/cov/corr: <= 1e-11 relative.
Against the C restatement of the reference the NaN masks are identical and the
GPU error never exceeds the reference's own error (both against the exact oracle).
"""

from __future__ import annotations

import numpy as np
import pytest
from numpy.testing import assert_allclose

from ._data import walk_array

pytestmark = pytest.mark.gpu

FUNCS1 = ["move_mean", "move_sum", "move_std", "move_var"]
FUNCS2 = ["move_cov", "move_corr"]


def ulp_err(got32, exact64):
    """|got - exact| in float32 ULPs of the exact value."""
    e = exact64.astype(np.float32)
    ulp = np.spacing(np.abs(e)).astype(np.float64)
    return np.abs(got32.astype(np.float64) - exact64) / ulp


def check_f32(func, got, want, scale=None):
    assert np.array_equal(np.isnan(got), np.isnan(want)), f"{func}: NaN mask differs"
    ok = ~np.isnan(want)
    if not ok.any():
        return
    err = ulp_err(got[ok], want[ok])
    if func in FUNCS2:
        absok = np.abs(got[ok] - want[ok]) <= 1e-6 * (scale[ok] if scale is not None else 1.0)
        assert np.all((err <= 2) | absok), f"{func}: max {err.max():.2f} ULP"
    else:
        assert err.max() <= 1.0, f"{func}: max {err.max():.3f} ULP"


@pytest.mark.parametrize("func", FUNCS1 + FUNCS2)
@pytest.mark.parametrize(
    "shape,window,min_count",
    [
        ((3, 500), 10, None),
        ((3, 500), 50, 3),
        ((4, 9000), 1000, 500),
        ((2, 20_000), 20, 20),
        ((2, 5000), 1, 0),
        ((1, 30_000), 12_000, 100),  # window longer than the LDS halo limit
        ((5, 4096), 4096, 1),
        ((3, 4097), 4097, 0),
    ],
)
def test_move_f32_against_exact(gpu_lib, func, shape, window, min_count):
    import numbagg_amd as nb
    from oracle import exact

    x = walk_array(*shape, seed=window + shape[1])
    y = walk_array(*shape, seed=window + shape[1] + 1) if func in FUNCS2 else None
    args = (x,) if y is None else (x, y)
    got = getattr(nb, func)(*args, window=window, min_count=min_count)
    assert got.dtype == np.float32 and got.shape == x.shape
    want = exact.move(func, x, window, min_count, y=y)
    check_f32(func, got, want, scale=np.ones_like(want))


@pytest.mark.parametrize("func", FUNCS1 + FUNCS2)
def test_move_f32_against_restated_reference(gpu_lib, func):
    """Same NaN mask as the reference restatement, and no larger error than the
    reference's own (float32-rounded products, running float64 sums), both
    measured against the exact oracle."""
    import numbagg_amd as nb
    from oracle import exact, restated

    x = walk_array(4, 6000, seed=5, offset=0.0)
    y = walk_array(4, 6000, seed=6, offset=0.0) if func in FUNCS2 else None
    args = (x,) if y is None else (x, y)
    got = getattr(nb, func)(*args, window=300, min_count=150)
    ref = restated.move(func, x, 300, 150, y=y)
    ex = exact.move(func, x, 300, 150, y=y)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    ok = ~np.isnan(ex)
    err_gpu = np.abs(got[ok].astype(np.float64) - ex[ok])
    err_ref = np.abs(ref[ok].astype(np.float64) - ex[ok])
    half_ulp = 0.5 * np.spacing(np.abs(ex[ok]).astype(np.float32)).astype(np.float64)
    assert err_gpu.max() <= max(err_ref.max(), half_ulp.max())
    assert np.mean(err_gpu) <= np.mean(err_ref) + np.mean(half_ulp)


@pytest.mark.parametrize("func", FUNCS1 + FUNCS2)
@pytest.mark.parametrize("window,min_count", [(20, 20), (7, 2), (300, 0)])
def test_move_f64_against_exact(gpu_lib, func, window, min_count):
    import numbagg_amd as nb
    from oracle import exact

    rng = np.random.default_rng(window)
    x = rng.standard_normal((20, 10_000))
    x[rng.random(x.shape) < 0.1] = np.nan
    y = rng.standard_normal((20, 10_000)) if func in FUNCS2 else None
    args = (x,) if y is None else (x, y)
    got = getattr(nb, func)(*args, window=window, min_count=min_count)
    want = exact.move(func, x, window, min_count, y=y)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    ok = ~np.isnan(want)
    if func == "move_sum":
        scale = exact.move("move_sum", np.abs(x), window, 0)
        assert np.all(np.abs(got[ok] - want[ok]) <= 1e-12 * scale[ok] + 1e-300)
    elif func == "move_mean":
        assert_allclose(got[ok], want[ok], rtol=1e-12)
    else:
        assert_allclose(got[ok], want[ok], rtol=1e-11, atol=1e-13)


def test_move_mean_f64_config1(gpu_lib):
    """(100, 10000) float64, window=20, min_count=20, 10% NaN: within 1e-12
    relative of the exact window mean."""
    import numbagg_amd as nb
    from oracle import exact

    rng = np.random.default_rng(20240601)
    x = rng.standard_normal((100, 10_000))
    x[rng.random(x.shape) < 0.10] = np.nan
    got = nb.move_mean(x, window=20, min_count=20)
    want = exact.move("move_mean", x, 20, 20)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    ok = ~np.isnan(want)
    assert np.max(np.abs(got[ok] - want[ok]) / np.abs(want[ok])) <= 1e-12


@pytest.mark.parametrize("func", FUNCS1 + FUNCS2)
@pytest.mark.parametrize("window", [10, 50])
@pytest.mark.parametrize("min_count", [None, 0, 1, 3, "window"])
def test_move_reference_pandas_vectors(gpu_lib, golden, func, window, min_count):
    import numbagg_amd as nb

    a, a2 = golden["array_3x500"], golden["array2_3x500"]
    mc = window if min_count == "window" else min_count
    want = golden[f"move_{func[5:]}_w{window}_mc{'None' if min_count is None else mc}"]
    args = (a, a2) if func in FUNCS2 else (a,)
    assert_allclose(getattr(nb, func)(*args, window=window, min_count=mc), want)


def test_move_known_answers(gpu_lib):
    import numbagg_amd as nb

    rs = np.random.RandomState(0)
    arr = (rs.random(1000) * 1e13).astype(np.float32)
    assert_allclose(nb.move_mean(arr, window=1), arr)
    arr = np.tile((rs.rand(10) * 1e13).astype(np.float32), 100)
    assert nb.move_sum(arr, window=10)[-1] == np.sum(arr[:10])


def test_move_axes_and_layouts(gpu_lib):
    import torch

    import numbagg_amd as nb
    from oracle import exact

    rng = np.random.default_rng(9)
    x = rng.standard_normal((5, 6, 700)).astype(np.float32)
    x[rng.random(x.shape) < 0.2] = np.nan
    for axis in (0, 1, 2, -1, -2):
        got = nb.move_mean(x, window=3, min_count=1, axis=axis)
        xm = np.moveaxis(x, axis, -1)
        want = exact.move("move_mean", xm.reshape(-1, xm.shape[-1]), 3, 1).reshape(xm.shape)
        want = np.moveaxis(want, -1, axis)
        assert np.array_equal(np.isnan(got), np.isnan(want))
        assert_allclose(got, want, rtol=1e-6, atol=1e-7)
    # device tensors stay on the device; an unaligned row start takes the scalar path
    t = torch.from_numpy(x).cuda()[:, :, 3:]
    got = nb.move_sum(t, window=5)
    assert got.is_cuda
    want = exact.move("move_sum", x[:, :, 3:].reshape(-1, 697), 5).reshape(5, 6, 697)
    assert_allclose(got.cpu().numpy(), want, rtol=1e-6)
    # broadcasting of the two inputs of move_corr
    a = x[0]
    b = rng.standard_normal(700).astype(np.float32)
    got = nb.move_corr(a, b, window=40)
    want = exact.move("move_corr", a, 40, None, y=np.broadcast_to(b, a.shape))
    assert_allclose(got, want, rtol=1e-5, atol=1e-6)
    # integer input runs on the float64 loop (numpy's safe-cast loop choice)
    i = rng.integers(-50, 50, size=(3, 100)).astype(np.int32)
    got = nb.move_mean(i, window=4)
    assert got.dtype == np.float64
    assert_allclose(got, exact.move("move_mean", i.astype(np.float64), 4), rtol=1e-14)
    assert nb.move_mean(i.astype(np.int16), window=4).dtype == np.float32



@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("func", FUNCS1 + FUNCS2)
@pytest.mark.parametrize("window", [1, 37, 1000, 2047, 2048, 4081, 4096, 6000])
def test_move_span_carried_halo_is_bitwise_neutral(gpu_lib, monkeypatch, func, dtype, window):
    """A workgroup walking a span of tiles carries each halo forward in LDS
    (and optionally prefetches the next tile into registers); outputs must be
    bitwise identical to one tile per workgroup (every tile evaluates its
    window from the same staged inputs)."""
    import numbagg_amd as nb

    x = walk_array(3, 5 * 4096 + 123, seed=window, dtype=dtype)
    y = walk_array(3, 5 * 4096 + 123, seed=window + 1, dtype=dtype) if func in FUNCS2 else None
    args = (x,) if y is None else (x, y)
    outs = []
    for span, prefetch in (("1", "0"), ("2", "0"), ("4", "1"), ("16", "0"), ("16", "1")):
        monkeypatch.setenv("NBG_MOVE_SPAN", span)
        monkeypatch.setenv("NBG_MOVE_PREFETCH", prefetch)
        outs.append(getattr(nb, func)(*args, window=window, min_count=1))
    for o in outs[1:]:
        np.testing.assert_array_equal(o.view(np.uint8), outs[0].view(np.uint8))


@pytest.mark.parametrize("func", ["move_sum", "move_mean"])
@pytest.mark.parametrize("shape,window,min_count", [((3, 500), 10, None), ((4, 9000), 1000, 500), ((2, 20_000), 20, 20),
                                                    ((1, 30_000), 12_000, 100)])
def test_move_f32_twosum_accumulator(gpu_lib, monkeypatch, func, shape, window, min_count):
    """The FP32 TwoSum accumulator (NBG_F32_ACCUMULATOR=twosum) meets the same
    bar as the float64 default: <= 1 float32 ULP of the exact value."""
    import numbagg_amd as nb
    from oracle import exact

    monkeypatch.setenv("NBG_F32_ACCUMULATOR", "twosum")
    x = walk_array(*shape, seed=window + shape[1] + 5)
    got = getattr(nb, func)(x, window=window, min_count=min_count)
    check_f32(func, got, exact.move(func, x, window, min_count))


def test_out_argument(gpu_lib):
    """out= is filled and returned (numbagg/decorators.py:341, :414, :487)."""
    import numbagg_amd as nb

    rng = np.random.default_rng(0)
    x = rng.standard_normal((3, 200))
    want = nb.move_mean(x, window=5)
    dest = np.empty_like(x)
    assert nb.move_mean(x, window=5, out=dest) is dest
    np.testing.assert_array_equal(dest, want)
    d32 = np.empty(x.shape, dtype=np.float32)
    assert nb.move_exp_nanmean(x, alpha=0.3, out=d32) is d32
    np.testing.assert_array_equal(d32, nb.move_exp_nanmean(x, alpha=0.3).astype(np.float32))
    xt = np.ascontiguousarray(x.T)
    dm = np.empty((200, 3, 3))
    assert nb.move_covmatrix(xt, window=10, out=dm) is dm
    np.testing.assert_array_equal(dm, nb.move_covmatrix(xt, window=10))
    df = np.empty_like(x)
    xn = x.copy()
    xn[:, ::3] = np.nan
    assert nb.ffill(xn, out=df) is df
    np.testing.assert_array_equal(df, nb.ffill(xn))
    with pytest.raises(ValueError):
        nb.move_mean(x, window=5, out=np.empty((3, 100)))


@pytest.mark.parametrize("func", ["move_sum", "move_mean", "move_var", "move_std", "move_corr"])
def test_element_aligned_rows_match_contiguous(gpu_lib, func):
    """Rows that start one element past a 16-byte boundary (a sliced device
    tensor) take the 16-byte vector paths at element alignment (streaming
    prefetch loads, LDS-staged stores): bitwise the results of an aligned
    contiguous copy."""
    import torch
    import numbagg_amd as nb

    x = torch.from_numpy(walk_array(3, 40_001, seed=21, offset=0.0)).cuda()
    y = torch.from_numpy(walk_array(3, 40_001, seed=22, offset=0.0)).cuda()
    xv, yv = x[:, 1:], y[:, 1:]
    assert xv.data_ptr() % 16 == 4
    args_v = (xv, yv) if func == "move_corr" else (xv,)
    args_c = tuple(a.contiguous() for a in args_v)
    got = getattr(nb, func)(*args_v, window=1000, min_count=500)
    want = getattr(nb, func)(*args_c, window=1000, min_count=500)
    assert torch.equal(got.view(torch.int32), want.view(torch.int32))


# column counts around the wave, lengths around the 32-position tile and the
# ranges of positions, windows from 1 to the longest the kernel takes
@pytest.mark.parametrize("func", FUNCS1 + FUNCS2)
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("shape,window,min_count", [
    ((1, 33, 32), 1, 0), ((2, 64, 64), 7, None), ((1, 200, 65), 64, 10), ((3, 129, 130), 128, 1),
    ((1, 1000, 33), 5, 2), ((1, 31, 200), 31, 4), ((2, 3000, 40), 100, 50)])
def test_move_inner_axis_kept(gpu_lib, func, dtype, shape, window, min_count):
    """Windows along an axis in front of the innermost (read as it lies, also
    at odd element offsets) against the exact oracle, with the bars above."""
    import torch

    import numbagg_amd as nb
    from numbagg_amd import _lib
    from oracle import exact

    code = _lib.NBG_F32 if dtype == np.float32 else _lib.NBG_F64
    assert _lib.query("nbg_move_cols_chunk", code, *shape, window) > 0
    full = [walk_array(shape[0] * (shape[2] + 1), shape[1], seed=s + shape[1], dtype=dtype)
            .reshape(shape[0], shape[2] + 1, shape[1]) for s in range(2 if func in FUNCS2 else 1)]
    rows = [np.ascontiguousarray(x[:, 1:]).reshape(-1, shape[1]) for x in full]
    tens = [torch.from_numpy(np.ascontiguousarray(x.transpose(0, 2, 1))).cuda()[:, :, 1:] for x in full]
    got = getattr(nb, func)(*tens, window=window, min_count=min_count, axis=1)
    assert tuple(got.shape) == shape
    assert got.movedim(1, -1).is_contiguous()  # the layout of the general path
    got = got.movedim(1, -1).reshape(-1, shape[1]).cpu().numpy()
    want = exact.move(func, rows[0], window, min_count, y=rows[1] if func in FUNCS2 else None)
    if dtype == np.float32:
        check_f32(func, got, want, scale=np.ones_like(want))
        return
    assert np.array_equal(np.isnan(got), np.isnan(want))
    ok = ~np.isnan(want)
    assert_allclose(got[ok], want[ok], rtol=1e-11, atol=1e-13)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_move_inner_axis_kept_infinities(gpu_lib, dtype):
    """An infinity shows in the windows that hold it and in no later one."""
    import torch

    import numbagg_amd as nb

    rng = np.random.default_rng(3)
    x = rng.standard_normal((300, 70)).astype(dtype)
    x[50, 3], x[52, 3], x[100, 4] = np.inf, np.inf, -np.inf
    t = torch.from_numpy(x).cuda()
    s = nb.move_sum(t, window=10, min_count=1, axis=0).cpu().numpy()
    v = nb.move_var(t, window=10, min_count=2, axis=0).cpu().numpy()
    assert (s[50:62, 3] == np.inf).all() and (s[100:110, 4] == -np.inf).all()
    hit = np.zeros(x.shape, bool)
    hit[50:62, 3] = hit[100:110, 4] = True
    assert np.isfinite(s[~hit]).all()
    assert np.isnan(v[hit]).all() and np.isfinite(v[1:][~hit[1:]]).all()


def test_move_inner_axis_kept_falls_back(gpu_lib):
    """Few columns, long windows, broadcast operands and unlike layouts run on
    the general path, with the same results."""
    import torch

    import numbagg_amd as nb

    x = torch.from_numpy(walk_array(3000, 48, seed=1)).cuda()
    y = torch.from_numpy(walk_array(48, 3000, seed=2)).cuda().t()
    for a, kw in (((x[:, :5],), dict(window=9)), ((x,), dict(window=1500, min_count=3))):
        want = nb.move_mean(a[0].t().contiguous(), axis=-1, **kw).t()
        assert torch.equal(nb.move_mean(*a, axis=0, **kw).nan_to_num(), want.nan_to_num())
    got = nb.move_cov(x, y, window=20, axis=0)
    want = nb.move_cov(x.t().contiguous(), y.t(), window=20, axis=-1).t()
    assert torch.equal(got.nan_to_num(), want.nan_to_num())


@pytest.mark.parametrize("dtype,n,cols", [(np.float32, 1021, 33_003), (np.float64, 517, 33_001)])
def test_move_inner_axis_kept_large_output(gpu_lib, dtype, n, cols):
    """Outputs over 128 MB leave line by line, at every offset of a series
    within its line: equal to the general path on a transposed copy up to one
    rounding of each (means of data around 1e4)."""
    import torch

    import numbagg_amd as nb

    g = torch.Generator(device="cuda").manual_seed(n)
    x = torch.randn(n, cols, generator=g, device="cuda", dtype=torch.float32 if dtype == np.float32 else torch.float64)
    x += 1e4
    x[torch.rand(n, cols, generator=g, device="cuda") < 0.1] = float("nan")
    got = nb.move_mean(x, window=30, min_count=20, axis=0).movedim(0, -1)
    want = nb.move_mean(x.t().contiguous(), window=30, min_count=20)
    assert torch.equal(got.isnan(), want.isnan())
    off = ((got - want).abs() / want.abs()).nan_to_num_(nan=0.0).max().item()
    assert off <= (1.2e-7 if dtype == np.float32 else 4.5e-16)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("func", ["move_var", "move_std", "move_cov", "move_corr"])
def test_move_inner_axis_kept_first_value_infinite(gpu_lib, func, dtype):
    """An infinity that comes first (in a series, after leading missing values,
    before or in a later range of positions) leaves with its window: the
    outputs of windows without one are those of the series with the infinities
    missing."""
    import torch

    import numbagg_amd as nb
    from numbagg_amd import _lib
    from oracle import exact

    n, cols, window = 600, 40, 10
    tc = _lib.query("nbg_move_cols_chunk", _lib.NBG_F32 if dtype == np.float32 else _lib.NBG_F64, 1, n, cols, window)
    assert 2 * window < tc < n // 4
    rng = np.random.default_rng(7)
    x, y = (rng.standard_normal((n, cols)).astype(dtype) + 3 for _ in range(2))
    for c, (lo, at) in enumerate([(0, 0), (0, 5), (tc - window, tc - window), (tc - window - 3, tc - 4), (tc, tc),
                                  (tc - window, tc + 2)]):
        for z, other in ((x, 2 * c), (y, 2 * c + 1)):
            z[lo:at, other] = np.nan
            z[at, other] = np.inf if c % 2 else -np.inf
    x[-1, 20] = np.inf  # the last window
    args = (x, y) if func in ("move_cov", "move_corr") else (x,)
    clean = [np.where(np.isinf(z), np.nan, z) for z in args]
    hit = np.zeros(x.shape, bool)
    for z in args:
        for t, c in np.argwhere(np.isinf(z)):
            hit[t:t + window, c] = True
    got = getattr(nb, func)(*(torch.from_numpy(z).cuda() for z in args), window=window, min_count=3, axis=0)
    got = got.cpu().numpy()
    want = exact.move(func, np.ascontiguousarray(clean[0].T), window, 3,
                      y=np.ascontiguousarray(clean[-1].T) if len(args) == 2 else None).T
    ok = ~hit
    assert np.array_equal(np.isnan(got[ok]), np.isnan(want[ok]))
    assert_allclose(got[ok], want[ok], rtol=2.4e-7 if dtype == np.float32 else 1e-11,
                    atol=1e-6 if dtype == np.float32 else 1e-13)


def test_move_inner_axis_kept_extreme_scales(gpu_lib):
    """float64 data whose sums of squares lie near the end of the range: the
    moments that the row kernel gives (shifts of 0 on both sides, so that the
    row kernel's squared sums of 100 values stay in range)."""
    import torch

    import numbagg_amd as nb
    from numbagg_amd import _lib

    rng = np.random.default_rng(2)
    x, y = (torch.from_numpy(rng.standard_normal((400, 48))).cuda() for _ in range(2))
    tc = _lib.query("nbg_move_cols_chunk", _lib.NBG_F64, 1, 400, 48, 100)
    for z in (x, y):  # the first value of each range's first window
        z[0] = 0
        z[[t for t in range(-100, 400, tc) if t >= 0 and (t + 100) % tc == 0]] = 0
    for func, scales in (("move_var", (2e152,)), ("move_std", (2e152,)), ("move_cov", (2e152, 2e152)),
                         ("move_corr", (2e75, 2e75)), ("move_corr", (1e152, 1.0))):
        args = [a * s for a, s in zip((x, y), scales)]
        got = getattr(nb, func)(*args, window=100, min_count=2, axis=0)
        want = getattr(nb, func)(*(a.t().contiguous() for a in args), window=100, min_count=2, axis=-1).t()
        assert torch.equal(got.isfinite(), want.isfinite()) and got[1:].isfinite().all(), func
        assert_allclose(got[1:].cpu().numpy(), want[1:].cpu().numpy(), rtol=1e-11,
                        atol=1e-11 if func == "move_corr" else 1e-11 * scales[0] * scales[-1], err_msg=func)


def test_move_inner_axis_kept_constant_windows_f64(gpu_lib):
    """float64 windows of one repeated value that follow other values have
    variance exactly zero and no correlation."""
    import torch

    import numbagg_amd as nb

    rng = np.random.default_rng(6)
    x = rng.uniform(-500, 500, (600, 200))
    x[70:] = x[70]
    y = rng.standard_normal(x.shape)
    a, b = torch.from_numpy(x).cuda(), torch.from_numpy(y).cuda()
    assert (nb.move_var(a, window=30, axis=0)[99:] == 0).all()
    assert (nb.move_std(a, window=30, axis=0)[99:] == 0).all()
    assert nb.move_corr(a, b, window=30, axis=0)[99:].isnan().all()


@pytest.mark.parametrize("axis", [-1, 0])
def test_move_corr_constant_windows(gpu_lib, axis):
    """Windows of one repeated value have no correlation, also where that value
    is not the shift: its sums and sums of squares are exact (24-bit values from
    a shift of 0, 30 of them)."""
    import torch

    import numbagg_amd as nb

    rng = np.random.default_rng(5)
    x = np.repeat(rng.uniform(-500, 500, (64, 1)).astype(np.float32), 200, axis=1)
    x[:, 0] = 0
    y = rng.standard_normal(x.shape).astype(np.float32)
    a, b = (torch.from_numpy(np.ascontiguousarray(z if axis else z.T)).cuda() for z in (x, y))
    got = nb.move_corr(a, b, window=30, min_count=2, axis=axis).cpu().numpy()
    got = got if axis else got.T
    assert np.isnan(got[:, 30:]).all()
