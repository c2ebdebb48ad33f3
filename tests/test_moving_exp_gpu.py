"""GPU parity of the exponentially weighted kernels.

Bars against the long-double exact oracle (NaN masks identical):
  float64 loop: count/mean/sum <= 1e-12 relative (+ 1e-12 of max|x|, for means
  that cancel to near zero); var/std/cov/corr <= 1e-9
  relative + 1e-9 absolute of the data scale (the reference formula
  E[x^2]-E[x]^2 loses digits for offset data);
  float32 loop: <= 2 float32 ULP (var/std/cov/corr: or 1e-6 absolute).
The reference's pandas vectors and known answers are reproduced.
"""

from __future__ import annotations

import numpy as np
import pytest
from numpy.testing import assert_allclose

from ._data import walk_array

pytestmark = pytest.mark.gpu

FUNCS1 = ["move_exp_nancount", "move_exp_nanmean", "move_exp_nansum", "move_exp_nanvar", "move_exp_nanstd"]
FUNCS2 = ["move_exp_nancov", "move_exp_nancorr"]
MOMENTS = {"move_exp_nanvar", "move_exp_nanstd", "move_exp_nancov", "move_exp_nancorr"}


def _args(func, x, y):
    return (x,) if func in FUNCS1 else (x, y)


@pytest.mark.parametrize("func", FUNCS1 + FUNCS2)
@pytest.mark.parametrize("shape,alpha", [((3, 500), 0.5), ((4, 70_000), 0.01), ((2, 9000), 0.001), ((1, 300_000), 0.05), ((33, 4097), 0.3)])
def test_exp_float64_loop_against_exact(gpu_lib, func, shape, alpha):
    """float32 data with a Python-float alpha runs on the float64 loop."""
    import numbagg_amd as nb
    from oracle import exact

    x = walk_array(*shape, seed=shape[1], offset=100.0)
    y = walk_array(*shape, seed=shape[1] + 7, offset=-50.0)
    got = getattr(nb, func)(*_args(func, x, y), alpha=alpha)
    assert got.dtype == np.float64
    want = exact.move_exp(func, x, alpha, y=y if func in FUNCS2 else None, loop_dtype=np.float64)
    assert np.array_equal(np.isnan(got), np.isnan(want)), func
    ok = ~np.isnan(want)
    scale = float(np.nanmax(np.abs(x)))
    if func in MOMENTS:
        assert_allclose(got[ok], want[ok], rtol=1e-9, atol=1e-9 * scale**2)
    else:
        # relative to the data's scale: a mean near zero is a cancellation
        assert_allclose(got[ok], want[ok], rtol=1e-12, atol=1e-12 * scale)


@pytest.mark.parametrize("two_pass", ["1", "0"])
@pytest.mark.parametrize("func", FUNCS1 + FUNCS2)
def test_exp_two_pass_against_exact(gpu_lib, monkeypatch, two_pass, func):
    """The two-pass path (tile aggregates, per-row scan, apply) and the
    single pass with look-back meet the same bars: rows of more than 256
    tiles (several chunks of the row scan), partial last tiles, NaN stretches
    longer than a tile, scalar and per-position alpha."""
    import numbagg_amd as nb
    from oracle import exact

    monkeypatch.setenv("NBG_EXP_TWO_PASS", two_pass)
    x = walk_array(2, 1_100_003, seed=11, offset=30.0)
    y = walk_array(2, 1_100_003, seed=12, offset=-20.0)
    x[0, 5000:20_000] = np.nan
    y[1, 700_000:720_000] = np.nan
    scale = float(np.nanmax(np.abs(x)))
    for alpha in (0.01, np.linspace(0.005, 0.05, x.shape[1])):
        got = getattr(nb, func)(*_args(func, x, y), alpha=alpha, min_weight=0.2)
        want = exact.move_exp(func, x, alpha, 0.2, y=y if func in FUNCS2 else None, loop_dtype=np.float64)
        assert np.array_equal(np.isnan(got), np.isnan(want)), func
        ok = ~np.isnan(want)
        if func in MOMENTS:
            assert_allclose(got[ok], want[ok], rtol=1e-9, atol=1e-9 * scale**2)
        else:
            assert_allclose(got[ok], want[ok], rtol=1e-12, atol=1e-12 * scale)
    # float32 loop (float32 alpha array), several rows of partial tiles
    x32 = walk_array(9, 300_001, seed=13, offset=0.0)
    y32 = walk_array(9, 300_001, seed=14, offset=0.0)
    al = np.full(300_001, 0.03, dtype=np.float32)
    got = getattr(nb, func)(*_args(func, x32, y32), alpha=al)
    want = exact.move_exp(func, x32, al, y=y32 if func in FUNCS2 else None, loop_dtype=np.float32)
    assert np.array_equal(np.isnan(got), np.isnan(want)), func
    ok = ~np.isnan(want)
    e = want[ok].astype(np.float32)
    ulps = np.abs(got[ok].astype(np.float64) - want[ok]) / np.spacing(np.abs(e)).astype(np.float64)
    if func in MOMENTS:
        assert np.all((ulps <= 2) | (np.abs(got[ok] - want[ok]) <= 1e-6 * np.maximum(1, np.abs(want[ok])))), ulps.max()
    else:
        assert ulps.max() <= 2, ulps.max()


@pytest.mark.parametrize("func", FUNCS1 + FUNCS2)
def test_exp_float32_loop_against_exact(gpu_lib, func):
    import numbagg_amd as nb
    from oracle import exact

    x = walk_array(6, 20_000, seed=3, offset=0.0)
    y = walk_array(6, 20_000, seed=4, offset=0.0)
    alpha = np.full(20_000, 0.02, dtype=np.float32)
    got = getattr(nb, func)(*_args(func, x, y), alpha=alpha, min_weight=0.5)
    assert got.dtype == np.float32
    want = exact.move_exp(func, x, alpha, 0.5, y=y if func in FUNCS2 else None, loop_dtype=np.float32)
    assert np.array_equal(np.isnan(got), np.isnan(want)), func
    ok = ~np.isnan(want)
    e = want[ok].astype(np.float32)
    ulps = np.abs(got[ok].astype(np.float64) - want[ok]) / np.spacing(np.abs(e)).astype(np.float64)
    if func in MOMENTS:
        assert np.all((ulps <= 2) | (np.abs(got[ok] - want[ok]) <= 1e-6 * np.maximum(1, np.abs(want[ok])))), ulps.max()
    else:
        assert ulps.max() <= 2, ulps.max()


@pytest.mark.parametrize("func", FUNCS1 + FUNCS2)
def test_exp_against_restated_reference(gpu_lib, func):
    import numbagg_amd as nb
    from oracle import restated

    rng = np.random.default_rng(11)
    x = rng.standard_normal((5, 12_345))
    x[rng.random(x.shape) < 0.05] = np.nan
    y = rng.standard_normal((5, 12_345))
    got = getattr(nb, func)(*_args(func, x, y), alpha=0.07, min_weight=0.3)
    ref = restated.move_exp(func, x, 0.07, 0.3, y=y if func in FUNCS2 else None)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert_allclose(got, ref, rtol=1e-10, atol=1e-12)


@pytest.mark.parametrize("func", FUNCS1 + FUNCS2)
@pytest.mark.parametrize("alpha", [0.5, 0.1])
def test_exp_reference_pandas_vectors(gpu_lib, golden, func, alpha):
    import numbagg_amd as nb

    a, a2 = golden["array_3x500"], golden["array2_3x500"]
    got = getattr(nb, func)(*_args(func, a, a2), alpha=alpha)
    assert_allclose(got, golden[f"{func}_a{alpha}"])
    # 1-D alpha along the axis, and the transposed layout (test_moving_exp.py:348-368)
    alphas = np.full(a.shape[-1], alpha)
    assert_allclose(getattr(nb, func)(*_args(func, a, a2), alpha=alphas), got)
    t_args = (a.T,) if func in FUNCS1 else (a.T, a2.T)
    assert_allclose(getattr(nb, func)(*t_args, alpha=alphas, axis=0).T, got)
    assert_allclose(getattr(nb, func)(*t_args, alpha=alpha, axis=0).T, got)


def test_exp_known_answers(gpu_lib):
    import numbagg_amd as nb

    assert_allclose(nb.move_exp_nanmean(np.array([10, 0, np.nan, 10]), alpha=0.5), [10.0, 3.3333333, 3.3333333, 8.1818182])
    assert_allclose(nb.move_exp_nanmean(np.array([10, 0, np.nan, 10]), alpha=0.25), [10.0, 4.2857143, 4.2857143, 7.1653543])
    assert_allclose(nb.move_exp_nancount(np.array([1, 0, np.nan, np.nan, 1, 0]), alpha=0.5), [1.0, 1.5, 0.75, 0.375, 1.1875, 1.59375])
    assert_allclose(nb.move_exp_nansum(np.array([10, 0, np.nan, 10]), alpha=0.25), [10.0, 7.5, 5.625, 14.21875])
    assert_allclose(
        nb.move_exp_nancorr(np.array([10, 0, 5, 10]), np.array([10, 0, 10, 5]), alpha=0.5),
        [np.nan, 1.0, 0.8485281, 0.2274294],
    )
    # count vs sum on ones, count before observations (test_moving_exp.py:123-157)
    for alpha in (0.1, 0.5, 0.9):
        arr = np.array([1, 1, np.nan, np.nan, 1, 1])
        assert_allclose(nb.move_exp_nancount(arr, alpha=alpha), nb.move_exp_nansum(arr, alpha=alpha))
        r = nb.move_exp_nancount(np.array([np.nan, np.nan, 1.0, np.nan, 1.0]), alpha=alpha)
        assert r[0] == 0.0 and r[1] == 0.0 and r[2] == 1.0
        assert np.all(np.isnan(nb.move_exp_nansum(np.full(4, np.nan), alpha=alpha)))


def test_exp_min_weight_and_nan_masks(gpu_lib):
    import numbagg_amd as nb

    from .test_oracle_moving_exp import MIN_WEIGHT_CASES, NAN_MASK_CASES

    array = np.ones(25)
    array[:5] = np.nan
    for func in ["move_exp_nancount", "move_exp_nanmean", "move_exp_nanstd", "move_exp_nansum", "move_exp_nanvar"]:
        for mw, alpha, expected in MIN_WEIGHT_CASES:
            out = getattr(nb, func)(array, min_weight=mw, alpha=alpha)
            assert np.sum(~np.isnan(out)[6:]) == expected, (func, mw, alpha)
    for func in ["move_exp_nanvar", "move_exp_nanstd", "move_exp_nancov", "move_exp_nancorr"]:
        for alpha in (0.1, 0.5, 0.9):
            for x, want, want_corr in NAN_MASK_CASES:
                x = np.array(x)
                exp_mask = want_corr if (func == "move_exp_nancorr" and want_corr is not None) else want
                args = (x,) if func in FUNCS1 else (x, x)
                assert list(np.isnan(getattr(nb, func)(*args, alpha=alpha))) == exp_mask, (func, x, alpha)


def test_exp_inf_and_big_values(gpu_lib):
    # numbagg/test/test_moving_exp.py:251-295
    import numbagg_amd as nb

    assert_allclose(nb.move_exp_nanmean(np.array([np.inf]), alpha=0.25), [np.inf])
    np.testing.assert_array_equal(nb.move_exp_nanmean(np.array([0, 0, np.inf], dtype=np.float16), alpha=1.0), [0, 0, np.inf])
    np.testing.assert_array_equal(nb.move_exp_nanmean(np.array([0, np.inf, np.inf], dtype=np.float16), alpha=1.0), [0, np.inf, np.nan])
    big = np.array([[0.00000000e000, 1.19846209e308], [1.19846209e308, 1.19846209e308]])
    np.testing.assert_array_equal(nb.move_exp_nanmean(big, alpha=1.0), big)
    np.testing.assert_array_equal(nb.move_exp_nanmean(np.array([[0, np.nan]]), alpha=1.0), [[0, np.nan]])
    np.testing.assert_array_equal(nb.move_exp_nanmean(np.array([[1, np.nan]]), alpha=1.0), [[1, np.nan]])


def test_exp_alpha_modes_and_dtypes(gpu_lib):
    import torch

    import numbagg_amd as nb
    from oracle import exact

    rng = np.random.default_rng(2)
    x = rng.standard_normal((4, 5, 3000)).astype(np.float32)
    x[rng.random(x.shape) < 0.1] = np.nan
    # N-D alpha laid out like the input
    al = rng.uniform(0.01, 0.5, size=x.shape)
    got = nb.move_exp_nanmean(x, alpha=al)
    want = exact.move_exp("move_exp_nanmean", x.reshape(-1, 3000), al.reshape(-1, 3000), loop_dtype=np.float64)
    assert_allclose(got.reshape(-1, 3000), want, rtol=1e-12, atol=1e-12 * np.nanmax(np.abs(x)))
    # axis=1 with an N-D alpha
    got = nb.move_exp_nanvar(x, alpha=al, axis=1)
    xm, am = np.moveaxis(x, 1, -1), np.moveaxis(al, 1, -1)
    want = exact.move_exp("move_exp_nanvar", xm.reshape(-1, 5), am.reshape(-1, 5), loop_dtype=np.float64).reshape(xm.shape)
    assert_allclose(got, np.moveaxis(want, -1, 1), rtol=1e-9, atol=1e-12)
    # axis tuple and empty tuple (test_moving_exp.py:371-391)
    arr = np.array([1.0, 2.0, 3.0, 4.0])
    assert_allclose(nb.move_exp_nansum(arr, alpha=0.5, axis=(0,)), nb.move_exp_nansum(arr, alpha=0.5, axis=0))
    assert_allclose(nb.move_exp_nansum(arr, alpha=np.full(4, 0.5), axis=(0,)), nb.move_exp_nansum(arr, alpha=0.5))
    assert nb.move_exp_nansum(arr, alpha=0.5, axis=()) is arr
    # float32 alpha keeps the float32 loop; device tensors stay on the device
    t = torch.from_numpy(x[0]).cuda()
    r = nb.move_exp_nanmean(t, alpha=np.float32(0.1))
    assert r.is_cuda and r.dtype == torch.float32
    # big-endian input (test_moving_exp.py:312-320)
    a = rng.random((3, 500))
    assert_allclose(nb.move_exp_nanmean(a.astype(">f8"), alpha=0.25), nb.move_exp_nanmean(a, alpha=0.25))


@pytest.mark.parametrize("two_pass", ["0", "1", ""])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("func", FUNCS1 + FUNCS2)
def test_exp_scalar_alpha_matches_alpha_array(gpu_lib, monkeypatch, func, dtype, two_pass):
    """One alpha for all positions (its own kernel, in one pass or two) against
    the same alpha as an array (the general kernel): lengths around the tiles,
    long gaps whose weights fall below 2**-200, infinities, alphas at and beyond
    the ends of [0, 1], weight thresholds. Both stay within 1e-12 (moments 1e-9)
    of the exact recurrence by this file's bars, so within twice that of each
    other."""
    import numbagg_amd as nb
    from oracle import exact

    monkeypatch.setenv("NBG_EXP_TWO_PASS", two_pass)
    cases = [(3, 2047, 0.3, 0), (1, 2049, 0.05, 0), (2, 4096, 1.0, 0), (2, 8193, 0.0, 0), (5, 16_385, 0.01, 0.2),
             (1, 300_001, 0.02, -1.0), (40, 5000, 0.05, 0), (2, 700, 1.5, 0)]
    for rows, n, alpha, mw in cases:
        x = walk_array(rows, n, seed=n, dtype=dtype, offset=5.0)
        y = walk_array(rows, n, seed=n + 1, dtype=dtype, offset=-3.0)
        if n > 16_000:
            x[0, 1000:14_000] = np.nan
            if func in FUNCS1:  # (a co-moment's infinity is signed by the data's shift)
                x[-1, 15_000] = np.inf
        got = getattr(nb, func)(*_args(func, x, y), alpha=alpha, min_weight=mw)
        if n > 16_000:
            # the exact recurrence, in which an infinity stays: where the decay of
            # its tile underflows, the general kernel turns it into NaN
            want = exact.move_exp(func, x, alpha, mw, y=y if func in FUNCS2 else None, loop_dtype=np.float64)
        else:
            want = getattr(nb, func)(*_args(func, x, y), alpha=np.full(n, alpha), min_weight=mw)
        assert got.dtype == want.dtype == np.float64
        tag = f"{func} {rows}x{n} alpha {alpha}"
        assert np.array_equal(np.isnan(got), np.isnan(want)), tag
        ok = np.isfinite(want)
        assert np.array_equal(got[~ok], want[~ok], equal_nan=True), tag
        if func in MOMENTS:
            scale = float(np.nanmax(np.abs(x[np.isfinite(x)])))
            assert_allclose(got[ok], want[ok], rtol=2e-9, atol=2e-9 * scale**2, err_msg=tag)
        else:
            assert_allclose(got[ok], want[ok], rtol=2e-12, atol=2e-12 * float(np.nanmax(np.abs(x[np.isfinite(x)]))),
                            err_msg=tag)


def test_exp_scalar_alpha_constant_rows(gpu_lib):
    """Rows of one value have variance and deviation exactly zero."""
    import numbagg_amd as nb

    x = np.full((2, 9000), 0.1, dtype=np.float32)
    x[0, ::5] = np.nan
    for func in ("move_exp_nanvar", "move_exp_nanstd"):
        got = getattr(nb, func)(x, alpha=0.1)
        assert np.isnan(got[:, 0]).all() and (got[:, 2:] == 0).all()


@pytest.mark.parametrize("two_pass", ["0", "1"])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("alpha,mw", [(0.05, 0), (0.3, 0.2), (0.002, 0)])
def test_exp_std_is_the_root_of_var(gpu_lib, monkeypatch, dtype, two_pass, alpha, mw):
    """std is the square root of var, to within one unit of the last place. (In
    one pass, rows of one tile: the carry between tiles is summed in an order
    that depends on the timing, so two calls differ in their last digits.)"""
    import numbagg_amd as nb

    monkeypatch.setenv("NBG_EXP_TWO_PASS", two_pass)
    x = walk_array(20 if two_pass == "0" else 4, 4000 if two_pass == "0" else 20_000, seed=11, dtype=dtype, offset=50.0)
    var = nb.move_exp_nanvar(x, alpha=alpha, min_weight=mw)
    std = nb.move_exp_nanstd(x, alpha=alpha, min_weight=mw)
    assert np.array_equal(np.isnan(var), np.isnan(std))
    ok = var > 0
    assert ok.sum() > 70_000
    root = np.sqrt(var[ok])
    assert (np.abs(std[ok] - root) <= np.spacing(root)).all()


@pytest.mark.parametrize("two_pass", ["0", "1"])
@pytest.mark.parametrize("func", ["move_exp_nanmean", "move_exp_nansum", "move_exp_nanvar", "move_exp_nanstd",
                                  "move_exp_nancov", "move_exp_nancorr"])
def test_exp_scalar_alpha_infinite_sums(gpu_lib, monkeypatch, func, two_pass):
    """Sums that an observation or its square makes infinite stay so in every
    position that follows, whatever thread or tile it falls to: where the
    outputs are not finite they are those of an array of alphas."""
    import numbagg_amd as nb

    monkeypatch.setenv("NBG_EXP_TWO_PASS", two_pass)
    rng = np.random.default_rng(3)
    n, alpha = 9000, 0.02
    x, y = (rng.standard_normal((6, n)) for _ in range(2))
    x[0, 37], x[1, 4100], x[2, 500] = np.inf, -np.inf, 1e160
    x[3, 70], x[3, 2100], y[4, 15], y[5, 77] = np.inf, -np.inf, np.inf, -1e160
    two = func in ("move_exp_nancov", "move_exp_nancorr")
    args = (x, y) if two else (x,)
    with np.errstate(all="ignore"):
        got = getattr(nb, func)(*args, alpha=alpha)
        want = getattr(nb, func)(*args, alpha=np.full(n, alpha))
    bad = ~np.isfinite(want)
    assert bad.any()
    assert np.array_equal(got[bad], want[bad], equal_nan=True)
    assert np.isfinite(got[~bad]).all()


@pytest.mark.parametrize("two_pass", ["0", "1", ""])
@pytest.mark.parametrize("func", ["move_exp_nanvar", "move_exp_nanstd", "move_exp_nancov", "move_exp_nancorr"])
@pytest.mark.parametrize("rows,n,alpha", [(2, 16_385, 0.01), (1, 300_001, 0.02), (40, 30_000, 0.2)])
def test_exp_scalar_alpha_moments_to_local_scale(gpu_lib, monkeypatch, func, rows, n, alpha, two_pass):
    """Rows of many tiles against the exact recurrence, to 1e-9 of the moment's
    own scale: sqrt(var_a var_b) at that position (1 for the correlation)."""
    import numbagg_amd as nb
    from oracle import exact

    monkeypatch.setenv("NBG_EXP_TWO_PASS", two_pass)
    x = walk_array(rows, n, seed=n, offset=5.0)
    y = walk_array(rows, n, seed=n + 1, offset=-3.0)
    two = func in ("move_exp_nancov", "move_exp_nancorr")
    got = getattr(nb, func)(*((x, y) if two else (x,)), alpha=alpha)
    want = exact.move_exp(func, x, alpha, y=y if two else None, loop_dtype=np.float64)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    if func == "move_exp_nancorr":
        scale = np.ones_like(want)
    elif func == "move_exp_nancov":
        scale = np.sqrt(np.abs(exact.move_exp("move_exp_nancov", x, alpha, y=np.where(np.isnan(y), y, x),
                                              loop_dtype=np.float64)
                               * exact.move_exp("move_exp_nancov", y, alpha, y=np.where(np.isnan(x), x, y),
                                                loop_dtype=np.float64)))
    else:
        scale = np.abs(want)
    ok = ~np.isnan(want)
    err = np.abs(got[ok] - want[ok]) / np.maximum(scale[ok], 1e-3)
    assert (err <= 1e-9).all(), err.max()


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_exp_var_is_as_accurate_as_cov(gpu_lib, dtype):
    """A variance, whose threads take twice the positions of a covariance's, is
    off by no more than the covariance of the array with itself: in units of
    the squared distance from the shift, mean square over 1.6M positions, 10%
    for chance."""
    import numbagg_amd as nb
    from oracle import exact

    x = walk_array(16, 100_000, seed=21, dtype=dtype, offset=50.0, p_nan=0.0)
    want = exact.move_exp("move_exp_nanvar", x, 0.01, loop_dtype=np.float64)
    unit = (x.astype(np.float64) - x[:, :1]) ** 2 * 2.0**-53
    at = unit > 1e4 * 2.0**-53
    assert at.sum() > 1_000_000
    rms = [np.sqrt(np.mean(((got - want)[at] / unit[at]) ** 2))
           for got in (nb.move_exp_nanvar(x, alpha=0.01), nb.move_exp_nancov(x, x, alpha=0.01))]
    assert rms[0] <= 1.1 * rms[1], rms


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("rows", [127, 128, 129, 135])
def test_exp_row_slots(gpu_lib, monkeypatch, rows, dtype):
    """One pass over a number of rows that its grid rounds up to a multiple of
    8 (from 128 on): what two passes give, with this file's bars."""
    import numbagg_amd as nb

    x = walk_array(rows, 20_001, seed=rows, dtype=dtype, offset=5.0)
    y = walk_array(rows, 20_001, seed=rows + 1, dtype=dtype, offset=-3.0)
    scale = float(np.nanmax(np.abs(x)))
    for func in FUNCS1 + FUNCS2:
        out = {}
        for two in ("0", "1"):
            monkeypatch.setenv("NBG_EXP_TWO_PASS", two)
            out[two] = getattr(nb, func)(*_args(func, x, y), alpha=0.05)
        bar = 2e-9 if func in MOMENTS else 2e-12
        assert np.array_equal(np.isnan(out["0"]), np.isnan(out["1"])), func
        assert_allclose(out["0"], out["1"], rtol=bar, atol=bar * (scale**2 if func in MOMENTS else scale), err_msg=func)
