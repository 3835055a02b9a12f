"""The fft time stage of short series on both sides of the plane sizes at which
the kernel with a column's transforms in registers takes over from the one with
them in LDS, on real hardware: the shortest and longest series of every
transform length, dense and sparse lag lists, columns that leave a workgroup
partly empty, columns marked for the recomputation."""

import numpy as np
import pytest

from fastddm_amd import next_fast_len
from oracle import oracle_np as onp

pytestmark = pytest.mark.gpu


def _check(out, ref, precision):
    if precision == "fp64":
        for s in range(ref.shape[0]):
            assert np.allclose(out[s], ref[s], rtol=1e-9, atol=1e-12 * np.max(np.abs(ref[s]))), s
    elif precision == "fp32c":
        assert np.allclose(out, ref, rtol=1e-3, atol=0)
        assert np.median(onp.relative_error(out, ref)) <= 1e-5
    else:
        assert np.isfinite(out).all()
        assert np.median(onp.relative_error(out, ref)) <= 1e-4


# 3, 819, 910, 1092, 1170, 1456 and 1560 columns: around 850, 1100 and 1500
PLANES = [(3, 1), (63, 24), (70, 24), (84, 24), (90, 24), (112, 24), (120, 24)]


@pytest.mark.parametrize("precision", ["fp64", "fp32c", "fp32"])
@pytest.mark.parametrize("H,W", PLANES)
def test_every_lag(hip, H, W, precision):
    ny, nx = next_fast_len(H, "hip"), next_fast_len(W, "hip")
    for L in (2, 3, 33, 64, 65, 128, 129, 200, 256, 257, 300, 512, 513, 1024):
        img = (900 + 200 * np.random.default_rng(L).random((L, H, W))).astype(np.uint16)
        lags = np.arange(1, L)
        ref = onp.ddm_fft(img, lags, nx, ny, 2 * L, None, subtract_mean=True)
        out = hip.ddm_fft(img, lags, nx, ny, next_fast_len(2 * L, "hip"), None, precision=precision)
        _check(out, ref, precision)


@pytest.mark.parametrize("precision", ["fp64", "fp32c", "fp32"])
@pytest.mark.parametrize("H,W", [(5, 9), (60, 50), (120, 140)])  # 25, 1560 and 8520 columns
def test_few_lags(hip, H, W, precision):
    ny, nx = next_fast_len(H, "hip"), next_fast_len(W, "hip")
    for L in (20, 128, 129, 256, 300, 512, 600):
        img = (900 + 200 * np.random.default_rng(L).random((L, H, W))).astype(np.uint16)
        lags = np.unique(np.geomspace(1, L - 1, max(2, min(7, L // 8))).astype(int))
        assert len(lags) <= L // 8
        ref = onp.ddm_fft(img, lags, nx, ny, 2 * L, None, subtract_mean=True)
        for out_dtype in (np.float64, np.float32):
            out = hip.ddm_fft(img, lags, nx, ny, next_fast_len(2 * L, "hip"), None, precision=precision, out_dtype=out_dtype)
            if precision == "fp64" and out_dtype == np.float32:
                assert np.allclose(out, ref, rtol=2e-7, atol=1e-12 * np.max(ref))
            else:
                _check(out, ref, precision)


@pytest.mark.parametrize("L,lag", [(100, 61), (250, 131), (600, 333), (1000, 701)])
def test_one_small_lag_marks_every_column(hip, L, lag):
    """Frames that recur once: D at that lag is 1e-5 of the variance, right only
    if the column is marked."""
    rng = np.random.default_rng(lag)
    H, W = 48, 64  # 1584 columns
    base = rng.normal(10000.0, 1000.0, (lag, H, W))
    img = np.concatenate([base, base[: L - lag]]) + rng.normal(0.0, 3.0, (L, H, W))
    img = np.rint(img).astype(np.uint16)
    ref = onp.ddm_diff(img, np.array([lag]), W, H, None)
    assert np.median(ref[0] / ref[-1]) < 1e-4
    out = hip.ddm_fft(img, np.arange(1, L), W, H, next_fast_len(2 * L, "hip"), None, precision="fp32c")
    assert np.allclose(out[lag - 1], ref[0], rtol=1e-3, atol=0)
