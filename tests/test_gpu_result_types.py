"""The register time kernels and the direct-difference kernels in every
precision with double and single results, on real hardware: the shortest and
longest series of every form; planes whose lag rows leave in whole vectors
(60 columns) and one by one (25), both with a workgroup that is partly empty."""

import numpy as np
import pytest

from fastddm_amd import next_fast_len
from oracle import oracle_np as onp

pytestmark = pytest.mark.gpu

TYPES = [("fp64", np.float32), ("fp32c", np.float32), ("fp32", np.float32), ("fp32", np.float64),
         ("fp64", np.float64), ("fp32c", np.float64)]


def _check(out, ref, precision, out_dtype):
    assert out.dtype == out_dtype
    if precision == "fp64":
        rtol = 1e-9 if out_dtype == np.float64 else 2e-7  # (and the rounding to float)
        for s in range(ref.shape[0]):
            assert np.allclose(out[s], ref[s], rtol=rtol, atol=1e-12 * np.max(np.abs(ref[s]))), s
    elif precision == "fp32c":
        assert np.allclose(out, ref, rtol=1e-3, atol=0)
        assert np.median(onp.relative_error(out, ref)) <= 1e-5
    else:
        # plain FP32 does not resolve D beside the mean intensity at k = 0
        assert np.isfinite(out).all()
        assert np.median(onp.relative_error(out, ref)) <= 1e-4


@pytest.mark.parametrize("precision,out_dtype", TYPES)
@pytest.mark.parametrize("H,W", [(5, 9), (12, 8)])
def test_time_kernels(hip, H, W, precision, out_dtype):
    nx, ny = next_fast_len(W, "hip"), next_fast_len(H, "hip")
    assert (nx // 2 + 1) * ny == (25 if W == 9 else 60)
    for L in (2, 128, 129, 256, 257, 512, 513, 1024, 1025, 2048, 2049, 4096):
        img = (900 + 200 * np.random.default_rng(L).random((L, H, W))).astype(np.uint16)
        for lags in (np.arange(1, L), np.unique(np.geomspace(1, L - 1, 7).astype(int))):
            ref = onp.ddm_fft(img, lags, nx, ny, 2 * L, None, subtract_mean=True)
            out = hip.ddm_fft(img, lags, nx, ny, next_fast_len(2 * L, "hip"), None, precision=precision, out_dtype=out_dtype)
            _check(out, ref, precision, out_dtype)


@pytest.mark.parametrize("precision,out_dtype", TYPES)
@pytest.mark.parametrize("H,W", [(5, 9), (12, 8)])
def test_difference_kernels(hip, H, W, precision, out_dtype):
    nx, ny = next_fast_len(W, "hip"), next_fast_len(H, "hip")
    for L in (2, 17, 160, 161, 320, 321, 640, 641, 2600, 5100, 10400, 20400):
        img = (900 + 200 * np.random.default_rng(L).random((L, H, W))).astype(np.uint16)
        few = np.unique(np.geomspace(1, L - 1, 9 if L < 4000 else 5).astype(int))
        for lags in (few, few[-1:]):
            ref = onp.ddm_diff(img, lags, nx, ny)
            out = hip.ddm_diff(img, lags, nx, ny, None, precision=precision, out_dtype=out_dtype)
            _check(out, ref, precision, out_dtype)
