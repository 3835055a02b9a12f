"""Transform lengths that are no power of two, on real hardware: every radix
of the pass plans (alone, paired with a factor 2, repeated), and the row
kernel's forms (four, two or one image row to a wave, long rows) at the edges
of their ranges, with image heights that leave part of a wave without a row."""

import numpy as np
import pytest

from fastddm_amd import next_fast_len
from oracle import oracle_np as onp

pytestmark = pytest.mark.gpu

# 2, 4, 8 and odd radices alone; 6 and 10 alone, together, repeated, beside 3s, 5s, 7s and 8s
FFT_SIZES = [2, 3, 5, 6, 7, 10, 12, 14, 20, 30, 36, 42, 60, 70, 90, 96, 100, 150, 210, 216, 336, 384, 480, 640, 735, 1000, 1080, 1920]


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-13), ("fp32", 2e-6)])
def test_fft_radices(hip, precision, tol):
    rng = np.random.default_rng(5)
    for n in FFT_SIZES:
        z = rng.standard_normal((3, n)) + 1j * rng.standard_normal((3, n))
        ref = np.fft.fft(z, axis=-1)
        got = hip.device_fft(z, precision)
        assert np.max(np.abs(got - ref)) <= tol * max(1.0, np.log2(n) / 4) * np.max(np.abs(ref)), n


# width -> transform length: 4 rows to a wave up to 160, 2 up to 320, 1 above
WIDTHS = [63, 96, 150, 160, 162, 201, 315, 320, 324, 768, 784]


@pytest.mark.parametrize("precision", ["fp64", "fp32c"])
@pytest.mark.parametrize("W", WIDTHS)
def test_row_forms_match_oracle(hip, W, precision):
    rng = np.random.default_rng(W)
    H, L = 21, 850  # 54 (FP32) or 107 (FP64) frame blocks x 21 rows: more than one round of the chip
    img = (900 + 200 * rng.random((L, H, W))).astype(np.uint16)
    nx, ny = next_fast_len(W, "hip"), next_fast_len(H, "hip")
    lags = np.array([1, 30, 600])
    ref = onp.ddm_diff(img, lags, nx, ny, None)
    got = hip.ddm_diff(img, lags, nx, ny, None, precision=precision)
    if precision == "fp64":
        for s in range(ref.shape[0]):
            assert np.allclose(got[s], ref[s], rtol=1e-9, atol=1e-12 * np.max(np.abs(ref[s]))), s
    else:
        assert np.allclose(got, ref, rtol=1e-3, atol=0)
        assert np.median(onp.relative_error(got, ref)) <= 1e-5
