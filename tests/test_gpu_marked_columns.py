"""Compensated FP32 with every column marked for the direct recomputation and
lags of few pairs beside it (one launch, fddm_edge.hip), on real hardware: a
stack that repeats itself, whose D is zero at the period."""

import numpy as np
import pytest

from fastddm_amd import next_fast_len
from oracle import oracle_np as onp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L", [30, 80, 700])
@pytest.mark.parametrize("out_dtype", [np.float64, np.float32])
def test_periodic_stack(hip, L, out_dtype):
    H, W, period = 96, 100, 16  # 4896 columns: more than there are workgroups
    img = np.random.default_rng(L).integers(800, 1200, (period, H, W)).astype(np.uint16)[np.arange(L) % period]
    lags = np.arange(1, L)
    out = hip.ddm_fft(img, lags, W, H, next_fast_len(2 * L, "hip"), None, precision="fp32c", out_dtype=out_dtype)
    for d in lags[L - lags > 32]:
        if d % period == 0:
            assert not out[d - 1].any(), d
    # whole periods of pairs: the mean over one is the mean over all
    for d in lags[(L - lags) % period == 0]:
        if d % period:
            F = onp.spectra(img[: period + d % period], W, H)
            D = np.fft.fftshift(np.mean(np.abs(F[d % period:] - F[:period]) ** 2, axis=0), axes=0)
            assert np.allclose(out[d - 1], D, rtol=1e-3, atol=0), d
    # few pairs
    for n in range(1, 9):
        d = L - n
        if d % period:
            F = onp.spectra(img[np.r_[0:n, d:L]], W, H)
            D = np.fft.fftshift(np.mean(np.abs(F[n:] - F[:n]) ** 2, axis=0), axes=0)
            assert np.allclose(out[d - 1], D, rtol=1e-3, atol=0), n
    assert np.isfinite(out).all()
