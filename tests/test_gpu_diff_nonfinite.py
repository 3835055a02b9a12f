"""Direct differences of stacks with frames that are not finite, on real
hardware: a lag none of whose pairs holds such a frame keeps its value,
whatever other lags its kernel works on beside it."""

import numpy as np
import pytest

from oracle import oracle_np as onp

pytestmark = pytest.mark.gpu

# series of every kernel: segments of 16 lanes, of 32, a column per workgroup, a column per wave
CASES = [("fp32c", 300), ("fp32c", 500), ("fp32c", 700), ("fp32c", 20400),
         ("fp64", 150), ("fp64", 300), ("fp64", 700), ("fp64", 10400)]


@pytest.mark.parametrize("precision,L", CASES)
def test_lags_without_the_frame_stay_finite(hip, precision, L):
    rng = np.random.default_rng(L)
    img = (900 + 200 * rng.random((L, 3, 4))).astype(np.float32)  # 9 columns
    f = L // 2 // 2 * 2  # frames f and f + 1 share one transform
    img[f, 1, 2] = np.nan
    img[f + 1, 0, 1] = np.inf
    # two lags with the frames in some pair, two without, all in one group of
    # four; then with remainders on both sides
    four = [L // 3, L * 9 // 20, L * 17 // 30, L * 2 // 3]
    for lags in (four, [1] + four, four + [L - 20, L - 10]):
        with np.errstate(invalid="ignore"):
            ref = onp.ddm_diff(img, np.array(lags), 4, 3)
        assert [bool(np.isfinite(r).all()) for r in ref[:-2]] == [d > max(f + 1, L - 1 - f) for d in lags]
        out = hip.ddm_diff(img, np.array(lags), 4, 3, None, precision=precision)
        assert np.array_equal(np.isfinite(out), np.isfinite(ref))
        ok = np.isfinite(ref)
        rtol = 1e-9 if precision == "fp64" else 1e-3
        assert np.allclose(out[ok], ref[ok], rtol=rtol, atol=1e-12 * np.max(ref[ok]) if precision == "fp64" else 0)
