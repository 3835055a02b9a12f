"""The workgroup column kernel on real hardware: image heights below 256 with
every radix of its plans alone, repeated and paired with a factor 2."""

import numpy as np
import pytest

from fastddm_amd import next_fast_len
from oracle import oracle_np as onp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "fp32c"])
def test_columns_match_oracle(hip, precision):
    for H in (1, 2, 3, 5, 6, 7, 10, 12, 27, 36, 49, 60, 63, 96, 100, 105, 120, 125, 128, 147, 150, 180, 200, 210, 216, 225, 240, 245, 250):
        L, W = 19, 6  # a last frame block that is not full
        img = np.random.default_rng(H).integers(800, 1200, (L, H, W)).astype(np.uint16)
        assert next_fast_len(H, "hip") == H
        lags = np.array([1, 9, 18])
        ref = onp.ddm_diff(img, lags, W, H)
        out = hip.ddm_diff(img, lags, W, H, None, precision=precision)
        if precision == "fp64":
            for s in range(ref.shape[0]):
                assert np.allclose(out[s], ref[s], rtol=1e-9, atol=1e-12 * np.max(np.abs(ref[s]))), (H, s)
        else:
            assert np.allclose(out, ref, rtol=1e-3, atol=0), H
