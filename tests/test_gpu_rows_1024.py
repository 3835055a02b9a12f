"""Rows of 1024 pixels on both sides of the launch size at which the persistent
row kernel takes over (8 rounds of the workgroups the chip holds, three to a
CU), with a last frame block that is not full."""

import numpy as np
import pytest

from oracle import oracle_np as onp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "fp32c"])
@pytest.mark.parametrize("L", [9, 73])  # 768-row blocks of 4 (FP64) or 8 frames: up to 2304, from 7680 rows against 6144
def test_rows_of_1024_match_oracle(hip, L, precision):
    H, W = 768, 1024
    img = np.random.default_rng(L).integers(800, 1200, (L, H, W)).astype(np.uint16)
    lags = np.array([1, L // 2])
    got = hip.ddm_diff(img, lags, W, H, None, precision=precision)
    ref = onp.ddm_diff(img, lags, W, H, None)
    if precision == "fp64":
        for s in range(ref.shape[0]):
            assert np.allclose(got[s], ref[s], rtol=1e-9, atol=1e-12 * np.max(np.abs(ref[s]))), s
    else:
        assert np.allclose(got, ref, rtol=1e-3, atol=0)
        assert np.median(onp.relative_error(got, ref)) <= 1e-5
