"""The direct-difference kernels at the edges of their ranges, on real
hardware: segments of 16 and 32 lanes, a column per workgroup of 4, 8 and 16
waves, a column per wave beyond the LDS; lag counts with remainders, columns
that leave the last workgroup partly empty."""

import numpy as np
import pytest

from oracle import oracle_np as onp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "fp32c"])
@pytest.mark.parametrize("L", [2, 5, 15, 16, 17, 33, 160, 161, 319, 320, 321, 640, 641, 2600, 5100, 10400, 20400])
def test_lengths_match_oracle(hip, L, precision):
    rng = np.random.default_rng(L)
    img = (900 + 200 * rng.random((L, 3, 4))).astype(np.uint16)  # 9 columns
    few = np.unique(np.geomspace(1, L - 1, 9 if L < 4000 else 5).astype(int))
    for lags in (few, few[:1], np.arange(1, min(L, 12))):
        ref = onp.ddm_diff(img, lags, 4, 3)
        out = hip.ddm_diff(img, lags, 4, 3, None, precision=precision)
        if precision == "fp64":
            for s in range(ref.shape[0]):
                assert np.allclose(out[s], ref[s], rtol=1e-9, atol=1e-12 * np.max(np.abs(ref[s]))), s
        else:
            assert np.allclose(out, ref, rtol=1e-3, atol=0)
