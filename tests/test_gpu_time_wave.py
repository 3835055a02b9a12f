"""The register-resident time kernels at the edges of their plans, on real
hardware: the shortest and longest series of every transform length, column
counts that leave a workgroup partly empty, dense and sparse lag lists."""

import numpy as np
import pytest

from fastddm_amd import next_fast_len
from oracle import oracle_np as onp

pytestmark = pytest.mark.gpu

# series of every transform length M = 128 ... 4096: its shortest, one with a
# remainder, its longest
LENGTHS = [2, 3, 33, 64, 65, 127, 128, 129, 200, 256, 257, 300, 512, 513, 700, 1024, 1025, 1500, 2048, 2049, 3000, 4096]


@pytest.mark.parametrize("precision", ["fp64", "fp32c"])
@pytest.mark.parametrize("L", LENGTHS)
def test_lengths_match_oracle(hip, L, precision):
    rng = np.random.default_rng(L)
    H, W = 5, 9  # 25 columns
    img = (900 + 200 * rng.random((L, H, W))).astype(np.uint16)
    nx, ny = next_fast_len(W, "hip"), next_fast_len(H, "hip")
    for lags in (np.arange(1, L), np.unique(np.geomspace(1, L - 1, 7).astype(int))):
        ref = onp.ddm_fft(img, lags, nx, ny, 2 * L, None, subtract_mean=True)
        out = hip.ddm_fft(img, lags, nx, ny, next_fast_len(2 * L, "hip"), None, precision=precision)
        if precision == "fp64":
            for s in range(ref.shape[0]):
                assert np.allclose(out[s], ref[s], rtol=1e-9, atol=1e-12 * np.max(np.abs(ref[s]))), s
        else:
            assert np.allclose(out, ref, rtol=1e-3, atol=0)
            assert np.median(onp.relative_error(out, ref)) <= 1e-5


# series whose frames recur once, at a lag that any lane of either wave can hold
RECURRENCES = [(100, 61), (250, 131), (600, 333), (1000, 701), (2000, 1101), (2200, 1101), (4000, 2005), (4000, 2500), (4000, 3901)]


@pytest.mark.parametrize("L,lag", RECURRENCES)
def test_one_small_lag_marks_the_column(hip, L, lag):
    """D at the one lag of a recurrence is 1e-5 of the variance: far below
    what the float transforms resolve, right only if the column is marked."""
    rng = np.random.default_rng(lag)
    base = rng.normal(10000.0, 1000.0, (lag, 8, 8))
    img = np.concatenate([base, base[: L - lag]]) + rng.normal(0.0, 3.0, (L, 8, 8))
    img = np.rint(img).astype(np.uint16)
    ref = onp.ddm_diff(img, np.array([lag]), 8, 8, None)
    assert np.median(ref[0] / ref[-1]) < 1e-4
    for lags in (np.arange(1, L), np.array([lag])):
        out = hip.ddm_fft(img, lags, 8, 8, next_fast_len(2 * L, "hip"), None, precision="fp32c")
        got = out[lag - 1 if len(lags) > 1 else 0]
        assert np.allclose(got, ref[0], rtol=1e-3, atol=0)
