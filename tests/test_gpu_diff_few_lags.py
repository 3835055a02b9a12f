"""Direct differences of few lags on real hardware, at the edges of what the
dispatch tells apart: two columns or one per wave, one per wave or per
workgroup, lags in batches of four or by themselves."""

import numpy as np
import pytest

from oracle import oracle_np as onp

pytestmark = pytest.mark.gpu

# longest series of a form and the next: two columns per wave with few lags and
# with more, one column per wave (4 byte and 8 byte samples); one per workgroup
# of 4, 8 and 16 waves
CASES = [("fp32c", (304, 305, 624, 625, 880, 881, 6000, 10200)), ("fp32", (304, 305, 432, 433, 880, 881, 6000)),
         ("fp64", (144, 145, 304, 305, 528, 529, 3000, 5100))]


@pytest.mark.parametrize("precision,L", [(p, L) for p, lengths in CASES for L in lengths])
def test_few_lags(hip, precision, L):
    img = (900 + 200 * np.random.default_rng(L).random((L, 3, 4))).astype(np.uint16)  # 9 columns
    for n in (1, 4, 5, 6, 9, 16, 17, 31, 32):
        lags = np.unique(np.linspace(1, L - 1, n).astype(int))
        assert len(lags) == n
        ref = onp.ddm_diff(img, lags, 4, 3)
        out = hip.ddm_diff(img, lags, 4, 3, None, precision=precision)
        if precision == "fp64":
            for s in range(ref.shape[0]):
                assert np.allclose(out[s], ref[s], rtol=1e-9, atol=1e-12 * np.max(np.abs(ref[s]))), s
        elif precision == "fp32c":
            assert np.allclose(out, ref, rtol=1e-3, atol=0)
            assert np.median(onp.relative_error(out, ref)) <= 1e-5
        else:
            assert np.isfinite(out).all()
            assert np.median(onp.relative_error(out, ref)) <= 1e-4
