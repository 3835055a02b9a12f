"""The FP64 edge frames of compensated analyses, whose rows are read where they
lie in the stack, in every form of the row kernels, on real hardware: stacks
shorter and longer than the edge frames together, an odd number of frames; four,
two and one image row to a wave, rows of a power of two."""

import numpy as np
import pytest

from fastddm_amd import next_fast_len
from oracle import oracle_np as onp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,W", [(400, 30), (400, 150), (400, 310), (24, 150), (24, 600), (16, 1000), (24, 256), (24, 512), (16, 1024)])
@pytest.mark.parametrize("L", [3, 9, 15, 16, 17, 40])
def test_few_pair_lags(hip, L, H, W):
    img = np.random.default_rng(L + W).integers(800, 1200, (L, H, W)).astype(np.uint16)
    lags = np.arange(max(1, L - 9), L)
    nx, ny = next_fast_len(W, "hip"), next_fast_len(H, "hip")
    plan = hip.Plan("diff", img.dtype, img.shape, lags, nx, ny, 0, None, "fp32c")
    d_img = hip.DeviceBuffer.from_array(img)
    d_out = hip.DeviceBuffer(plan.output_size())
    d_ws = hip.DeviceBuffer(plan.workspace_size())
    plan.execute(d_img, d_out, d_ws)
    hip.synchronize()
    out = d_out.to_array(plan.out_shape, np.float64)
    for buf in (d_img, d_out, d_ws):
        buf.free()
    plan.destroy()
    ref = onp.ddm_diff(img, lags, nx, ny)
    for i, d in enumerate(lags):
        if L - d <= 8:  # (from FP64 spectra)
            assert np.allclose(out[i], ref[i], rtol=1e-9, atol=1e-12 * np.max(ref[i])), d
    assert np.allclose(out, ref, rtol=1e-3, atol=0)
