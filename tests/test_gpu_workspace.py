"""Device memory of compensated plans for tall images (two frames to a block,
where the FP64 edge frames weigh most), on real hardware: analyses that fill
the static workspace or the memory budget."""

import numpy as np
import pytest

from oracle import oracle_np as onp

pytestmark = pytest.mark.gpu


def _check(out, ref):
    assert np.allclose(out, ref, rtol=1e-3, atol=0)
    assert np.median(onp.relative_error(out, ref)) <= 1e-5


def test_tall_stack_in_the_static_workspace(hip):
    L, H, W = 4, 4096, 512
    img = np.random.default_rng(1).integers(100, 250, (L, H, W)).astype(np.uint8)
    lags = np.array([1, 3])
    plan = hip.Plan("diff", img.dtype, img.shape, lags, W, H, 0, None, "fp32c")
    assert plan.workspace_size() <= hip.Plan.STATIC_SCRATCH_BYTES
    d_img = hip.DeviceBuffer.from_array(img)
    d_out = hip.DeviceBuffer(plan.output_size())
    plan.execute_static(d_img, d_out)
    hip.synchronize()
    out = d_out.to_array(plan.out_shape, np.float64)
    plan.destroy()
    _check(out, onp.ddm_diff(img, lags, W, H))


@pytest.mark.parametrize("mode", ["diff", "fft"])
def test_tall_stack_within_a_small_budget(hip, mode):
    L, H, W = 40, 4096, 64
    img = np.random.default_rng(2).integers(100, 250, (L, H, W)).astype(np.uint8)
    lags = np.array([1, 7, 36])  # the last has 4 pairs
    # 19 frames (the first, 16 edge frames, a block of 2); for every q the FP64
    # rows and spectra of 16 + 1 + 16 + 1 frames and the FP32 ones of 6, in
    # bytes; and 1 % for the small pieces
    pixels, q = H * W, H * (W // 2 + 1)
    hip.set_memory_budget(int(1.01 * (19 * pixels + (34 * 16 + 6 * 8) * q)))
    try:
        if mode == "diff":
            out = hip.ddm_diff(img, lags, W, H, None, precision="fp32c")
        else:
            out = hip.ddm_fft(img, lags, W, H, 2 * L, None, precision="fp32c")
        assert hip.last_call_chunks()["mode"] == 2
    finally:
        hip.set_memory_budget(0)
    _check(out, onp.ddm_diff(img, lags, W, H))
