"""Host-buffer calls whose row and column passes run beside the copy of the
later frames against one launch per pass over the same stack in device
memory: bit for bit, where pieces (4 MiB, or an eighth of the stack) end
inside a frame and inside a frame block, with a piece smaller than a frame
block, and with one piece only."""

import numpy as np
import pytest

from fastddm_amd import next_fast_len
from fastddm_amd.window import blackman_harris

pytestmark = pytest.mark.gpu

CASES = [
    # mode, precision, pixel type, (L, H, W)
    ("fft", "fp32c", np.uint8, (257, 256, 256)),  # one frame left over
    ("fft", "fp32c", np.uint16, (311, 147, 201)),  # frames and blocks straddle pieces, mixed-radix and odd sides
    ("fft", "fp64", np.float64, (70, 200, 256)),
    ("diff", "fp32c", np.uint16, (130, 256, 320)),
    ("fft", "fp32", np.float32, (9, 1500, 1200)),  # a frame block is larger than a piece
    ("diff", "fp64", np.uint8, (23, 41, 37)),  # one piece
]


@pytest.mark.parametrize("mode,precision,dtype,shape", CASES)
def test_overlapped_copy_equals_device_plan(hip, mode, precision, dtype, shape):
    L, H, W = shape
    rng = np.random.default_rng(L + H)
    img = rng.integers(0, 255, shape).astype(dtype)
    win = blackman_harris((H, W)) if mode == "fft" else None
    lags = np.unique(np.geomspace(1, L - 1, 40).astype(int))
    nx, ny = next_fast_len(W, "hip"), next_fast_len(H, "hip")
    nt = next_fast_len(2 * L, "hip") if mode == "fft" else 0
    if mode == "fft":
        got = hip.ddm_fft(img, lags, nx, ny, nt, win, precision=precision)
    else:
        got = hip.ddm_diff(img, lags, nx, ny, win, precision=precision)
    assert hip.last_call_chunks()["mode"] == 0
    plan = hip.Plan(mode, img.dtype, shape, lags, nx, ny, nt, win, precision)
    d_img = hip.DeviceBuffer.from_array(img)
    d_out = hip.DeviceBuffer(plan.output_size())
    d_ws = hip.DeviceBuffer(plan.workspace_size())
    plan.execute(d_img, d_out, d_ws)
    hip.synchronize()
    ref = d_out.to_array(got.shape, got.dtype)
    plan.destroy()
    assert np.array_equal(got, ref)
