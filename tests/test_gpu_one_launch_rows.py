"""Row kernels that only a launch of many image rows takes, on real hardware:
stacks in device memory through a plan, whose row pass is one launch (a host
stack is transformed in the pieces in which it arrives).  Rows of 1024 on both
sides of the size at which the persistent kernel takes over; mixed-radix rows
of every form (four, two or one to a wave) at the edges of their ranges, with
image heights that leave part of a wave without a row and a last frame block
that is not full."""

import numpy as np
import pytest

from fastddm_amd import next_fast_len
from oracle import oracle_np as onp

pytestmark = pytest.mark.gpu


def _run(hip, img, lags, nx, ny, precision):
    plan = hip.Plan("diff", img.dtype, img.shape, lags, nx, ny, 0, None, precision)
    d_img = hip.DeviceBuffer.from_array(img)
    d_out = hip.DeviceBuffer(plan.output_size())
    d_ws = hip.DeviceBuffer(plan.workspace_size())
    plan.execute(d_img, d_out, d_ws)
    hip.synchronize()
    out = d_out.to_array(plan.out_shape, np.float64)
    for buf in (d_img, d_out, d_ws):
        buf.free()
    plan.destroy()
    return out


def _check(got, ref, precision):
    if precision == "fp64":
        for s in range(ref.shape[0]):
            assert np.allclose(got[s], ref[s], rtol=1e-9, atol=1e-12 * np.max(np.abs(ref[s]))), s
    else:
        assert np.allclose(got, ref, rtol=1e-3, atol=0)
        assert np.median(onp.relative_error(got, ref)) <= 1e-5


@pytest.mark.parametrize("dtype", [np.uint16, np.float32])
@pytest.mark.parametrize("precision", ["fp64", "fp32c"])
@pytest.mark.parametrize("L", [9, 73])  # 768-row blocks of 4 (FP64) or 8 frames: up to 2304, from 7680 rows against 6144
def test_rows_of_1024(hip, L, precision, dtype):
    H, W = 768, 1024
    img = np.random.default_rng(L).integers(800, 1200, (L, H, W)).astype(dtype)
    lags = np.array([1, L // 2])
    _check(_run(hip, img, lags, W, H, precision), onp.ddm_diff(img, lags, W, H, None), precision)


@pytest.mark.parametrize("dtype", [np.uint8, np.uint16, np.float32])
@pytest.mark.parametrize("precision", ["fp32", "fp32c"])
def test_rows_of_1024_same_in_pieces(hip, precision, dtype):
    """Launches of any size give the same bits, whichever kernel they take."""
    L, H, W = 200, 1024, 1024  # 25600 rows in one launch
    img = np.random.default_rng(7).integers(0, 255, (L, H, W)).astype(dtype)
    lags = np.array([1, 100])
    whole = _run(hip, img, lags, W, H, precision)
    assert np.array_equal(hip.ddm_diff(img, lags, W, H, None, precision=precision), whole)


# width -> transform length: 4 rows to a wave up to 160, 2 up to 320, 1 above
@pytest.mark.parametrize("precision", ["fp64", "fp32c"])
@pytest.mark.parametrize("W", [63, 96, 150, 160, 162, 201, 315, 320, 324, 768, 784])
def test_mixed_radix_rows(hip, W, precision):
    H, L = 21, 850  # 54 (FP32) or 107 (FP64) frame blocks x 21 rows: more than one round of the chip
    img = (900 + 200 * np.random.default_rng(W).random((L, H, W))).astype(np.uint16)
    nx, ny = next_fast_len(W, "hip"), next_fast_len(H, "hip")
    lags = np.array([1, 30, 600])
    _check(_run(hip, img, lags, nx, ny, precision), onp.ddm_diff(img, lags, nx, ny, None), precision)
