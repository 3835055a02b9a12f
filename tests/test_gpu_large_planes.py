"""Work beyond what one launch holds (2^32 threads), on real hardware: planes
of more columns, averages of more rows and bins.  Every output is written,
with its value."""

import numpy as np
import pytest

from fastddm_amd import next_fast_len
from fastddm_amd.azimuthalaverage import _reduce

pytestmark = pytest.mark.gpu


def test_diff_columns_beyond_one_launch(hip):
    L, H, W, lag = 897, 8, 8, 448  # a column per workgroup of 256 threads
    nx, ny = 8192, 4116
    nxh = nx // 2 + 1
    assert nxh * ny > 2**24 and next_fast_len(ny, "hip") == ny
    rng = np.random.default_rng(3)
    img = rng.standard_normal((L, H, W)).astype(np.float32)
    plan = hip.Plan("diff", img.dtype, img.shape, [lag], nx, ny, 0, None, "fp32", np.float32)
    need = plan.input_size() + plan.output_size() + plan.workspace_size()
    d_img = hip.DeviceBuffer.from_array(img)
    d_out = hip.DeviceBuffer.from_array(np.full(plan.out_shape, np.nan, np.float32))
    d_ws = hip.DeviceBuffer(plan.workspace_size())
    plan.execute(d_img, d_out, d_ws)
    hip.synchronize()
    out = d_out.to_array(plan.out_shape, np.float32)
    for buf in (d_img, d_out, d_ws):
        buf.free()
    plan.destroy()
    assert np.isfinite(out).all()

    # sampled columns, the first and last and those at the end of a launch among them
    flat = np.concatenate([rng.integers(0, nxh * ny, 500), [0, nxh * ny - 1], np.arange(2**24 - 16, 2**24 + 16)])
    row, kx = flat // nxh, flat % nxh
    ky = (row - ny // 2) % ny
    y, x = np.arange(H), np.arange(W)
    F = np.empty((L, len(flat)), np.complex128)
    for i in range(len(flat)):
        e = np.exp(-2j * np.pi * (ky[i] * y[:, None] / ny + kx[i] * x[None, :] / nx))
        F[:, i] = (img * e).sum(axis=(1, 2))
    F /= np.sqrt(nx * ny)
    D = np.mean(np.abs(F[lag:] - F[:-lag]) ** 2, axis=0)
    assert np.allclose(out[0, row, kx], D, rtol=1e-4, atol=0)

    # the same in pieces, whose columns are stored by their place in the piece
    hip.set_memory_budget(need - 1)
    try:
        pieces = hip.ddm_diff(img, [lag], nx, ny, None, precision="fp32", out_dtype=np.float32)
        assert hip.last_call_chunks()["mode"] == 1
    finally:
        hip.set_memory_budget(0)
    assert np.array_equal(pieces, out)


def test_azimuthal_outputs_beyond_one_launch(hip):
    # 2^29 averages and a few more, eight threads each
    rows, nq, nbins = 2**19 + 9, 64, 1024
    data = np.random.default_rng(5).standard_normal((rows, nq)).astype(np.float32)
    d_data = hip.DeviceBuffer.from_array(data)
    bins = np.arange(nq, dtype=np.int32)  # a pixel to a bin: each average is that pixel
    avg, _ = _reduce(d_data.ptr, True, rows, 1, nq, bins, np.ones(nq), None, nbins, False)
    d_data.free()
    hip.release_cache()
    assert np.array_equal(avg[:nq], data.T.astype(np.float64))
    assert np.isnan(avg[nq:]).all()
