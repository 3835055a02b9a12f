"""Azimuthal average at the edges of its 128-pixel tiles: planes of one pixel,
of less than, exactly and just over a tile, odd pixel counts (pairs that start
off their own alignment), columns so short that a tile holds many rows, bins
of one pixel and of whole rows, NaN in masked neighbours of used pixels."""

import numpy as np
import pytest

import fastddm_amd as fddm
from fastddm_amd.azimuthalaverage import _half_plane_counts, _k_modulus, azimuthal_average_device, bin_maps
from oracle import oracle_np as onp

pytestmark = pytest.mark.gpu

# rows, height, width (width // 2 + 1 columns), bins
CASES = [(3, 1, 1, 1), (9, 5, 1, 2), (11, 64, 2, 9), (8, 7, 4, 3), (10, 16, 14, 6), (17, 43, 4, 5), (21, 31, 64, 200),
         (5, 33, 256, 2), (30, 90, 97, 40)]


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("rows,height,width,bins", CASES)
def test_tile_edges_match_oracle(hip, rows, height, width, bins, dtype):
    rng = np.random.default_rng(rows + height)
    nxh = width // 2 + 1
    data = (1 + rng.random((rows, height, nxh))).astype(dtype)
    kx = 2 * np.pi * np.fft.fftfreq(width)[:nxh]
    ky = 2 * np.pi * np.fft.fftshift(np.fft.fftfreq(height))
    mask = rng.random((height, nxh)) > 0.2
    mask[0, 0] = True
    dist = _k_modulus(np.abs(kx), ky)
    counts = _half_plane_counts(dist.shape, width)
    bi, w, w2, edges, k = bin_maps(dist, bins, None, mask, None, counts, True)
    ref, ref_err = onp.azimuthal_average_array(data.astype(np.float64), dist, edges, w, w2, True)
    data[:, ~mask] = np.nan
    d = hip.DeviceBuffer.from_array(data)
    tau = np.arange(1, rows - 1, dtype=np.float64)
    a = azimuthal_average_device(d, data.shape, np.abs(kx), ky, tau, width, dtype, bins=bins, mask=mask)
    assert np.allclose(a._data, ref, rtol=1e-12, atol=0, equal_nan=True)
    assert np.allclose(a._err, ref_err, rtol=1e-9, atol=1e-15, equal_nan=True)
    d.free()
