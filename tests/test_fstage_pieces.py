"""F-stage launches stay below the 2^32 work items of a grid: the kernels run up
to L/8 threads per (station, FFT), and longer subintegrations go in pieces."""
import ctypes

import numpy as np
import pytest
import torch

import gcorr_amd


@pytest.mark.parametrize("L", [64, 512, 1024, 2048, 32768])
@pytest.mark.parametrize("nant", [1, 3, 32])
def test_pieces_fit_a_grid(L, nant):
    most = ctypes.CDLL(gcorr_amd._lib.LIB_PATH)._ZN3gxc16fstage_most_fftsEii(L, nant)
    assert most >= 1 and nant * most * (L // 8) + 1024 < 2 ** 32
    # no more pieces than needed: one up to half of the limit
    assert nant * most * (L // 8) > 2 ** 31 or most == 2 ** 31 - 1


@pytest.mark.gpu
def test_one_chunk_beyond_a_grid(gpu):
    """32 stations of the same samples x 64 points, FP8, 16.9 million FFTs in one
    chunk (69 GB of spectra) against the default chunks of 32 GiB."""
    if torch.cuda.mem_get_info()[0] < 150 << 30:
        pytest.skip("needs 150 GB of free GPU memory")
    nant, nchan, numffts = 32, 32, 16_900_000
    out = []
    for chunk in (numffts, 0):
        k = gcorr_amd.FxKernel(nant, nchan, numffts, 2, 1.65e9, 64e6, precision="fp8", autos=True, chunk_ffts=chunk)
        g = torch.Generator(device="cuda").manual_seed(7)
        buf = torch.randint(0, 256, (k.station_bytes,), dtype=torch.uint8, device="cuda", generator=g)
        k.setInputDevice([buf.data_ptr()] * nant, keepalive=buf)
        k.setDelays(np.zeros((nant, 3)), np.zeros(nant))
        k.process()
        out.append((k.visibilities(), k.row_counts()))
        k.close()
        del buf
        torch.cuda.empty_cache()
    (v, n), (ref, nref) = out
    assert np.all(n == numffts) and np.array_equal(n, nref)
    power = np.abs(ref[0, 0]).mean()
    assert power > 0 and np.max(np.abs(v - ref)) < 1e-4 * power
