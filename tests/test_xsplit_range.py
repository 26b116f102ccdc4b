"""Channel counts of the streaming X-stage.  Its rows are at 24-bit products of
a row number and a row's bytes, so rows of 2^24 bytes and more (2^22 channels
of 16 bits) take the general X-stage."""
import ctypes

import numpy as np
import pytest

import gcorr_amd

F32, F16, BF16, FP8 = range(4)
WIDE = 1 << 22  # channels of a 16-bit row of 2^24 bytes


@pytest.mark.parametrize("mode,M,nchan,want", [
    (F16, 2, 64, 64), (F16, 32, 32768, 64), (BF16, 32, WIDE - 64, 64), (F16, 2, WIDE - 64, 64),
    (F16, 2, WIDE, 0), (BF16, 32, WIDE, 0), (F16, 16, WIDE + 64, 0), (BF16, 2, 64 * WIDE, 0),
    (F32, 32, WIDE // 2 - 32, 32), (F32, 32, WIDE // 2, 0), (F32, 64, WIDE // 2, 0),
    (F16, 2, 96, 0), (F16, 34, 64, 0), (FP8, 2, 64, 0)])
def test_rows_of_24_bits_only(mode, M, nchan, want):
    channels = ctypes.CDLL(gcorr_amd._lib.LIB_PATH)._ZN3gxc15xsplit_channelsEiii
    assert channels(mode, M, nchan) == want


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["fp16", "bf16"])
@pytest.mark.parametrize("nchan", [WIDE - 64, WIDE, WIDE + 64])
def test_widest_rows(gpu, precision, nchan):
    """Small whole numbers: products and sums of two FFTs are exact."""
    rng = np.random.default_rng(nchan)
    x = rng.integers(-8, 9, (2, 2, nchan, 2)).astype(np.float32).view(np.complex64)[..., 0]
    got = gcorr_amd.xengine(x, 1, autos=True, precision=precision)[0]
    for p in range(4):
        assert np.array_equal(got[p], (x[:, p >> 1] * x[:, p & 1].conj()).sum(0) / 2)
