"""FFT splits of the streaming X-stage by shape: a workgroup per CU for long
subintegrations, fewer for short ones (whole passes timed at every split)."""
import ctypes

import pytest

import gcorr_amd

F32, F16 = 0, 1


def splits(mode, M, nchan, nt):
    return ctypes.CDLL(gcorr_amd._lib.LIB_PATH)._ZN3gxc20xsplit_choose_splitsEiiii(mode, M, nchan, nt)


@pytest.mark.parametrize("mode,M,nchan,nt,want", [
    (F32, 12, 1024, 62500, 8), (F32, 32, 4096, 15625, 2), (F32, 64, 1024, 6000, 4), (F32, 8, 128, 12500, 64),
    (F16, 20, 2048, 5001, 8), (F16, 16, 32768, 1000, 1), (F32, 60, 256, 64, 4), (F32, 60, 256, 500, 8),
    (F32, 32, 128, 500, 12), (F16, 32, 128, 500, 12), (F32, 6, 32, 5000, 84), (F32, 16, 256, 2000, 32),
    (F32, 24, 4096, 50, 1), (F32, 32, 2048, 60, 1), (F32, 2, 32, 1, 1), (F32, 2, 32, 17, 1), (F32, 6, 256, 64, 4),
    (F16, 12, 1024, 200, 4), (F16, 32, 512, 200, 4), (F16, 16, 512, 200, 8), (F16, 24, 4096, 50, 1)])
def test_choice(mode, M, nchan, nt, want):
    assert splits(mode, M, nchan, nt) == want


@pytest.mark.parametrize("mode,nchans", [(F32, [32, 128, 4096, 16384]), (F16, [64, 1024, 32768])])
def test_bounds(mode, nchans):
    for M in range(2, 66, 2):
        for nchan in nchans:
            for nt in (1, 15, 16, 31, 33, 64, 100, 1000, 60000):
                s = splits(mode, M, nchan, nt)
                assert 1 <= s <= min(256, max(1, nt)), (M, nchan, nt)
                assert s <= 2 or s % 4 == 0
