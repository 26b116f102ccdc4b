"""The workgroup sizes that gxc_config.fblock accepts, which earlier tuning runs
may have written down: the default first."""
import ctypes

import pytest

import gcorr_amd

SHORT = [256, 128, 512]
ACCEPTED = {  # FFT length: (real, complex)
    64: ([256, 128], [256, 128]), 128: (SHORT, [256, 128]), 256: (SHORT, SHORT), 512: (SHORT, SHORT),
    1024: (SHORT, SHORT), 2048: (SHORT + [64], SHORT + [64]), 4096: ([256, 512, 128], [256, 512, 128]),
    8192: ([512, 256], [512, 256]), 16384: ([512], [512]), 32768: ([1024], [1024])}


@pytest.mark.parametrize("L", sorted(ACCEPTED))
@pytest.mark.parametrize("cplx", [False, True])
def test_accepted_values(L, cplx):
    out = (ctypes.c_int * 4)()
    n = ctypes.CDLL(gcorr_amd._lib.LIB_PATH)._ZN3gxc13fstage_blocksEibPi(L, cplx, out)
    assert list(out[:n]) == ACCEPTED[L][cplx]
