"""Lag S/N at the edges of the in-LDS form (one channel pair, fewer butterflies
than threads, the longest) and of the form beyond it, against the oracle: the
peak where rounding does not decide it, the S/N to 1e-4 as in the other lag
tests (|lag| in FP32 of a transform of log2 n roundings; 1e-3 at 2 and 4 lags,
whose deviation is a difference of a few close values)."""
import numpy as np
import pytest

import gcorr_amd
from oracle.lagref import lag_snr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 4, 256, 512, 8192, 16384])
def test_forms_match_the_oracle(gpu, n):
    rng = np.random.default_rng(n)
    v = (rng.standard_normal((9, n)) + 1j * rng.standard_normal((9, n))).astype(np.complex64)
    c = np.arange(n)
    v += 3 * np.exp(-2j * np.pi * c * np.arange(9)[:, None] * (n // 2 + 1) / n)
    v[8] = 0  # no signal at all: not a number, as numpy
    snr, peak = gcorr_amd.lag_snr(v)
    with np.errstate(all="ignore"):
        want, wpeak = lag_snr(v)
    lags = np.sort(np.abs(np.fft.ifft(v.astype(np.complex128), axis=-1)), axis=-1)
    clear = lags[:, -1] > lags[:, -2] * (1 + 1e-3)
    np.testing.assert_array_equal(peak[clear], wpeak[clear])
    ok = np.isfinite(want)
    np.testing.assert_allclose(snr[ok], want[ok], rtol=1e-4 if n > 4 else 1e-3)
    assert np.isnan(snr[8])
