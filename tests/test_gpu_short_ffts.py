"""The shortest FFTs, whose bins leave in runs of less than 64 bytes, in every
format: 16-bit against FP32 visibilities of the same samples.  Rounding of the
spectra to u = 2^-11 (FP16) or 2^-9 (BF16) moves V_ab by at most 2 u + u^2 of
sqrt(V_aa V_bb), subnormal values and the FP32 sums by less than 1e-5 more; FP8
(e4m3, u = 2^-4, rms 32 of a range up to 448, so unclipped) likewise."""
import numpy as np
import pytest

import gcorr_amd
from gcorr_amd import synth

pytestmark = pytest.mark.gpu

U = {"fp16": 2.0 ** -11, "bf16": 2.0 ** -9, "fp8": 2.0 ** -4}


def correlate(nant, nchan, numffts, is_complex, **kw):
    w = synth.Workload("s", nant=nant, nchan=nchan, numffts=numffts, bw=16e6, lo=1.65e9, is_complex=is_complex, seed=2)
    rng = np.random.default_rng(nchan)
    if is_complex:
        data = [np.clip(np.rint(20 * rng.standard_normal(w.station_bytes)), -127, 127).astype(np.int8).view(np.uint8)
                for _ in range(nant)]
    else:
        data = [rng.integers(0, 256, w.station_bytes, dtype=np.uint8) for _ in range(nant)]
    k = gcorr_amd.FxKernel(nant, nchan, numffts, w.nbit, w.lo, w.bw, is_complex, autos=True, **kw)
    k.setInputData(data)
    k.setDelays(*synth.make_delays(w))
    k.process()
    out = k.visibilities(), k.row_counts()
    k.close()
    return out


@pytest.mark.parametrize("precision", sorted(U))
@pytest.mark.parametrize("nant,nchan,numffts,is_complex", [
    (3, 32, 700, False), (3, 64, 333, False), (5, 128, 101, False), (3, 64, 333, True), (5, 128, 101, True)])
def test_formats_agree(gpu, precision, nant, nchan, numffts, is_complex):
    ref, cnt = correlate(nant, nchan, numffts, is_complex)
    v, c = correlate(nant, nchan, numffts, is_complex, precision=precision)
    assert c.any() and np.array_equal(c, cnt)
    nbl = nant * (nant - 1) // 2
    power = np.sqrt(ref[nbl:, [0, 3]].real * cnt[nbl:, None, None])  # [station][pol][channel]
    rows = [(j, k) for j in range(nant) for k in range(j + 1, nant)] + [(j, j) for j in range(nant)]
    u = U[precision]
    for r, (j, k) in enumerate(rows):
        for p in range(4):
            bound = (2 * u + u * u + 1e-5) * power[j, p >> 1] * power[k, p & 1]
            assert np.all(np.abs(v[r, p] - ref[r, p]) * cnt[r] <= bound), (r, p)
