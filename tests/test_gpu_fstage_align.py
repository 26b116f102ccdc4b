"""F-stage spectra at every alignment of the packed window.

The kernels read a window's samples as aligned 32-bit words (2048 points and
more, 2-bit) or as bytes and words at the sample's own address, in items of a
workgroup that share a wave below 1024 points.  Nine stations whose net delays
are 0..8 samples read their windows at every offset modulo 8 samples (every
byte of a 32-bit word at both nibble parities), with an item count that leaves
the last workgroup part empty, against the oracle within the FP32 bound of
the other F-stage tests (2e-5 of the spectrum's RMS: phases and transform both
round to a few 1e-7).
"""
import numpy as np
import pytest

import gcorr_amd
from gcorr_amd import synth
from oracle import fxref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nchan,is_complex", [(32, False), (128, False), (256, False), (512, False), (1024, False),
                                              (2048, False), (4096, False), (8192, False), (128, True), (512, True),
                                              (2048, True), (8192, True)])
def test_every_window_alignment(gpu, nchan, is_complex):
    nant, numffts = 9, 5
    w = synth.Workload("a", nant=nant, nchan=nchan, numffts=numffts, bw=64e6, lo=1.65e9 + 0.25, is_complex=is_complex,
                       seed=71)
    rng = np.random.default_rng(nchan + is_complex)
    data = [rng.integers(0, 256, w.station_bytes, dtype=np.uint8) for _ in range(nant)]
    poly, _ = synth.make_delays(w)
    offs = poly[:, 2] - np.arange(nant) * w.sampletime
    k = gcorr_amd.FxKernel(nant, nchan, numffts, w.nbit, w.lo, w.bw, is_complex)
    k.setInputData(data)
    k.setDelays(poly, offs)
    spec, valid = k.fstage(0, numffts)
    k.close()
    cfg = fxref.make_config(nant, nchan, numffts, w.lo, w.bw, nbit=w.nbit, is_complex=is_complex)
    seen = 0
    for a in range(nant):
        for t in range(numffts):
            ref, ok = fxref.station_spectrum(cfg, data[a], poly[a], offs[a], t)
            assert bool(valid[a, t]) == ok, (a, t)
            got = spec[t, 2 * a:2 * a + 2]
            if not ok:
                assert not np.any(got)
                continue
            seen += 1
            rms = np.sqrt(np.mean(np.abs(ref) ** 2))
            assert np.max(np.abs(got - ref)) / rms < 2e-5, (a, t)
    assert seen >= nant * (numffts - 2)
