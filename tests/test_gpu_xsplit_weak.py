"""The weakest spectra of the FP32 F-stage through the streaming X-stage: one
complex sample of one level per FFT window, |X| = 1 in every channel where the
f16 scale is made for |X| up to 181 L.

The bound is that of the strongest spectra (test_gpu_xsplit.py): per product
either factor rounds by 2^-24 and the dropped term is 2^-24 at most, plus the
sums: 15 * 2^-24 = 9e-7 of sqrt(V_aa V_bb).  Sizes: both sides of the line at
4096 points, the longest FFT, one, two and four MFMA blocks with padded inputs,
FFT counts below, at and beyond a K-step, several splits and chunks."""
import numpy as np
import pytest

import gcorr_amd
from gcorr_amd import synth
from test_gpu_xsplit import TOL, reference, rows_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nant,nchan,numffts,kw", [
    (2, 1024, 17, {}), (3, 2048, 20, {}), (2, 4096, 9, {}), (8, 4096, 40, {"xsplits": 2}), (3, 32768, 16, {}),
    (9, 4096, 33, {}), (16, 8192, 12, {"xsplits": 3}), (10, 32768, 5, {}), (17, 4096, 10, {}),
    (32, 4096, 23, {"chunk_ffts": 8}), (32, 32768, 2, {})])
def test_one_sample_of_one_level(gpu, nant, nchan, numffts, kw):
    w = synth.Workload("x", nant=nant, nchan=nchan, numffts=numffts, bw=64e6, lo=1.65e9, is_complex=True, seed=5)
    rng = np.random.default_rng(nant + nchan)
    data = []
    for a in range(nant):
        d = np.zeros((w.station_bytes // 4, 4), np.int8)
        at = np.arange(0, len(d), nchan) + rng.integers(nchan // 4, 3 * nchan // 4)
        d[at, 0] = 1   # polarisation A, real part
        d[at, 3] = -1  # polarisation B, imaginary part
        data.append(d.reshape(-1).view(np.uint8))
    poly, offs = synth.make_delays(w)
    k = gcorr_amd.FxKernel(nant, nchan, numffts, 8, w.lo, w.bw, True, autos=True, **kw)
    k.setInputData(data)
    k.setDelays(poly, offs)
    k.process()
    v, cnt = k.visibilities(), k.row_counts()
    spec, _ = k.fstage(0, numffts)
    k.close()
    ref, scale = reference(spec, rows_of(nant))
    n = np.maximum(cnt, 1)[:, None, None]
    assert cnt.any() and np.max(np.abs(v * n - ref) / np.where(scale > 0, scale, 1)) < TOL
