"""Subbands of one FFT length share an F-stage launch, and short ones of several
lengths as well.  The batch must give what a
batch of each subband alone gives, whose F-stage is a launch with one subband's
parameters, bit for bit: FFT counts below 64 leave one X split either way.

Sizes: two and three subbands of every length in mixed order, odd FFT and
station counts (units of several FFTs partly empty at the seams), one subband
with every FFT out of its buffer, one and several chunks, overlap."""
import numpy as np
import pytest

import gcorr_amd
from gcorr_amd import synth

pytestmark = pytest.mark.gpu

BANDS = [(128, 33), (1024, 5), (256, 17), (128, 63), (4096, 9), (512, 40), (2048, 7), (256, 3), (512, 61),
         (1024, 60), (4096, 3), (128, 1), (2048, 13), (512, 1), (1024, 2)]


def inputs(nant, bands):
    out = []
    for i, (nchan, numffts) in enumerate(bands):
        w = synth.Workload("g", nant=nant, nchan=nchan, numffts=numffts, bw=32e6, lo=1.65e9 + 1e6 * i, seed=i)
        rng = np.random.default_rng(100 * nant + i)
        poly, offs = synth.make_delays(w)
        if i == 3:
            offs = offs + 1.0
        data = [rng.integers(0, 256, w.station_bytes, dtype=np.uint8) for _ in range(nant)]
        out.append(((nchan, numffts, w.lo, w.bw), data, poly, offs))
    return out


def correlate(nant, subs, **kw):
    b = gcorr_amd.Batch(nant, [s[0] for s in subs], autos=True, **kw)
    for i, (_, data, poly, offs) in enumerate(subs):
        b.set_input(i, data)
        b.set_delays(i, poly, offs)
    b.process()
    b.process()  # the second one replays the graph
    out = [(b.visibilities(i), b.row_counts(i)) for i in range(len(subs))]
    b.close()
    return out


@pytest.mark.parametrize("precision", ["fp32", "fp16", "bf16", "fp8"])
@pytest.mark.parametrize("nant,kw", [(3, {}), (5, {}), (3, {"graph": False}), (18, {})])
def test_equals_each_subband_alone(gpu, precision, nant, kw):
    subs = inputs(nant, BANDS)
    got = correlate(nant, subs, precision=precision, **kw)
    for i, s in enumerate(subs):
        (v, c), = correlate(nant, [s], precision=precision, **kw)
        assert np.array_equal(got[i][1], c) and (c.any() or i == 3)
        assert np.array_equal(got[i][0].view(np.uint32), v.view(np.uint32)), s[0]


@pytest.mark.parametrize("kw", [{"chunks": 3}, {"chunks": 4, "overlap": True}, {"fstage_mfma": 1, "precision": "fp16"},
                                {"fstage_mfma": 1}, {"fstage_mfma": 2}])
def test_chunks_and_kernels(gpu, kw):
    subs = inputs(3, [b for b in BANDS if b[1] >= 5])
    got = correlate(3, subs, **kw)
    for i, s in enumerate(subs):
        (v, c), = correlate(3, [s], **kw)
        assert np.array_equal(got[i][1], c)
        assert np.array_equal(got[i][0].view(np.uint32), v.view(np.uint32)), s[0]


@pytest.mark.parametrize("precision", ["fp32", "fp16", "fp8"])
@pytest.mark.parametrize("nchan", [128, 256, 512, 1024, 2048, 4096])
def test_one_length(gpu, precision, nchan):
    """Subbands of one length only: the launch of that length."""
    subs = inputs(5, [(nchan, 7), (nchan, 1), (nchan, 45), (nchan, 2)])
    got = correlate(5, subs, precision=precision)
    for i, s in enumerate(subs):
        (v, c), = correlate(5, [s], precision=precision)
        assert np.array_equal(got[i][1], c)
        assert np.array_equal(got[i][0].view(np.uint32), v.view(np.uint32)), s[0]


@pytest.mark.parametrize("nfft,kw", [(25, {}), (25, {"precision": "bf16"}), (26, {}), (26, {"graph": False})])
def test_launch_limit(gpu, nfft, kw):
    """Two lengths on both sides of 1500 units: 17 stations x (25 or 26 FFTs of
    2048 points and 63 of 1024)."""
    subs = inputs(17, [(1024, nfft), (512, 63)])
    got = correlate(17, subs, **kw)
    for i, s in enumerate(subs):
        (v, c), = correlate(17, [s], **kw)
        assert np.array_equal(got[i][1], c)
        assert np.array_equal(got[i][0].view(np.uint32), v.view(np.uint32)), s[0]
