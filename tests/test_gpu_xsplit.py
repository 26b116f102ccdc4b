"""The streaming X-stage: FP32 handles (f16 hi + lo products) against 64-bit sums
of the same spectra and against the general X-stage (FP32 products); FP16 and
BF16 against the general X-stage, which takes the channel counts that the
streaming one does not.

V_ab / sqrt(V_aa V_bb) must agree to 1e-6 of 64-bit sums: per product, hi + lo
of either factor rounds by 2^-24 and the dropped term is 2^-24 at most; a sum
of at most 7 K-steps of 16 FFTs adds 7 roundings of 2^-24, and the split,
normalisation and output another few: 15 * 2^-24 = 9e-7.

Sizes: every number of MFMA blocks with its first, last and padded inputs (2,
16, 18, 32, 34, 64), one and several channel groups, FFT counts below, at and
beyond a stage and a K-step, splits with no FFT left over, chunks.
"""
import numpy as np
import pytest

import gcorr_amd
from gcorr_amd import synth

pytestmark = pytest.mark.gpu

TOL = 1e-6


def reference(spec, rows):
    x = spec.astype(np.complex128)  # [t][input][chan]
    v = np.einsum("tac,tbc->abc", x, x.conj())
    out = np.empty((len(rows), 4, spec.shape[2]), np.complex128)
    for r, (j, k) in enumerate(rows):
        for p in range(4):
            out[r, p] = v[2 * j + (p >> 1), 2 * k + (p & 1)]
    power = np.sqrt(np.einsum("tac,tac->ac", x, x.conj()).real)
    scale = np.empty(out.shape)
    for r, (j, k) in enumerate(rows):
        for p in range(4):
            scale[r, p] = power[2 * j + (p >> 1)] * power[2 * k + (p & 1)]
    return out, scale


def rows_of(nant):
    return [(j, k) for j in range(nant) for k in range(j + 1, nant)] + [(j, j) for j in range(nant)]


@pytest.mark.parametrize("nant,nchan,numffts,is_complex,kw", [
    (1, 32, 1, False, {}), (2, 32, 7, False, {}), (3, 64, 16, False, {}), (6, 128, 33, False, {"xsplits": 2}),
    (8, 64, 100, False, {"xsplits": 3}), (8, 32, 5, False, {"xsplits": 5}), (9, 32, 17, False, {}),
    (10, 64, 40, True, {"xsplits": 2}), (16, 64, 100, False, {}), (16, 256, 97, False, {"chunk_ffts": 31}),
    (17, 32, 19, False, {}), (24, 64, 50, True, {"xsplits": 3}), (32, 32, 100, False, {}),
    (32, 64, 37, True, {"chunk_ffts": 10})])
def test_matches_64_bit_sums_and_general_path(gpu, nant, nchan, numffts, is_complex, kw):
    w = synth.Workload("x", nant=nant, nchan=nchan, numffts=numffts, bw=64e6, lo=1.65e9, is_complex=is_complex, seed=5)
    rng = np.random.default_rng(nant * 1000 + numffts)
    data = [rng.integers(0, 256, w.station_bytes, dtype=np.uint8) for _ in range(nant)]
    poly, offs = synth.make_delays(w)
    k = gcorr_amd.FxKernel(nant, nchan, numffts, w.nbit, w.lo, w.bw, is_complex, autos=True, **kw)
    k.setInputData(data)
    k.setDelays(poly, offs)
    k.process()
    v, cnt = k.visibilities(), k.row_counts()
    spec, valid = k.fstage(0, numffts)
    k.close()
    rows = rows_of(nant)
    ref, scale = reference(spec, rows)
    assert all(cnt[r] == np.sum(valid[j] & valid[kk]) for r, (j, kk) in enumerate(rows))
    n = np.maximum(cnt, 1)[:, None, None]
    scale = np.where(scale > 0, scale, 1)
    assert np.max(np.abs(v * n - ref) / scale) < TOL
    general = gcorr_amd.xengine(spec, nant, autos=True)  # divided by numffts
    assert np.max(np.abs(v * n - general.astype(np.complex128) * numffts) / scale) < 2 * TOL


@pytest.mark.parametrize("nchan,is_complex", [(32, False), (4096, False), (16384, False), (64, True), (32768, True)])
def test_largest_spectra(gpu, nchan, is_complex):
    """Full-scale constant samples: |X[0]| is the bound that the scale is made for."""
    nant, numffts = 2, 3
    w = synth.Workload("x", nant=nant, nchan=nchan, numffts=numffts, bw=64e6, lo=1.65e9, is_complex=is_complex, seed=1)
    data = [np.full(w.station_bytes, 0x80 if is_complex else 0xff, np.uint8)] * nant
    k = gcorr_amd.FxKernel(nant, nchan, numffts, w.nbit, w.lo, w.bw, is_complex, autos=True)
    k.setInputData(data)
    k.setDelays(np.zeros((nant, 3)), np.zeros(nant))
    k.process()
    v = k.visibilities()
    k.close()
    L = nchan if is_complex else 2 * nchan
    want = (L * 128.0) ** 2 * 2 if is_complex else (L * float(np.float32(3.3359))) ** 2
    np.testing.assert_allclose(v[:, :, 0].real, want, rtol=2e-6)
    assert np.all(np.isfinite(v.view(np.float32)))


@pytest.mark.parametrize("precision", ["fp16", "bf16"])
@pytest.mark.parametrize("nant,nfft", [(1, 1), (3, 7), (8, 16), (8, 33), (9, 100), (13, 8), (16, 41), (16, 100)])
def test_16_bit_matches_general_path(gpu, precision, nant, nfft):
    """The first 32 of 64 channels (streaming) and the 32 alone (general)."""
    rng = np.random.default_rng(nant * 100 + nfft)
    spec = (rng.standard_normal((nfft, 2 * nant, 64)) + 1j * rng.standard_normal((nfft, 2 * nant, 64))).astype(np.complex64)
    got = gcorr_amd.xengine(spec, nant, autos=True, precision=precision)[..., :32].astype(np.complex128)
    want = gcorr_amd.xengine(spec[..., :32], nant, autos=True, precision=precision).astype(np.complex128)
    _, scale = reference(spec[..., :32], rows_of(nant))
    assert np.max(np.abs(got - want) * nfft / scale) < TOL
