"""The streaming X-stage at 17 and more inputs, which it serves from 256 groups of
channels on whatever the FFT count: FP32 handles against 64-bit sums of their
own spectra, FP16 and BF16 against the general X-stage on 32 of the channels.

Bound and edges as in test_gpu_xsplit.py and test_gpu_xsplits_xtiles.py: two and
four MFMA blocks with their first, last and padded inputs, FFT counts below, at
and beyond a stage and a K-step, splits, chunks; the line to the general X-stage
by size, from either side."""
import ctypes

import numpy as np
import pytest

import gcorr_amd
from gcorr_amd import synth
from test_gpu_xsplit import TOL, reference, rows_of

F32, F16 = 0, 1


def better(mode, M, nchan, nt):
    f = ctypes.CDLL(gcorr_amd._lib.LIB_PATH)._ZN3gxc13xsplit_betterEiiii
    f.restype = ctypes.c_bool
    return f(mode, M, nchan, nt)


@pytest.mark.parametrize("mode,M,nchan,nt,want", [
    (F32, 2, 32, 1, True), (F32, 16, 32, 1, True), (F16, 16, 64, 1, True), (F16, 16, 32, 100000, False),
    (F32, 18, 4096, 50, False), (F32, 18, 8192, 1, True), (F32, 32, 512, 400, False), (F32, 32, 512, 800, True),
    (F32, 20, 2048, 100, False), (F32, 20, 2048, 200, True), (F16, 32, 512, 800, False), (F16, 32, 512, 1600, True),
    (F16, 20, 8192, 20, False), (F16, 18, 16384, 1, True), (F32, 34, 2048, 20, False), (F32, 34, 4096, 1, True),
    (F32, 64, 512, 100, False), (F32, 64, 512, 200, True), (F16, 34, 32768, 1000, False), (F32, 32, 4096, 15625, True),
    (F32, 64, 1024, 6000, True), (F16, 20, 2048, 5001, True), (F16, 32, 4096, 15625, True)])
def test_choice(mode, M, nchan, nt, want):
    assert better(mode, M, nchan, nt) == want


@pytest.mark.gpu
@pytest.mark.parametrize("nant,nchan,numffts,is_complex,kw", [
    (9, 8192, 1, False, {}), (9, 8192, 17, False, {}), (10, 8192, 40, True, {"xsplits": 2}),
    (13, 8192, 5, False, {"xsplits": 5}), (16, 8192, 33, False, {"xsplits": 3}), (16, 8192, 50, False, {"chunk_ffts": 17}),
    (16, 256, 900, False, {}), (17, 4096, 7, False, {}), (24, 4096, 19, True, {"xsplits": 3}),
    (32, 4096, 16, False, {}), (32, 4096, 21, True, {"chunk_ffts": 8}), (32, 256, 300, False, {})])
def test_fp32_matches_64_bit_sums(gpu, nant, nchan, numffts, is_complex, kw):
    assert better(F32, 2 * nant, nchan, min(numffts, kw.get("chunk_ffts", numffts)))
    w = synth.Workload("x", nant=nant, nchan=nchan, numffts=numffts, bw=64e6, lo=1.65e9, is_complex=is_complex, seed=5)
    rng = np.random.default_rng(nant * 1000 + numffts)
    data = [rng.integers(0, 256, w.station_bytes, dtype=np.uint8) for _ in range(nant)]
    k = gcorr_amd.FxKernel(nant, nchan, numffts, w.nbit, w.lo, w.bw, is_complex, autos=True, **kw)
    k.setInputData(data)
    k.setDelays(*synth.make_delays(w))
    k.process()
    v, cnt = k.visibilities(), k.row_counts()
    spec, _ = k.fstage(0, numffts)
    k.close()
    some = np.concatenate([np.arange(40), nchan - 1 - np.arange(40), rng.integers(0, nchan, 40)])
    ref, scale = reference(spec[:, :, some], rows_of(nant))
    n = np.maximum(cnt, 1)[:, None, None]
    assert (cnt.any() or numffts == 1) and np.max(np.abs(v[..., some] * n - ref) / np.where(scale > 0, scale, 1)) < TOL


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["fp16", "bf16"])
@pytest.mark.parametrize("nant,nfft", [(9, 1), (9, 7), (12, 8), (13, 33), (16, 41)])
def test_16_bit_matches_general_path(gpu, precision, nant, nfft):
    rng = np.random.default_rng(nant * 100 + nfft)
    part = (rng.standard_normal((nfft, 2 * nant, 32)) + 1j * rng.standard_normal((nfft, 2 * nant, 32))).astype(np.complex64)
    spec = np.tile(part, (1, 1, 512))  # 16384 channels
    assert better(F16, 2 * nant, 16384, nfft)
    got = gcorr_amd.xengine(spec, nant, autos=True, precision=precision).astype(np.complex128)
    want = gcorr_amd.xengine(part, nant, autos=True, precision=precision).astype(np.complex128)
    _, scale = reference(part, rows_of(nant))
    got = got.reshape(got.shape[:2] + (512, 32))
    assert np.max(np.abs(got - want[:, :, None]) * nfft / scale[:, :, None]) < TOL
