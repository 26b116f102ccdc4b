"""What gxc_config.xsplits and xtile still vary.

xsplits: one split, odd counts and as many splits as FFTs (fewer than a stage
each), FP32 against 64-bit sums of the handle's own spectra and 16-bit against
one split of the same spectra (up to 16 inputs the streaming X-stage, above, at
these sizes, the general one; test_gpu_xsplit_wide.py has the streaming one).  The bound is that of
test_gpu_xsplit.py, 15 * 2^-24 of sqrt(V_aa V_bb): at most 7 K-steps of 16 FFTs
(13 of 8) per split, splits summed with compensation.
xtile: FP8, and FP16 and BF16 at 33 and more inputs, where it chooses among
kernels.  A channel's sums run in the same order whatever the tile, so the
results are equal bit for bit."""
import numpy as np
import pytest

import gcorr_amd
from gcorr_amd import synth
from test_gpu_xsplit import TOL, reference, rows_of

pytestmark = pytest.mark.gpu


def correlate(nant, nchan, numffts, spectra=False, is_complex=False, **kw):
    w = synth.Workload("x", nant=nant, nchan=nchan, numffts=numffts, bw=64e6, lo=1.65e9, is_complex=is_complex, seed=5)
    rng = np.random.default_rng(nant * 1000 + numffts)
    data = [rng.integers(0, 256, w.station_bytes, dtype=np.uint8) for _ in range(nant)]
    k = gcorr_amd.FxKernel(nant, nchan, numffts, w.nbit, w.lo, w.bw, is_complex, autos=True, **kw)
    k.setInputData(data)
    k.setDelays(*synth.make_delays(w))
    k.process()
    out = k.visibilities(), k.row_counts(), k.fstage(0, numffts)[0] if spectra else None
    k.close()
    return out


SPLITS = [(1, 64, 5, 1), (2, 64, 5, 5), (8, 64, 100, 1), (8, 64, 100, 7), (8, 128, 100, 100), (9, 64, 50, 13),
          (16, 64, 100, 33), (16, 64, 97, 97)]


@pytest.mark.parametrize("nant,nchan,numffts,xsplits", SPLITS + [(24, 32, 61, 5), (32, 64, 37, 37)])
def test_fp32_splits(gpu, nant, nchan, numffts, xsplits):
    v, cnt, spec = correlate(nant, nchan, numffts, True, xsplits=xsplits)
    ref, scale = reference(spec, rows_of(nant))
    n = np.maximum(cnt, 1)[:, None, None]
    assert cnt.any() and np.max(np.abs(v * n - ref) / np.where(scale > 0, scale, 1)) < TOL


@pytest.mark.parametrize("precision", ["fp16", "bf16"])
@pytest.mark.parametrize("nant,nchan,numffts,xsplits", SPLITS)
def test_16_bit_splits(gpu, precision, nant, nchan, numffts, xsplits):
    v, cnt, _ = correlate(nant, nchan, numffts, precision=precision, xsplits=xsplits)
    one, cnt1, _ = correlate(nant, nchan, numffts, precision=precision, xsplits=1)
    assert cnt.any() and np.array_equal(cnt, cnt1)
    nbl = nant * (nant - 1) // 2
    power = np.sqrt(np.maximum(one[nbl:, [0, 3]].real * cnt1[nbl:, None, None], 0))  # [station][pol][channel]
    for r, (j, k) in enumerate(rows_of(nant)):
        for p in range(4):
            scale = power[j, p >> 1] * power[k, p & 1]
            assert np.all(np.abs(v[r, p] - one[r, p]) * cnt[r] <= TOL * scale), (r, p)


@pytest.mark.parametrize("precision,nant", [("fp8", 2), ("fp8", 8), ("fp8", 10), ("fp8", 16), ("fp8", 20),
                                            ("fp8", 32), ("fp16", 17), ("fp16", 32), ("bf16", 20)])
@pytest.mark.parametrize("xsplits", [1, 3])
def test_tiles(gpu, precision, nant, xsplits):
    base, cnt, _ = correlate(nant, 128, 70, precision=precision, xsplits=xsplits)
    ran = 0
    for xtile in (4, 8, 16, 32, 64):
        try:
            v, c, _ = correlate(nant, 128, 70, precision=precision, xsplits=xsplits, xtile=xtile)
        except gcorr_amd.GxcError:
            continue  # not a tile of this shape
        assert np.array_equal(c, cnt) and np.array_equal(v.view(np.uint32), base.view(np.uint32)), xtile
        ran += 1
    assert ran >= (1 if precision == "fp8" and nant > 16 else 2)  # FP8: one tile at 33 and more inputs
