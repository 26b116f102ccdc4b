"""What the autotuners time: FP32 has one F-stage per length, reduced precision
two where the matrix-core F-stage covers it."""
import numpy as np
import pytest

import gcorr_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,fstages", [("fp32", 1), ("fp16", 2)])
@pytest.mark.parametrize("nchan", [512, 1024, 2048])
def test_handle(gpu, precision, fstages, nchan):
    k = gcorr_amd.FxKernel(2, nchan, 8, 2, 1.65e9, 64e6, precision=precision)
    k.setInputData([np.zeros(k.station_bytes, np.uint8)] * 2)
    k.setDelays(np.zeros((2, 3)), np.zeros(2))
    t = k.autotune()
    k.close()
    # eager as created, F-stages, one tile and split count (8 FFTs), eager and graph as chosen
    assert t["candidates"] == 1 + (fstages if nchan >= 1024 else 1) + 1 + 2
    assert precision != "fp32" or t["fblock"] == 256


@pytest.mark.parametrize("precision,fstages", [("fp32", 1), ("fp16", 2)])
def test_batch(gpu, precision, fstages):
    b = gcorr_amd.Batch(2, [(512, 8, 1.65e9, 16e6), (2048, 8, 1.65e9, 16e6)], precision=precision)
    for s in range(2):
        b.set_input(s, [np.zeros(gcorr_amd.station_bytes(2, b.subbands[s][0], 8), np.uint8)] * 2)
        b.set_delays(s, np.zeros((2, 3)), np.zeros(2))
    t = b.autotune()
    b.close()
    assert t["candidates"] == 1 + 4 * fstages + 1  # as created, X unit counts, graph
    assert precision != "fp32" or t["fblock"] == 256
