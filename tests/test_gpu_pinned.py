"""Delays, station pointers, row counts and visibilities through pinned host
memory: the host copy in chunks (below one, several, a ragged last one) equals
a direct copy into pinned memory bit for bit, also from two threads; the last
values written before a call are the ones it uses."""
import ctypes
import threading

import numpy as np
import pytest
import torch

import gcorr_amd
from gcorr_amd import _lib, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nant,nchan", [(1, 32), (2, 32), (8, 512), (16, 1024)])
def test_results_equal_a_direct_copy(gpu, nant, nchan):
    numffts = 20
    w = synth.Workload("p", nant=nant, nchan=nchan, numffts=numffts, bw=64e6, lo=1.65e9, seed=3)
    rng = np.random.default_rng(nchan)
    data = [rng.integers(0, 256, w.station_bytes, dtype=np.uint8) for _ in range(nant)]
    poly, offs = synth.make_delays(w)
    k = gcorr_amd.FxKernel(nant, nchan, numffts, w.nbit, w.lo, w.bw, autos=True)
    k.setInputData([d[::-1] for d in data])
    k.setDelays(np.zeros((nant, 3)), np.full(nant, 1.0))
    k.setInputData(data)
    k.setDelays(poly, offs)
    spec, valid = k.fstage(0, numffts)  # before any process: the delays are there
    k.process()
    v = k.visibilities()
    pinned = torch.empty(v.size, dtype=torch.complex64, pin_memory=True)
    _lib.check(_lib.load().gxc_get_visibilities(k._h, ctypes.c_void_p(pinned.data_ptr()), v.size), k._h)
    assert np.array_equal(v.ravel().view(np.uint32), pinned.numpy().view(np.uint32))
    seen = [None, None]

    def read(i):
        for _ in range(5):
            seen[i] = k.visibilities()

    ts = [threading.Thread(target=read, args=(i,)) for i in range(2)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    for s in seen:
        assert np.array_equal(s.view(np.uint32), v.view(np.uint32))
    rows = [(j, m) for j in range(nant) for m in range(j + 1, nant)] + [(j, j) for j in range(nant)]
    assert list(k.row_counts()) == [int(np.sum(valid[j] & valid[m])) for j, m in rows]
    k.setDelays(poly, offs + 1.0)  # every window out of the buffer
    k.process()
    assert not k.row_counts().any() and not np.any(k.visibilities())
    k.close()
