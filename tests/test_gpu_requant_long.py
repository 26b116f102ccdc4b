"""The 2-bit requantiser beyond the samples of one grid (2^32 work items of 8),
one buffer as both polarisations."""
import pytest
import torch

import gcorr_amd

pytestmark = pytest.mark.gpu


def test_more_samples_than_one_grid(gpu):
    n = 35_000_000_002
    if torch.cuda.mem_get_info()[0] < 180 << 30:
        pytest.skip("needs 180 GB of free GPU memory")
    x = torch.zeros(n, device="cuda")
    out = torch.empty(n // 2, dtype=torch.uint8, device="cuda")
    at = [0, 1, (1 << 34) - 1, 1 << 34, (1 << 34) + 2048, 1 << 35, n - 2, n - 1]
    level = [-2.0, -0.5, 0.5, 2.0, -2.0, 2.0, -0.5, -2.0]
    for i, v in zip(at, level):
        x[i] = v
    gcorr_amd.requantise_2bit(x.data_ptr(), x.data_ptr(), n, 1.0, out.data_ptr(),
                              stream=torch.cuda.current_stream().cuda_stream)
    code = {-2.0: 0, -0.5: 1, 0.5: 2, 2.0: 3}
    want = {}  # byte -> codes of its two samples, each twice
    for i, v in zip(at, level):
        want.setdefault(i // 2, [2, 2])[i % 2] = code[v]
    for b, (c0, c1) in want.items():
        assert int(out[b]) == c0 * 5 | c1 * 5 << 4, b
        out[b] = 0xaa
    step = 1 << 32
    assert all(bool((out[s:s + step] == 0xaa).all()) for s in range(0, out.numel(), step))
