"""Row pointers of a delay matrix as the C calls read them.  A one-row array that
numpy calls contiguous may have any first stride, zero among them."""
import numpy as np
import pytest

from gcorr_amd import _lib

ONE = np.arange(3.0) + 0.5


@pytest.mark.parametrize("d", [
    ONE[None], np.broadcast_to(ONE, (1, 3)), np.expand_dims(ONE, 0), np.arange(12.0).reshape(4, 3)[1:2],
    np.arange(24.0).reshape(8, 3)[::8], np.arange(96.0).reshape(32, 3)])
def test_rows_by_shape_not_stride(d):
    a = np.ascontiguousarray(d, dtype=np.float64).reshape(d.shape)
    rows = _lib.row_pointers(a)
    assert [[rows[i][j] for j in range(3)] for i in range(a.shape[0])] == a.tolist()
