"""Parameters written by the host reach the device with the next flush that
succeeds: one whose launch the host refuses (a grid of no work items, or no
device) leaves them pending."""
import ctypes

import gcorr_amd


class Mailbox(ctypes.Structure):  # gxc::host::Mailbox
    _fields_ = [("h", ctypes.c_void_p), ("d", ctypes.c_void_p), ("size", ctypes.c_size_t), ("dirty", ctypes.c_bool)]


def test_a_failed_flush_keeps_the_parameters_pending():
    flush = ctypes.CDLL(gcorr_amd._lib.LIB_PATH)._ZN3gxc4host7Mailbox5flushEP12ihipStream_t
    flush.argtypes = [ctypes.c_void_p, ctypes.c_void_p]
    box = Mailbox(None, None, 0, True)
    assert flush(ctypes.byref(box), None) != 0
    assert box.dirty
    box.dirty = False
    assert flush(ctypes.byref(box), None) == 0  # nothing to do


def test_pinned_memory_of_a_readout():
    """Nothing for no rows, one chunk for a copy of one, two for longer ones."""
    size = ctypes.CDLL(gcorr_amd._lib.LIB_PATH)._ZN3gxc4host7HostOut5bytesEm
    size.argtypes, size.restype = [ctypes.c_size_t], ctypes.c_size_t
    assert [size(n) for n in (0, 48 << 10, 512 << 10, (512 << 10) + 32, 1 << 30)] == \
        [0, 48 << 10, 512 << 10, 1 << 20, 1 << 20]
