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
