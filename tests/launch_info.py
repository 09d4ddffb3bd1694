"""The launches of a buffer's last batch (myers_launch_info of the library)."""
import ctypes

import myers_amd as M

BIN, SLICE, FIRST_ROWS, WIDE_SLICE, QUEUE, LONG, SPLIT, HANDOVERS, CUT = (1 << k for k in range(9))


class Info(ctypes.Structure):
    _fields_ = [("ran", ctypes.c_uint32), ("split_words", ctypes.c_uint32), ("split_slots", ctypes.c_uint32)]


def launch_info(m, i=0):
    out = Info()
    fn = M.lib().myers_launch_info
    fn.argtypes = [ctypes.c_void_p, ctypes.c_void_p]
    M.check(fn(m.buffer(i), ctypes.byref(out)), "myers_launch_info")
    return out
