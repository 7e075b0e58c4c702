"""The clearing kernel (wc::fill_ranges, called by its exported C++ name) on
poisoned memory: every byte of a range is set and none beside it, for lengths
around its 16-byte words, values 0 and 0xFF, more ranges than one launch takes,
empty ranges, and ranges longer than one pass of the grid."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NAME = "_ZN2wc11fill_rangesEP12ihipStream_tSt16initializer_listINS_4FillEE"


class Fill(C.Structure):
    _fields_ = [("p", C.c_void_p), ("bytes", C.c_int64), ("value", C.c_int)]


SMALL = [1, 15, 16, 17, 31, 0, 32, 33, 4095, 4096, 4097, 125, 210, 504, 832, 3332]
LARGE = [4096 * 256 * 16 + 16 * 77 + 5, 3, (1 << 20) + 9]  # above what the grid covers at once


@pytest.mark.parametrize("lengths", [SMALL, SMALL + SMALL[::-1], [31], [0], [], LARGE],
                         ids=["16", "32", "one", "empty", "none", "large"])
def test_fill_ranges(wc, lengths):
    hip = wc.lib()
    gap = 16  # poisoned bytes between two ranges, at least
    at, end = [], 0
    for n in lengths:
        at.append(end)
        end = (end + n + gap + 15) // 16 * 16
    size = end + 64
    host = np.full(size, 0xA5, dtype=np.uint8)
    dev = C.c_void_p()
    assert hip.hipMalloc(C.byref(dev), C.c_size_t(size)) == 0
    try:
        ptr = host.ctypes.data_as(C.c_void_p)
        assert hip.hipMemcpy(dev, ptr, C.c_size_t(size), 1) == 0  # host to device
        want = host.copy()
        fills = (Fill * max(1, len(lengths)))()
        for k, (o, n) in enumerate(zip(at, lengths)):
            fills[k] = Fill(dev.value + o, n, 0xFF if k % 3 == 1 else 0)
            want[o:o + n] = 0xFF if k % 3 == 1 else 0
        fn = getattr(hip, NAME)
        fn.restype = None
        # (an initializer_list is passed as its address and length)
        fn(C.c_void_p(None), C.cast(fills, C.c_void_p), C.c_size_t(len(lengths)))
        assert hip.hipMemcpy(ptr, dev, C.c_size_t(size), 2) == 0  # waits for the fills
        bad = np.flatnonzero(host != want)
        assert bad.size == 0, (bad[:8], bad.size)
    finally:
        assert hip.hipFree(dev) == 0
