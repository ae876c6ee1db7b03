"""Dims, axes and wires as C arrays: every form of list that the entry points take."""
import ctypes

import numpy as np
import pytest

from qtnh_amd import ops


@pytest.mark.parametrize("convert,ctype,top", [(ops._u64, ctypes.c_uint64, 2 ** 64 - 1),
                                               (ops._u16, ctypes.c_uint16, 2 ** 16 - 1)])
def test_lists_as_c_arrays(convert, ctype, top):
    for values in ([3, 1, 2], (0, top), np.array([5, 7]), [np.int32(4), True], [2.0, 6.0], range(4), iter([1, 2]), b"\x03"):
        values = list(values)
        keep, arg = convert(values)
        got = ctypes.cast(arg, ctypes.POINTER(ctype))
        assert [got[i] for i in range(len(values))] == [int(v) for v in values]
    keep, arg = convert([])
    assert ctypes.cast(arg, ctypes.POINTER(ctype))[0] == 0
    for refused in ([-1], [top + 1], ["x"]):
        with pytest.raises((OverflowError, ValueError)):
            convert(refused)
