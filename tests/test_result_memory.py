"""The arrays of a SolveResult share the native result's memory: it is freed
once, when the last of them (or of their views) is gone, and not before."""
import ctypes as C
import gc

import numpy as np

import warchest_wave as ww


def test_native_result_lives_as_long_as_its_arrays(monkeypatch):
    freed = []

    class Library:
        @staticmethod
        def wc_result_free(ptr):
            freed.append(ptr)

    monkeypatch.setattr(ww, "_lib", Library())
    memory = (C.c_float * 6)(*range(6))
    held = ww._ResultMemory(7)
    strategy = held.array(C.cast(memory, C.POINTER(C.c_float)), 6, "<f4")
    carries = held.array(C.cast(memory, C.POINTER(C.c_uint16)), 12, "<f2").reshape(3, 4)
    empty = held.array(None, 0, "<f4")
    assert empty.size == 0 and strategy.dtype == np.float32 and carries.dtype == np.float16
    np.testing.assert_array_equal(strategy, np.arange(6, dtype=np.float32))
    assert strategy.flags.writeable
    del held, strategy
    gc.collect()
    assert freed == []
    part = carries[1:, 2]
    del carries
    gc.collect()
    assert freed == []
    del part
    gc.collect()
    assert freed == [7]
