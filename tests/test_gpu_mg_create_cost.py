"""Making a handle: a small mixed-precision one has some 170 constant arrays, and
takes less time than allocating and filling 100 of them one by one would."""
import ctypes
import time

import numpy as np
import pytest

import saras_amd as S

pytestmark = pytest.mark.gpu


def fastest(f, count=20):
    best = float("inf")
    for _ in range(count):
        t = time.perf_counter()
        keep = f()
        best = min(best, time.perf_counter() - t)
        del keep
    return best


def test_small_handle():
    hip = ctypes.CDLL("libamdhip64.so")   # the runtime that the library has loaded
    hip.hipMalloc.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_size_t]
    hip.hipMemcpy.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_int]
    hip.hipFree.argtypes = [ctypes.c_void_p]
    g, p = S.grid_desc((32, 32, 32)), S.mg_params(solve_flag=1, precision=S.PREC_MIXED)
    S.Multigrid(g, p)   # the library's own start
    src = np.zeros(32)

    class Pairs:
        def __init__(self):
            self.at = []
            for _ in range(100):
                q = ctypes.c_void_p()
                assert hip.hipMalloc(ctypes.byref(q), src.nbytes) == 0
                self.at.append(q)
                assert hip.hipMemcpy(q, src.ctypes.data, src.nbytes, 1) == 0   # host to device

        def __del__(self):
            for q in self.at:
                hip.hipFree(q)

    pairs, handle = fastest(Pairs), fastest(lambda: S.Multigrid(g, p))
    print(f"100 pairs {pairs * 1e3:.3f} ms, handle {handle * 1e3:.3f} ms")
    assert handle < pairs
