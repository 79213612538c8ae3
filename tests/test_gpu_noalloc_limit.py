"""The allocation-free entry point at the limit of its scratch: 8.34M rows take
66.7 MB of vectors, and the statistics partials of the smallest tiles (one per
256 rows) still fit beside them."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

import mlem_amd as M
from mlem_amd._native import lib

pytestmark = pytest.mark.gpu


def test_rows_just_below_the_limit():
    rows, cols = 8_340_000, 5
    rowidx = (np.arange(1, rows + 1, dtype=np.uint64) // 9)
    el = np.zeros(int(rowidx[-1]), M.ELEMENT_DTYPE)
    el["column"] = np.arange(el.size) % cols
    el["value"] = 1.0
    y = (np.arange(rows) % 3).astype(np.int32)
    with M.Csr4Matrix.from_arrays(rows, cols, rowidx, el) as A:
        assert A.launch()["fwd"] == ("dict", 8)
        x0, _ = M.initImage(A, M.calcColumnSums(A), y)
        want, ll, _ = M.mlem(A, y, x0.copy(), 2, x0_given=True, stats=True)
        hip = C.CDLL("libamdhip64.so")
        hip.hipMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t]
        hip.hipMemcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]
        hip.hipFree.argtypes = [C.c_void_p]
        yd, xd = C.c_void_p(), C.c_void_p()
        assert hip.hipMalloc(C.byref(yd), y.nbytes) == 0
        assert hip.hipMalloc(C.byref(xd), x0.nbytes) == 0
        try:
            assert hip.hipMemcpy(yd, y.ctypes.data, y.nbytes, 1) == 0
            assert hip.hipMemcpy(xd, x0.ctypes.data, x0.nbytes, 1) == 0
            l2 = np.zeros(2)
            rc = lib().mlem_reconstruct_noalloc(A.handle, yd, rows, xd, cols, 2,
                                                M.MODES["fast"], l2.ctypes.data, None)
            assert rc == 0, lib().mlem_last_error().decode()
            got = np.empty(cols, np.float32)
            assert hip.hipMemcpy(got.ctypes.data, xd, got.nbytes, 2) == 0
            assert np.array_equal(got, want) and np.array_equal(l2, ll)
        finally:
            hip.hipFree(yd)
            hip.hipFree(xd)
