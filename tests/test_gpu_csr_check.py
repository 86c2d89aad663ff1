"""The input check of two CSR matrices (gpk_csr_check) where a chunk of 2,048
entries spans many empty rows: its flags against those computed row by row, with
runs of empty rows around the 8,192 that a chunk marks and a fault at a row's
start, end or chunk edge."""
import ctypes as C

import numpy as np
import pytest

import gp_ffi

pytestmark = pytest.mark.gpu


class Side(C.Structure):
    _fields_ = [("ptr", C.c_void_p), ("idx", C.c_void_p), ("rows", C.c_int32), ("cols", C.c_int32),
                ("nnz", C.c_int32), ("pad", C.c_int32), ("chunk_row", C.c_void_p), ("flags", C.c_void_p)]


def flags_of(sides):
    L = gp_ffi.lib()
    L.gpk_csr_check.argtypes = [Side, Side, C.c_void_p]
    L.gpk_csr_check_chunks.argtypes = [C.c_int32]
    flags = gp_ffi.DeviceArray(np.zeros(4 * len(sides), np.int32))
    keep, args = [], []
    for k, (ptr, idx, cols) in enumerate(sides):
        d = [gp_ffi.DeviceArray(ptr), gp_ffi.DeviceArray(idx),
             gp_ffi.DeviceArray(size=max(L.gpk_csr_check_chunks(len(idx)), 1), dtype=np.int32)]
        keep.append(d)
        args.append(Side(d[0].ptr, d[1].ptr, len(ptr) - 1, cols, len(idx), 0, d[2].ptr, flags.ptr + 16 * k))
    gp_ffi.hip_check(L.gpk_csr_check(*args, None), "check")
    return flags.numpy().reshape(-1, 4)


def expected(ptr, idx, cols):
    inner = np.ones(len(idx), bool)
    inner[ptr[:-1][np.diff(ptr) > 0]] = False
    before = np.concatenate([[0], idx[:-1]])
    return [0, int(((idx < 0) | (idx >= cols)).any()), int((inner & (idx == before)).any()),
            int((inner & (idx < before)).any())]


FAULTS = {"none": [], "equal": [0], "descending": [1], "range": [2], "last-row": [3]}


@pytest.mark.parametrize("fault", list(FAULTS))
@pytest.mark.parametrize("gaps", [[0], [8100], [8190, 8191, 8192, 8193], [30_000, 1, 9000], [300_000]])
def test_chunks_that_span_empty_rows(gaps, fault):
    """Every row starts at column 0, below the end of the row before it: an
    entry is a neighbour's equal or less only where a row starts."""
    lens = [5] * 700
    for g in gaps:
        lens += [0] * g + [1, 7, 3, 2048, 900]
    lens += [0] * 9000
    ptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    row = np.repeat(np.arange(len(lens)), lens)
    idx = (np.arange(ptr[-1]) - ptr[row]).astype(np.int32)
    after = 700 + gaps[0] + 1  # the row of 7 entries behind the first gap
    if fault == "equal":
        idx[ptr[after] + 1] = idx[ptr[after]]
    elif fault == "descending":
        idx[ptr[after + 1] - 1] = 2
    elif fault == "range":
        idx[ptr[after] + 6] = 5000
    elif fault == "last-row":
        idx[-1] = idx[-2]
    sound = (np.array([0, 2, 2, 3], np.int32), np.array([4, 9, 1], np.int32), 10)
    got = flags_of([(ptr, idx, 3000), sound])
    assert got[0].tolist() == expected(ptr, idx, 3000)
    assert got[1].tolist() == [0, 0, 0, 0]
    assert got[0].any() == (fault != "none")
