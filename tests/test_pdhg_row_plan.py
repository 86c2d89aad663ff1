"""The solver's row blocks with long rows in parts (gpk_pdhg_row_plan, on the
CPU) and the kernels that walk them, at the lengths where a row changes from a
thread to a wave, to a workgroup, to parts: each sum within its rounding bound
of the exact one and the same bits every time."""
import ctypes as C
import math
import os
import shutil
import subprocess

import numpy as np
import pytest

import gp_ffi

BUDGET = 2048
EDGES = [31, 32, 33, 63, 64, 65, 255, 256, 257, 2047, 2048, 2049, 4095, 4096, 4097, 6000]
CASES = {
    "edges": EDGES + [0, 1, 2] * 300 + EDGES[::-1],
    "neighbours": [2049] * 5 + [257] * 9 + [33] * 70 + [0] * 600 + [1],
    "many-parts": [0, 600_000, 3, 40_000],
    "short": [3] * 1000,
    "few-rows-by-wave": [100] * 61 + [200, 33, 32, 1, 0] * 30 + [150] * 40,
    "many-rows-by-wave": [200, 256, 40] + [3] * 240 + [150] + [0] * 30 + [33] + [7] * 150,
    "empty": [0] * 700,
}


class Rows(C.Structure):
    _fields_ = [("M", gp_ffi.T.GpCsr), ("blk", C.c_void_p), ("blocks", C.c_int32), ("part_sum", C.c_void_p),
                ("part_count", C.c_void_p)]


def plan(ptr):
    f = gp_ffi.lib().gpk_pdhg_row_plan
    f.restype, f.argtypes = C.c_int32, [C.c_void_p, C.c_int32, C.c_void_p]
    nb = f(ptr.ctypes.data, len(ptr) - 1, None)
    out = np.full((nb + 1, 4), -1, np.int32)
    assert f(ptr.ctypes.data, len(ptr) - 1, out.ctypes.data) == nb
    return out


@pytest.mark.parametrize("case", list(CASES))
def test_plan_covers_every_entry_once(case):
    ptr = np.concatenate([[0], np.cumsum(CASES[case])]).astype(np.int32)
    b = plan(ptr)
    assert b[-1].tolist() == [len(ptr) - 1, ptr[-1], 0, 0]
    row, entry, part, parts = b[:-1].T
    assert np.all(np.diff(b[:, 1]) <= BUDGET) and entry[0] == 0 and row[0] == 0
    multi = parts == 0
    assert np.all(entry[multi] == ptr[row[multi]]) and np.all(b[1:, 0][multi] - row[multi] <= 256)
    for k in np.nonzero(parts > 1)[0]:
        assert ptr[row[k]] + part[k] * BUDGET == entry[k] and row[k - part[k]] == row[k]
        assert parts[k] == -(-int(ptr[row[k] + 1] - ptr[row[k]]) // BUDGET)


def test_plan_says_which_blocks_the_waves_sum():
    """The rows past 32 entries of a block of several rows go to the waves where
    their 200 ns each on four waves are less than the longest's 15 ns an entry."""
    for lens, want in (([40] * 51, 0), ([100] * 20, -1), ([33] + [8] * 200, -1), ([32] * 64, 0), ([200, 1], -1),
                       ([60] * 18 + [8] * 20, 0), ([60] * 17 + [8] * 20, -1)):
        ptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
        b = plan(ptr)
        assert len(b) == 2 and b[0, 3] == want, lens


def test_no_plan_has_more_blocks_than_its_bound():
    f = gp_ffi.lib().gpk_pdhg_row_plan_most
    f.restype, f.argtypes = C.c_int64, [C.c_int32, C.c_int32]
    rng = np.random.default_rng(3)
    shapes = list(CASES.values()) + [[257, 0] * 500, [257] * 999, [256] * 999, [1, 257] * 400, [225] * 777, [0] * 5000]
    shapes += [rng.integers(0, 600, 3000).tolist(), [], [1], [2048, 2049] * 50]
    for lens in shapes:
        ptr = np.concatenate([[0], np.cumsum(np.asarray(lens, np.int64))]).astype(np.int32)
        assert len(plan(ptr)) - 1 <= f(len(lens), int(ptr[-1]))


@pytest.mark.parametrize("arch,compiles", [("gfx950", True), ("gfx942", False)])
def test_split_rows_are_tied_to_their_target(arch, compiles):
    """The order of a row's parts is gfx950's: no other target may compile it."""
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    csrc = os.path.join(root, "gpu-presolver_amd", "csrc")
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    r = subprocess.run([hipcc, f"--offload-arch={arch}", "--cuda-device-only", "-fsyntax-only", "-std=c++17",
                        "-I" + os.path.join(root, "include"), "-I" + csrc, os.path.join(csrc, "k_pdhg.hip")],
                       capture_output=True, text=True, timeout=100)
    assert (r.returncode == 0) == compiles, r.stderr
    assert compiles or "as gfx950 does" in r.stderr


@pytest.mark.gpu
@pytest.mark.parametrize("case", list(CASES))
def test_row_kernels(case):
    lens = CASES[case]
    m, n = len(lens), max(max(lens), 1)
    rng = np.random.default_rng(5)
    ptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    idx = np.concatenate([rng.choice(n, size=k, replace=False) for k in lens]).astype(np.int32)
    val = rng.standard_normal(len(idx))
    v, dc, dr = rng.standard_normal(n), 0.5 + rng.random(n), 0.5 + rng.random(m)
    A = gp_ffi.DeviceCsr(m, n, ptr, idx, val)
    b = plan(ptr)
    nb = len(b) - 1
    dev = {k: gp_ffi.DeviceArray(a) for k, a in dict(
        blk=b.reshape(-1), part_sum=np.zeros(nb), part_count=np.zeros(nb, np.int32), v=v, dc=dc, dr=dr,
        y=np.zeros(m), out=np.zeros(max(len(idx), 1)), partial=np.zeros(4 * nb), res=np.zeros(4),
        sumsq=np.array([2.0])).items()}
    R = Rows(A.g, dev["blk"].ptr, nb, dev["part_sum"].ptr, dev["part_count"].ptr)
    L = gp_ffi.lib()
    vp = C.c_void_p

    def call(name, *args):
        f = getattr(L, name)
        f.restype, f.argtypes = C.c_int32, [Rows] + [vp] * len(args)
        assert f(R, *args) == 0

    def rows_near(got, terms, what):
        for r in range(m):
            t = terms[ptr[r]:ptr[r + 1]]
            # each of the sums adds every term once, rounded at most len times
            assert abs(got[r] - math.fsum(t)) <= (len(t) + 4) * 2.0 ** -53 * np.abs(t).sum(), (what, r, len(t))

    for sumsq, x in ((None, v), (dev["sumsq"].ptr, v * (1.0 / math.sqrt(2.0)))):
        runs = []
        for _ in range(3):
            call("gpk_pdhg_spmv", dev["v"].ptr, sumsq, dev["y"].ptr, None)
            runs.append(dev["y"].numpy())
        assert np.array_equal(runs[0], runs[1]) and np.array_equal(runs[0], runs[2])
        rows_near(runs[0], val * x[idx], "spmv")
    call("gpk_pdhg_spmv_sq", dev["v"].ptr, dev["y"].ptr, dev["partial"].ptr, dev["res"].ptr, None)
    y = dev["y"].numpy()
    rows_near(y, val * v[idx], "spmv_sq")
    want = math.fsum(y * y)
    assert abs(dev["res"].numpy()[0] - want) <= (m + 4) * 2.0 ** -53 * want
    call("gpk_pdhg_scale_csr", dev["dr"].ptr, dev["dc"].ptr, dev["out"].ptr, None)
    rows = np.repeat(np.arange(m), lens)
    assert np.array_equal(dev["out"].numpy()[:len(idx)], val * dr[rows] * dc[idx])
    call("gpk_pdhg_ruiz", dev["dr"].ptr, None)
    top = np.array([np.abs(val[ptr[r]:ptr[r + 1]]).max(initial=0.0) for r in range(m)])
    assert np.allclose(dev["dr"].numpy(), np.where(top > 0, dr / np.sqrt(np.where(top > 0, top, 1.0)), dr),
                       rtol=2.0 ** -51, atol=0.0)
