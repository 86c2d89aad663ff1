"""Walks of rows that end at the last entries a matrix can hold (2^31 - 1): the
positions that a group of lanes forms past a row's end (csrc/gp_walk.hpp,
compiled here for the host, where overflow is an error), and on the GPU the row
activity of a matrix with every entry."""
import os
import subprocess

import numpy as np
import pytest

import gp_ffi

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "gpu-presolver_amd", "csrc")
LAST = 2 ** 31 - 1

PROGRAM = r"""
#include <climits>
#include <cstdio>
#include <initializer_list>
#include "gp_walk.hpp"
using namespace gpdev;

// Every entry of [b, e) met once, in order, by `lanes` lanes that read `ahead`
// steps past the one they are at.
static bool walk(int32_t b, int32_t e, uint32_t lanes, uint32_t ahead) {
  const uint32_t n = row_length(b, e);
  uint32_t met = 0;
  for (uint32_t c = 0; c < n; c += lanes)
    for (uint32_t lane = 0; lane < lanes; ++lane) {
      const int32_t p = row_entry(b, e, c + lane), next = row_entry(b, e, c + ahead * lanes + lane);
      if (p < b || p >= e || next < p || next >= e) return false;
      if (c + lane < n) {
        if (p != b + static_cast<int32_t>(met)) return false;
        ++met;
      }
    }
  return met == n;
}

int main() {
  int bad = 0;
  for (int32_t len : {1, 63, 64, 65, 128, 129, 255, 256, 257, 511, 512, 513, 3000})
    for (int32_t end : {len, 5000, INT_MAX - 600, INT_MAX - 257, INT_MAX - 64, INT_MAX - 1, INT_MAX})
      for (uint32_t lanes : {8u, 64u, 256u, 2048u})
        if (end >= len && !walk(end - len, end, lanes, 1)) bad += std::printf("row [%d, %d), %u lanes\n", end - len, end, lanes);
  if (row_length(0, INT_MAX) != static_cast<uint32_t>(INT_MAX) || row_entry(0, INT_MAX, 0xffffff00u) != INT_MAX - 1)
    bad += std::printf("the longest row\n");
  return bad != 0;
}
"""


def test_positions_of_the_last_rows(tmp_path):
    src, exe = tmp_path / "walk.cpp", tmp_path / "walk"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-ftrapv", "-I", CSRC, str(src), "-o", str(exe)],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout


@pytest.mark.gpu
@pytest.mark.parametrize("tail", [255, 127])
def test_row_activity_up_to_the_last_entry(tail):
    """Rows of 128 entries and a last one that a wave (255) or a tile (127) takes."""
    rows = (LAST - tail) // 128
    assert rows * 128 + tail == LAST
    ptr = np.append(np.arange(rows + 1, dtype=np.int64) * 128, LAST).astype(np.int32)
    m = rows + 1
    d_ptr = gp_ffi.DeviceArray(ptr)
    idx, val = gp_ffi.DeviceArray(size=LAST, dtype=np.int32), gp_ffi.DeviceArray(size=LAST)
    gp_ffi.hip_check(gp_ffi.hip().hipMemset(idx.ptr, 0, 4 * LAST), "hipMemset")
    gp_ffi.hip_check(gp_ffi.hip().hipMemset(val.ptr, 0x3f, 8 * LAST), "hipMemset")
    v = np.frombuffer(b"\x3f" * 8, np.float64)[0]
    l, u = gp_ffi.DeviceArray(np.array([1.0])), gp_ffi.DeviceArray(np.array([2.0]))
    out = [gp_ffi.DeviceArray(size=m), gp_ffi.DeviceArray(size=m), gp_ffi.DeviceArray(size=m, dtype=np.int32),
           gp_ffi.DeviceArray(size=m, dtype=np.int32)]
    A = gp_ffi.T.GpCsr(m, 1, LAST, d_ptr.ptr, idx.ptr, val.ptr)
    gp_ffi._check(gp_ffi.lib().gp_row_activity(gp_ffi.C.byref(A), l.ptr, u.ptr, 1e-10, *[o.ptr for o in out], None))
    low, high, neg, pos = [o.numpy() for o in out]
    sums = np.cumsum(np.full(255, v))  # one after the other, as a row is added
    assert np.all(low[:-1] == sums[127]) and np.all(high[:-1] == 2 * sums[127])
    assert low[-1] == sums[tail - 1] and high[-1] == 2 * sums[tail - 1]
    assert not neg.any() and not pos.any()
