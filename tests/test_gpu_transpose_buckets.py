"""Transposes large enough for the buckets of columns, against the oracle, bit
for bit: one column, one bucket and many columns to a bucket, chunks whose rows
are long, empty or many, a bucket over the limit (the sort then), and sizes on
both sides of the rule."""
import numpy as np
import pytest

import gp_ffi
import oracle_ffi as O
from helpers import assert_same_array

pytestmark = pytest.mark.gpu

MIN = 1 << 20


def matrix(lens, n, seed, hot=0):
    """Rows of the given lengths, ascending columns; `hot` entries of the first
    rows sit in column 3."""
    rng = np.random.default_rng(seed)
    ptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    nnz = int(ptr[-1])
    rows = np.repeat(np.arange(len(lens)), lens)
    k = np.arange(nnz) - ptr[rows]
    stride = max(n // max(int(max(lens)), 1), 1)
    idx = (rng.integers(0, stride, nnz) + k * stride).astype(np.int32)
    idx[ptr[:-1][np.asarray(lens) > 0][:hot]] = 3 if stride > 3 else 0
    return ptr, idx, rng.standard_normal(nnz)


def lengths(kind, nnz):
    if kind == "short":
        lens = np.full(nnz // 5 + 1, 5)
    elif kind == "long":
        lens = np.full(nnz // 3000 + 1, 3000)
    elif kind == "one-row":
        lens = np.array([nnz])
    else:  # empty rows in between, by the thousand
        lens = np.zeros(400_000, np.int64)
        at = np.random.default_rng(1).choice(400_000, nnz // 40 + 1, replace=False)
        lens[at] = 40
    cut = int(lens.sum()) - nnz
    lens[np.nonzero(lens)[0][-1]] -= cut
    return lens


@pytest.mark.parametrize("kind,n,nnz,hot", [
    ("short", 1_500_000, MIN, 0), ("short", 1_500_000, MIN - 1, 0), ("short", 1024, MIN + 4097, 0),
    ("short", 1025, MIN + 1, 0), ("short", 256, MIN + 1, 0), ("short", 257, MIN + 1, 0), ("short", 2_097_152, MIN + 5, 0), ("short", 2_097_153, MIN + 5, 0),
    ("long", 100_003, MIN + 17, 0), ("long", 3000, MIN + 17, 0), ("empty", 70_000, MIN + 3, 0),
    ("short", 200_000, MIN + 7, 65_000), ("short", 200_000, MIN + 7, 120_000), ("one-row", 1_500_000, MIN + 9, 0),
])
def test_transpose_by_buckets(kind, n, nnz, hot):
    lens = lengths(kind, nnz)
    m = len(lens)
    ptr, idx, val = matrix(lens, n, 7, hot)
    assert len(idx) == nnz and idx.min() >= 0 and idx.max() < n
    got = gp_ffi.transpose_csr(m, n, ptr, idx, val)
    want = O.transpose_csr(m, n, ptr, idx, val)
    assert got[:2] == want[:2]
    for name, a, b in zip(("ptr", "idx", "val"), got[2:], want[2:]):
        assert_same_array(name, a, b)
