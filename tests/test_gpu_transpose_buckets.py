"""Transposes large enough for the buckets of columns, against the oracle, bit
for bit: one column, one bucket and many columns to a bucket, chunks whose rows
are long, empty or many, buckets of one tile and of several, buckets split into
pieces, and sizes on both sides of the rule."""
import ctypes as C

import numpy as np
import pytest

import gp_ffi
import oracle_ffi as O
from helpers import assert_same_array

MIN, TILE = 1 << 20, 4096


def route(n, nnz):
    """(buckets, low) of the library's rule; 0 buckets: the sort."""
    low = C.c_int32()
    return gp_ffi.lib().gpk_transpose_buckets(n, nnz, C.byref(low)), low.value


def shape(n, idx):
    """(entries of each bucket, tiles of the largest whole one, pieces of each)."""
    buckets, low = route(n, len(idx))
    assert buckets > 0
    sizes = np.bincount(idx >> low, minlength=buckets)
    share = max(16384, len(idx) // 128 + 1)
    pieces = np.maximum(-(-sizes // share), 1)
    return sizes, -(-int(sizes[pieces == 1].max(initial=0)) // TILE), pieces


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
    elif kind == "gap":  # a tile that spans more empty rows than it marks, others a few more or less
        lens = np.concatenate([np.full(nnz // 10 - 5040, 5)] + [np.r_[np.zeros(g, np.int64), np.full(700, 6)] for g in
                               (8186, 8190, 8192, 8193, 8200, 300_000)] + [np.full(nnz // 10 + 2, 5)])
    else:  # empty rows in between, by the thousand
        lens = np.zeros(400_000, np.int64)
        at = np.random.default_rng(1).choice(400_000, nnz // 40 + 1, replace=False)
        lens[at] = 40
    cut = int(lens.sum()) - nnz
    lens[np.nonzero(lens)[0][-1]] -= cut
    return lens


def check(m, n, ptr, idx, val):
    got = gp_ffi.transpose_csr(m, n, ptr, idx, val)
    want = O.transpose_csr(m, n, ptr, idx, val)
    assert got[:2] == want[:2]
    for name, a, b in zip(("ptr", "idx", "val"), got[2:], want[2:]):
        assert_same_array(name, a, b)


KINDS = [
    ("short", 1_500_000, MIN, 0), ("short", 1_500_000, MIN - 1, 0), ("short", 1024, MIN + 4097, 0),
    ("short", 1025, MIN + 1, 0), ("short", 256, MIN + 1, 0), ("short", 257, MIN + 1, 0), ("short", 2_097_152, MIN + 5, 0), ("short", 2_097_153, MIN + 5, 0),
    ("long", 100_003, MIN + 17, 0), ("long", 3000, MIN + 17, 0), ("empty", 70_000, MIN + 3, 0),
    ("short", 200_000, MIN + 7, 15_000), ("short", 200_000, MIN + 7, 65_000), ("short", 200_000, MIN + 7, 120_000),
    ("one-row", 1_500_000, MIN + 9, 0), ("gap", 70_000, MIN + 3, 0),
]


@pytest.mark.gpu
@pytest.mark.parametrize("kind,n,nnz,hot", KINDS)
def test_transpose_by_buckets(kind, n, nnz, hot):
    lens = lengths(kind, nnz)
    ptr, idx, val = matrix(lens, n, 7, hot)
    assert len(idx) == nnz and idx.min() >= 0 and idx.max() < n
    check(len(lens), n, ptr, idx, val)


def of_buckets(n, nnz, given, columns=None):
    """Short rows with `given` entries in the first buckets, the others' spread
    over the rest (columns: all entries in the first so many columns)."""
    rng = np.random.default_rng(nnz)
    buckets, low = route(n, nnz)
    if columns:
        idx = rng.integers(0, columns, nnz)
    else:
        bucket = np.concatenate([np.repeat(np.arange(len(given)), given),
                                 rng.integers(len(given), buckets, nnz - sum(given))])
        last = np.minimum(((bucket + 1) << low) - 1, n - 1)
        idx = rng.integers(bucket << low, last + 1)
    m = nnz // 7 + 1
    rows = rng.integers(0, m, nnz)
    order = np.lexsort((idx, rows))
    ptr = np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=m))]).astype(np.int32)
    return m, ptr, idx[order].astype(np.int32), rng.standard_normal(nnz)


EDGES = [4096, 4097, 8191, 8192, 8193, 12288, 12289, 16383, 16384, 16385, 32768, 32769, 49153]
# n, nnz, the first buckets' entries, columns; tiles of the largest whole bucket, most pieces
SHAPES = {
    "edges": (1_500_000, MIN + 500_001, EDGES, 0, 4, 4),
    "several-tiles": (1_500_000, 8_000_003, [], 0, 3, 1),
    "several-tiles-few-columns": (3000, 6_000_001, [], 0, 3, 1),
    "one-bucket": (1_500_000, MIN + 5, [], 2048, 0, 65),
    "one-column": (1_500_000, MIN + 5, [], 1, 0, 65),
    "hot": (1_500_000, 2_000_000, [300_000, 5, 100_000, 0, 200_000], 0, 1, 19),
}


@pytest.mark.parametrize("case", list(SHAPES))
def test_shapes_take_the_path_they_name(case):
    n, nnz, given, columns, tiles, most = SHAPES[case]
    m, ptr, idx, val = of_buckets(n, nnz, given, columns)
    sizes, whole_tiles, pieces = shape(n, idx)
    assert sizes[:len(given)].tolist() == given and sizes.sum() == nnz == ptr[-1]
    assert (whole_tiles, int(pieces.max())) == (tiles, most)
    assert route(n, nnz)[1] > 0  # several columns to a bucket
    assert pieces.sum() <= len(sizes) + 128 and pieces[pieces > 1].sum() <= 256


@pytest.mark.gpu
@pytest.mark.parametrize("case", list(SHAPES))
def test_tiles_and_pieces_of_buckets(case):
    n, nnz, given, columns, _, _ = SHAPES[case]
    m, ptr, idx, val = of_buckets(n, nnz, given, columns)
    check(m, n, ptr, idx, val)
