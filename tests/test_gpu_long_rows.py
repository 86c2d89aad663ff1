"""Rows far longer than their neighbours: the kernels that give such a row a
wave (or a tile of its own entries) against the oracle, bit for bit, at the
lengths where the split happens and with neighbouring long rows."""
import numpy as np
import pytest

import gp_ffi
import lp_synth
import oracle_ffi as O
from helpers import assert_same_array

pytestmark = pytest.mark.gpu


def csr_of_lengths(lengths, n, seed):
    """Random dyadic CSR with the given row lengths (columns ascending)."""
    rng = np.random.default_rng(seed)
    ptr = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    idx = np.concatenate([np.sort(rng.choice(n, size=int(k), replace=False)) for k in lengths] or [np.zeros(0)])
    val = np.round(rng.uniform(0.5, 2.0, len(idx)) * 8) / 8 * rng.choice([-1.0, 1.0], len(idx))
    return ptr, idx.astype(np.int32), val


def lengths_with_long_rows(seed):
    """Edges of the 128-entry split and of the 256-entry chunk, scattered and
    adjacent, between short and empty rows."""
    rng = np.random.default_rng(seed)
    edges = [127, 128, 129, 255, 256, 257, 383, 384, 511, 512, 513, 767, 1023, 1025, 2047, 2048, 2049, 2999]
    out = [int(k) for k in rng.integers(0, 9, 300)]
    for e in edges:
        out += [e, int(rng.integers(0, 9))]
    out += [int(k) for k in rng.integers(0, 9, 200)] + edges + [0, 1] + [700] * 70
    return out


@pytest.mark.parametrize("lengths", [[129], [128], [0, 3000, 0], lengths_with_long_rows(1),
                                     [1500] * 257 + [3] * 9000 + [400] * 3])
def test_row_activity_long_rows(lengths):
    m, n = len(lengths), 3000
    ptr, idx, val = csr_of_lengths(lengths, n, 5)
    val[::7] = 0.0  # explicit zeros are skipped
    rng = np.random.default_rng(6)
    l, u = -np.round(rng.uniform(0, 4, n) * 1024) / 1024, np.round(rng.uniform(0, 4, n) * 1024) / 1024
    l[rng.random(n) < 0.1], u[rng.random(n) < 0.1] = -np.inf, np.inf
    val *= 1.0 + rng.random(len(val)) * 2.0 ** -20  # sums that round: the order of the terms shows
    got = gp_ffi.row_activity(m, n, ptr, idx, val, l, u, 1e-10)
    want = O.row_activity(m, n, ptr, idx, val, l, u, 1e-10)
    for name, a, b in zip(("min_fin", "max_fin", "neg_inf", "pos_inf"), got, want):
        assert_same_array(name, a, b)
