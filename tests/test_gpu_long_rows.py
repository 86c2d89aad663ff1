"""Rows far longer than their neighbours: the kernels that give such a row a
wave (or a tile of its own entries) against the oracle, bit for bit, at the
lengths where the split happens and with neighbouring long rows."""
import ctypes as C

import numpy as np
import pytest

import gp_ffi
import lp_synth
import oracle_ffi as O
from helpers import assert_same_array, assert_same_lp, assert_same_record

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


def scattered_lengths(seed):
    """Long rows between short and empty ones in every tile of 256, at its ends
    and alone in it."""
    rng = np.random.default_rng(seed)
    out = [129, 0, 1] * 85 + [129]
    out += [0, 300] * 128 + [5] * 255 + [140] + [140] + [5] * 255 + [200] * 256 + [0] * 255 + [131] + [0] * 256
    out += [int(k) for k in np.where(rng.random(3000) < 0.05, rng.integers(120, 300, 3000), rng.integers(0, 60, 3000))]
    return out


@pytest.mark.parametrize("lengths", [[129], [128], [0, 3000, 0], lengths_with_long_rows(1),
                                     [1500] * 257 + [3] * 9000 + [400] * 3, scattered_lengths(2)])
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


@pytest.mark.parametrize("m", [262_144, 262_145, 600_000, 1_200_001])
def test_long_rows_of_large_matrices(m):
    """Long rows where the waves' shares of the rows change: single rows up to
    262,144 of them, groups of 16 past that; first and last row, neighbours in a
    group, both sides of a group's end and of the rows that one look covers."""
    n, group = 3000, 1 if m <= 262_144 else 16
    longs = [129, 130, 255, 256, 257, 500, 3000, 1000, 200, 300]
    at = {0, 1, m - 1, m - 2, 1603, 1604, 1615, 1616, m // 2 // 16 * 16 - 1, m // 2 // 16 * 16}
    while True:  # the looks' length follows the entries: 8 x 64 rows for each wave
        rows = sorted(at)
        lengths = np.zeros(m, np.int64)
        lengths[::37] = 2
        lengths[rows] = np.resize(longs, len(rows))
        most = min(m, int(lengths.sum()) // 129 + 1)
        waves = 4 * min(2048, -(-most // 4))
        look = 8 * 64 * waves
        more = {r for k in range(1, m // look + 1) for r in (k * look - 1, k * look) if r < m}
        more |= {r for r in (group * waves - 1, group * waves, 524_287, 524_288) if r < m}
        if more <= at or len(at) > 200:
            break
        at |= more
    ptr, idx, val = csr_of_lengths(lengths[lengths > 0], n, 19)
    ptr = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    val *= 1.0 + np.random.default_rng(20).random(len(val)) * 2.0 ** -20
    l, u = np.full(n, -1.0), np.full(n, 2.0)
    u[::11] = np.inf
    got = gp_ffi.row_activity(m, n, ptr, idx, val, l, u, 1e-10)
    want = O.row_activity(m, n, ptr, idx, val, l, u, 1e-10)
    for name, a, b in zip(("min_fin", "max_fin", "neg_inf", "pos_inf"), got, want):
        assert_same_array(name, a, b)


def compact_lengths(case):
    rng = np.random.default_rng(11)
    if case == "edges":  # chunks of 2,048 entries: rows that end, start and straddle there
        return [2048, 2048, 2047, 1, 4096, 0, 0, 1, 2046, 1, 3, 5000, 0, 2049] + [0] * 300 + [7]
    if case == "long":
        return lengths_with_long_rows(12)
    if case == "empty-gap":  # one chunk spans more empty rows than it marks in its bitmap
        return [3] * 100 + [0] * 20000 + [5, 0, 900] + [0] * 9000
    if case == "empty-ends":
        return [0] * 5000 + [1] * 4100 + [0] * 5000
    if case == "counts":  # more rows than a tile counts again
        return list(rng.integers(0, 3, 262144 + 4001))
    if case == "scan":  # more chunks than a block sums
        return [1400] * 3010
    if case == "large-chunks":  # the first size of 2,048-entry chunks
        return [1024] * 1024 + [1]
    if case == "small-chunks":
        return [1024] * 1024
    return list(rng.integers(0, 9, 40000))  # "recount"


@pytest.mark.parametrize("case", ["edges", "long", "empty-gap", "empty-ends", "counts", "scan", "recount",
                                  "large-chunks", "small-chunks"])
@pytest.mark.parametrize("drop", [0.0, 0.3, 1.0])
def test_compaction_by_chunks(case, drop):
    lengths = compact_lengths(case)
    m, n = len(lengths), 5001
    ptr, idx, val = csr_of_lengths([min(int(k), n) for k in lengths], n, 13)
    rng = np.random.default_rng(14)
    kr, kc = (rng.random(m) >= drop).astype(np.uint8), (rng.random(n) >= drop / 2).astype(np.uint8)
    got = gp_ffi.compact_csr(m, n, ptr, idx, val, kr, kc)
    want = O.compact_csr(m, n, ptr, idx, val, kr, kc)
    assert got[:2] == want[:2]
    for name, a, b in zip(("ptr", "idx", "val"), got[2:], want[2:]):
        assert_same_array(name, a, b)


@pytest.mark.parametrize("m", [2048, 5000, 9_000_000])
def test_compaction_masks_at_an_odd_address(m):
    """Masks that no 16-byte load can read; 9,000,000 rows take the look-back."""
    rng = np.random.default_rng(m)
    lengths = np.zeros(m, np.int64)
    lengths[rng.choice(m, 1500, replace=False)] = rng.integers(1, 6, 1500)
    n = 777
    ptr, idx, val = csr_of_lengths(lengths if m < 10000 else lengths[lengths > 0], n, 15)
    ptr = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    kr, kc = (rng.random(m) < 0.6).astype(np.uint8), (rng.random(n) < 0.6).astype(np.uint8)
    A = gp_ffi.DeviceCsr(m, n, ptr, idx, val)
    dr, dc = gp_ffi.DeviceArray(np.concatenate([[9], kr]).astype(np.uint8)), gp_ffi.DeviceArray(np.concatenate([[9], kc]).astype(np.uint8))
    out = gp_ffi.T.GpCsr()
    gp_ffi._check(gp_ffi.lib().gp_compact_csr(C.byref(A.g), dr.ptr + 1, dc.ptr + 1, C.byref(out)))
    got = (out.rows, out.cols) + gp_ffi._take_csr(out)
    want = O.compact_csr(m, n, ptr, idx, val, kr, kc)
    assert got[:2] == want[:2]
    for name, a, b in zip(("ptr", "idx", "val"), got[2:], want[2:]):
        assert_same_array(name, a, b)


def with_dense_rows(lp, lengths, seed):
    """The LP with further rows of the given lengths (wide or one-sided
    bounds), every third one a scaled copy of the one before it."""
    rng = np.random.default_rng(seed)
    m, n = lp["m"], lp["n"]
    rows, cols, vals, AL, AU = [], [], [], [], []
    for k, length in enumerate(lengths):
        if k % 3 == 2:
            f = -2.0
            c, v, lo, hi = cols[-1], f * vals[-1], f * AU[-1], f * AL[-1]
        else:
            c = np.sort(rng.choice(n, size=min(length, n), replace=False))
            v = np.round(rng.uniform(0.5, 2.0, len(c)) * 8) / 8 * rng.choice([-1.0, 1.0], len(c))
            lo, hi = (-np.inf, 2.0 ** 21) if k % 2 else (-2.0 ** 21, 2.0 ** 21)
        rows.append(np.full(len(c), m + k))
        cols.append(c)
        vals.append(v)
        AL.append(lo)
        AU.append(hi)
    r0 = np.repeat(np.arange(m), np.diff(lp["A_ptr"]))
    M = m + len(lengths)
    ptr, idx, val = lp_synth.csr_from_coo(M, n, np.concatenate([r0] + rows), np.concatenate([lp["A_idx"]] + cols),
                                          np.concatenate([lp["A_val"]] + vals))
    tptr, tidx, tval = lp_synth.transpose_csr(M, n, ptr, idx, val)
    return dict(lp, m=M, A_ptr=ptr, A_idx=idx, A_val=val, AT_ptr=tptr, AT_idx=tidx, AT_val=tval,
                AL=np.concatenate([lp["AL"], AL]), AU=np.concatenate([lp["AU"], AU]))


@pytest.mark.parametrize("lengths,kw", [
    ([127, 128, 128, 129, 130, 130, 255, 256, 257] * 3, {}),
    ([2500, 2500, 2500, 600, 300, 300] * 4, dict(record_postsolve_tape_cpu=1)),
    # more deltas in a row than a wave places by rank, and more columns than its bitmap holds
    ([4400, 4000, 4000] * 3, dict(doubleton_equations_min_selected_per_batch=1,
                                  doubleton_equations_min_selected_ratio=0.0)),
    ([17000, 16384, 16385, 9000, 200], dict(doubleton_equations_min_selected_per_batch=1,
                                            doubleton_equations_min_selected_ratio=0.0)),
    ([700] * 60, dict(use_tiered_scheduler=0)),
])
def test_presolve_with_dense_rows(lengths, kw):
    big = max(lengths) > 4400
    lp = lp_synth.generate(14000 if big else 3000, 18000 if big else 4500, seed=31, mean_row_len=4.0,
                           frac_doubleton=0.25, frac_fixed_cols=0.05, frac_singleton_cols=0.15)
    lp = with_dense_rows(lp, lengths, 32)
    kw = dict(kw, enable_structure_specific_rules=0, doubleton_equations_max_fill_in_proxy=100000)
    sg, rg, lg = gp_ffi.presolve(lp, gp_ffi.params(**kw), True)
    so, ro, lo = O.presolve(lp, O.params(**kw), True)
    assert (sg["reduced_rows"], sg["reduced_cols"], sg["reduced_nnz"]) == (so["reduced_rows"], so["reduced_cols"],
                                                                           so["reduced_nnz"])
    assert sg["obj_constant_delta"] == so["obj_constant_delta"]
    assert_same_record(rg, ro)
    assert_same_lp(lg, lo)


def with_dense_columns(lp, lengths, seed):
    """The LP with further columns of the given lengths, every third one a
    scaled copy of the one before it, and an equality of every sixth with a
    column of the LP."""
    rng = np.random.default_rng(seed)
    m, n, k = lp["m"], lp["n"], len(lengths)
    rows, cols, vals, c = [], [], [], []
    for j, length in enumerate(lengths):
        if j % 3 == 2:
            r, v, cost = rows[-1], -2.0 * vals[-1], -2.0 * c[-1]
        else:
            r = np.sort(rng.choice(m, size=min(length, m), replace=False))
            v = np.round(rng.uniform(0.5, 2.0, len(r)) * 8) / 8 * rng.choice([-1.0, 1.0], len(r))
            cost = float(rng.integers(-8, 9)) / 8
        rows.append(r)
        cols.append(np.full(len(r), n + j))
        vals.append(v)
        c.append(cost)
    pairs = rng.choice(n, size=k, replace=False)
    eq = np.arange(0, k, 6)
    r0 = np.repeat(np.arange(m), np.diff(lp["A_ptr"]))
    M, N = m + len(eq), n + k
    ptr, idx, val = lp_synth.csr_from_coo(
        M, N, np.concatenate([r0] + rows + [m + np.arange(len(eq)), m + np.arange(len(eq))]),
        np.concatenate([lp["A_idx"]] + cols + [n + eq, pairs[eq]]),
        np.concatenate([lp["A_val"]] + vals + [np.full(len(eq), 2.0), np.full(len(eq), -1.0)]))
    tptr, tidx, tval = lp_synth.transpose_csr(M, N, ptr, idx, val)
    big = 2.0 ** 24
    return dict(lp, m=M, n=N, A_ptr=ptr, A_idx=idx, A_val=val, AT_ptr=tptr, AT_idx=tidx, AT_val=tval,
                c=np.concatenate([lp["c"], c]), l=np.concatenate([lp["l"], np.full(k, -big)]),
                u=np.concatenate([lp["u"], np.full(k, big)]), AL=np.concatenate([lp["AL"], np.zeros(len(eq))]),
                AU=np.concatenate([lp["AU"], np.zeros(len(eq))]))


@pytest.mark.parametrize("lengths,kw", [
    ([127, 128, 128, 129, 130, 130, 255, 256, 256, 8, 9, 9] * 2, {}),
    ([2500, 2500, 2500, 600, 300, 300] * 4, dict(doubleton_equations_max_fill_in_proxy=100000)),
    ([2900, 7, 7, 16, 17, 17, 1000, 1000, 1000] * 3, dict(record_postsolve_tape_cpu=1)),
])
def test_presolve_with_dense_columns(lengths, kw):
    lp = lp_synth.generate(3000, 4500, seed=51, mean_row_len=4.0, frac_doubleton=0.25, frac_fixed_cols=0.05,
                           frac_singleton_cols=0.15, frac_dup_rows=0.0, frac_eq=0.0)
    lp = with_dense_columns(lp, lengths, 52)
    kw = dict(kw, enable_structure_specific_rules=0)
    sg, rg, lg = gp_ffi.presolve(lp, gp_ffi.params(**kw), True)
    so, ro, lo = O.presolve(lp, O.params(**kw), True)
    assert (sg["reduced_rows"], sg["reduced_cols"], sg["reduced_nnz"]) == (so["reduced_rows"], so["reduced_cols"],
                                                                           so["reduced_nnz"])
    assert sg["obj_constant_delta"] == so["obj_constant_delta"]
    assert_same_record(rg, ro)
    if not so["has_infeasible"]:  # the first LP's rules end at a contradiction, after doubletons and duplicates
        assert_same_lp(lg, lo)
    assert sg["has_infeasible"] == so["has_infeasible"]


def test_presolve_with_long_columns_past_262144():
    """More columns than the waves share one by one, some of them long."""
    lp = lp_synth.generate(60_000, 264_000, seed=61, mean_row_len=5.0, frac_doubleton=0.1, frac_singleton_cols=0.1)
    lp = with_dense_columns(lp, [129, 300, 300, 128, 2500, 2500, 700, 140, 140] * 3, 62)
    kw = dict(enable_structure_specific_rules=0)
    sg, rg, lg = gp_ffi.presolve(lp, gp_ffi.params(**kw), True)
    so, ro, lo = O.presolve(lp, O.params(**kw), True)
    assert lp["n"] > 262_144 and not so["has_infeasible"]
    assert sg["obj_constant_delta"] == so["obj_constant_delta"]
    assert_same_record(rg, ro)
    assert_same_lp(lg, lo)


@pytest.mark.parametrize("n", [4097, 2048 * 16, 2048 * 16 + 1, 2048 * 17 - 1, 2048 * 64, 2048 * 64 + 1])
def test_radix_sort_at_histogram_batches(n):
    rng = np.random.default_rng(n)
    keys, vals = rng.integers(0, 1 << 20, n).astype(np.uint64), np.arange(n, dtype=np.int32)
    k, v = gp_ffi.radix_sort(keys, vals, 20)
    order = np.argsort(keys, kind="stable")
    assert_same_array("keys", k, keys[order])
    assert_same_array("vals", v, order.astype(np.int32))


@pytest.mark.parametrize("lengths,first,last", [
    ([3] * 9000, 700, 8000), ([3] * 9000, 0, 8000), ([3] * 9000, 700, 9000),  # small chunks
    ([5000] + [2] * 3000 + [4000] * 3, 1, 3001), ([2048] * 700, 2, 690),  # large chunks, whole ones before and after
    ([40] * 300 + [0] * 20000 + [7] + [0] * 9000 + [40] * 300, 200, 29350),  # a chunk that spans many empty rows
])
def test_compaction_of_rows_of_a_larger_matrix(lengths, first, last):
    """Row pointers that begin past entry 0 or end before the matrix's nnz."""
    n = 5001
    ptr, idx, val = csr_of_lengths(lengths, n, 17)
    rng = np.random.default_rng(18)
    m = last - first
    kr, kc = (rng.random(m) < 0.7).astype(np.uint8), (rng.random(n) < 0.7).astype(np.uint8)
    A = gp_ffi.DeviceCsr(len(lengths), n, ptr, idx, val)
    view = gp_ffi.T.GpCsr(m, n, len(idx), A.g.row_ptr + 4 * first, A.g.col_idx, A.g.val)
    dr, dc = gp_ffi.DeviceArray(kr), gp_ffi.DeviceArray(kc)
    out = gp_ffi.T.GpCsr()
    gp_ffi._check(gp_ffi.lib().gp_compact_csr(C.byref(view), dr.ptr, dc.ptr, C.byref(out)))
    got = (out.rows, out.cols) + gp_ffi._take_csr(out)
    b, e = ptr[first], ptr[last]
    want = O.compact_csr(m, n, ptr[first:last + 1] - b, idx[b:e], val[b:e], kr, kc)
    assert got[:2] == want[:2]
    for name, a, w in zip(("ptr", "idx", "val"), got[2:], want[2:]):
        assert_same_array(name, a, w)


SPLIT = [127, 128, 128, 129, 130, 130, 255, 256, 256, 8, 9, 9] * 2


def columns_at_the_split(seed):
    lp = lp_synth.generate(3000, 4500, seed=seed, mean_row_len=4.0, frac_doubleton=0.25, frac_fixed_cols=0.05,
                           frac_singleton_cols=0.15, frac_dup_rows=0.0, frac_eq=0.0)
    return with_dense_columns(lp, SPLIT, 52)


@pytest.mark.parametrize("seed", [53, 60, 72])
def test_presolve_with_columns_at_the_split(seed):
    """LPs that the rules leave feasible, so the reduced costs of columns of 127 to
    130 entries, which the column singletons change, are compared."""
    lp = columns_at_the_split(seed)
    kw = dict(enable_structure_specific_rules=0)
    so, ro, lo = O.presolve(lp, O.params(**kw), True)
    assert not so["has_infeasible"]
    length = np.diff(lp["AT_ptr"])[ro["col_red2org"]]
    changed = set(length[lo["c"] != lp["c"][ro["col_red2org"]]].tolist())
    assert changed & {127, 128} and changed & {129, 130, 131}, sorted(changed)
    sg, rg, lg = gp_ffi.presolve(lp, gp_ffi.params(**kw), True)
    assert sg["obj_constant_delta"] == so["obj_constant_delta"] and not sg["has_infeasible"]
    assert_same_record(rg, ro)
    assert_same_lp(lg, lo)
