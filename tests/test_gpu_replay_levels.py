"""Tapes written by hand for the postsolve replay, against the oracle's
record-by-record replay, bit for bit: lines around the 16 and 32 entries that
are loaded ahead, every record type in one level, levels around a wave's and a
workgroup's records of either kind (those that walk a line and the
others) and around the sizes that take a launch of their own, chains of single
records, and records without rows or an original model."""
import numpy as np
import pytest

import gp_ffi
import lp_synth
import oracle_ffi as O
from helpers import assert_same_array

pytestmark = pytest.mark.gpu

INF = np.inf
LENGTHS = [1, 2, 15, 16, 17, 31, 32, 33, 47, 48, 49, 64, 65, 100]


def original(m, n, seed):
    """An LP whose rows have LENGTHS entries each in turn, in random columns."""
    rng = np.random.default_rng(seed)
    lens = np.resize(LENGTHS, m)
    rows = np.repeat(np.arange(m), lens)
    cols = np.concatenate([np.sort(rng.choice(n, size=k, replace=False)) for k in lens])
    vals = rng.choice([-2.0, -1.0, -0.5, 0.5, 1.0, 2.0], len(cols)) * (1.0 + rng.random(len(cols)) * 2.0 ** -20)
    ptr, idx, val = lp_synth.csr_from_coo(m, n, rows, cols, vals)
    tptr, tidx, tval = lp_synth.transpose_csr(m, n, ptr, idx, val)
    return dict(m=m, n=n, A_ptr=ptr, A_idx=idx, A_val=val, AT_ptr=tptr, AT_idx=tidx, AT_val=tval,
                c=rng.standard_normal(n), l=np.where(rng.random(n) < 0.5, 0.0, -INF), u=np.full(n, INF),
                AL=np.full(m, -INF), AU=np.full(m, 1.0), obj=0.0)


def record_of(m, n, records, seed):
    rng = np.random.default_rng(seed)
    kept = np.sort(rng.choice(n, size=n * 3 // 4, replace=False)).astype(np.int32)
    gone = np.setdiff1d(np.arange(n), kept).astype(np.int32)
    return dict(m0=m, n0=n, m1=m, n1=len(kept), row_red2org=np.arange(m, dtype=np.int32), col_red2org=kept,
                fixed_idx=gone, fixed_val=np.ones(len(gone)), types=np.array([r[0] for r in records], np.int32),
                index_starts=np.cumsum([0] + [len(r[1]) for r in records]).astype(np.int32),
                value_starts=np.cumsum([0] + [len(r[2]) for r in records]).astype(np.int32),
                indices=np.concatenate([r[1] for r in records]).astype(np.int32),
                vals=np.concatenate([r[2] for r in records]).astype(np.float64))


def random_record(rng, lp):
    """A record of a random type on random variables; x is 0 or 1 at first, so
    bound changes to 1 are often tight."""
    m, n = lp["m"], lp["n"]
    t = int(rng.choice([0, 1, 2, 3, 4, 5, 10, 12, 12, 12, 13, 14]))
    k = int(rng.choice(LENGTHS + [0]))
    f = lambda size=None: rng.choice([-2.0, -1.0, -0.5, 0.5, 1.0, 2.0], size) * (1 + rng.random(size) * 2.0 ** -20)
    cols, rows = rng.choice(n, size=k + 3, replace=False), rng.choice(m, size=k + 3, replace=False)
    small = rng.standard_normal(k) / 64
    if t == 0:
        return t, np.r_[cols[0], rows[:k]], np.r_[1.0, f(), small]
    if t == 1:
        return t, np.r_[1, cols[0], 2, cols[:2], 1, cols[0]], np.r_[2.0, 0.5, 1.0, f(2), 0.25, f()]
    if t == 2:
        return t, np.r_[cols[0], rows[0], k, cols[3:]], np.r_[f(), 1.0, 0.0, 0.0, f(), rng.integers(0, 2), small]
    if t == 3:
        return t, cols[:2], np.r_[f(), 0.0, 1.0, -1.0, INF]
    if t == 4:
        return t, rows[:2], np.r_[f(), rng.choice([-INF, 0.0, 1.0]), 1.0, rng.choice([-INF, 0.5]), 2.0]
    if t == 5:
        return t, np.r_[rows[0], cols[0]], np.r_[-INF, 1.0, f()]
    if t == 10:
        return t, rows[:1], np.r_[f()]
    if t == 12:
        row = int(rng.integers(m))
        line = lp["A_idx"][lp["A_ptr"][row]:lp["A_ptr"][row + 1]]
        col = cols[0] if rng.random() < 0.1 else rng.choice(line)
        return t, np.r_[col, row], rng.choice([[0.0, INF, 1.0, INF], [-INF, 3.0, -INF, 1.0], [0.0, 1.0, 0.0, 1.0]])
    if t == 13:
        head = np.r_[4.0, f(), 1.0, 0.0, 0.0, 0.0, 4.0, 0.5, 2.0, f()]
        form = rng.integers(0, 3)  # without bounds' sources, with them, with the line in the tape
        if form < 2:
            return t, np.r_[cols[:2], rows[0]], np.r_[head, rng.choice([0.0, 1.0, 2.0], 2)][:10 + 2 * form]
        return t, np.r_[cols[:2], rows[0], k, rows[3:]], np.r_[head, rng.choice([0.0, 1.0, 2.0], 2), small]
    return t, np.r_[2, cols[0], 0, rows[:2], cols[1:3]], np.r_[1.0, f(), 2.0, 0.25, rng.standard_normal(2) / 64]



def check(lp, records, seed, with_original=True):
    rec = record_of(lp["m"], lp["n"], records, seed)
    rng = np.random.default_rng(seed + 1)
    point = (rng.integers(0, 2, rec["n1"]).astype(float), rng.standard_normal(rec["m1"]), rng.standard_normal(rec["n1"]))
    orig = lp if with_original else None
    with np.errstate(all="ignore"):
        want = O.postsolve(rec, *point, original=orig)
    assert all(np.isfinite(w).all() for w in want)
    got = gp_ffi.postsolve(rec, *point, original=orig)
    for name, a, b in zip("xyz", got, want):
        assert_same_array(name, a, b)


@pytest.mark.parametrize("count,with_original", [(1, True), (40, True), (700, True), (700, False), (4000, True)])
def test_random_tapes(count, with_original):
    lp = original(6000, 9000, 41)
    rng = np.random.default_rng(42 + count)
    check(lp, [random_record(rng, lp) for _ in range(count)], 43, with_original)


def test_levels_of_simple_records():
    """A wave, the workgroup, a launch of their own; launches and runs in turn."""
    m = 2100
    lp = original(m, 900, 51)
    rng = np.random.default_rng(52)
    sizes = [1, 3, 4, 5, 63, 64, 65, 127, 128, 129, 511, 512, 513, 1023, 1024, 1025, 2047, 2048, 2049, 1, 2049, 700]
    records = [(10, np.r_[row], np.r_[rng.standard_normal()]) for size in sizes for row in range(size)]
    check(lp, records, 53)
    rec = record_of(m, 900, records, 53)
    plan = gp_ffi.PostsolvePlan(rec, original=lp)
    assert plan.shape()["dual_levels"] == len(sizes)
    plan.free()


def disjoint_rows(m, k):
    """An LP whose row r holds the columns k r .. k r + k - 1, all at 1 there."""
    rng = np.random.default_rng(m)
    rows, cols = np.repeat(np.arange(m), k), np.arange(m * k)
    vals = rng.choice([-2.0, -0.5, 0.5, 2.0], m * k) * (1.0 + rng.random(m * k) * 2.0 ** -20)
    ptr, idx, val = lp_synth.csr_from_coo(m, m * k, rows, cols, vals)
    tptr, tidx, tval = lp_synth.transpose_csr(m, m * k, ptr, idx, val)
    n = m * k
    return dict(m=m, n=n, A_ptr=ptr, A_idx=idx, A_val=val, AT_ptr=tptr, AT_idx=tidx, AT_val=tval, c=rng.standard_normal(n),
                l=np.zeros(n), u=np.full(n, INF), AL=np.full(m, -INF), AU=np.full(m, 1e6), obj=0.0)


# line records (bound changes: a row of four entries each), then the others (type 10 on further rows) of a level
MIXED = [(1, 0), (1, 1), (3, 5), (4, 60), (5, 64), (16, 65), (59, 64), (60, 64), (60, 65), (61, 64), (63, 1), (64, 0),
         (64, 1), (64, 1024), (64, 1100), (1, 960), (1, 961), (4, 1025), (65, 0), (65, 700), (2, 2048), (2, 2049), (64, 64)]


def test_levels_of_both_kinds():
    m, k = 2200, 4
    lp = disjoint_rows(m, k)
    rng = np.random.default_rng(71)
    records = []
    for level, (lines, others) in enumerate(MIXED):
        for r in range(lines):
            records.append((12, np.r_[r * k + level % k, r], np.r_[0.0, INF, 1.0, INF]))
        for r in range(100, 100 + others):
            records.append((10, np.r_[r], np.r_[rng.standard_normal()]))
        records.append((10, np.r_[0], np.r_[0.25]))  # ties the next level's rows to this one's
    rec = record_of(lp["m"], lp["n"], records, 72)
    rec.update(n1=lp["n"], col_red2org=np.arange(lp["n"], dtype=np.int32), fixed_idx=np.zeros(0, np.int32),
               fixed_val=np.zeros(0))
    point = (np.ones(lp["n"]), rng.standard_normal(m), rng.standard_normal(lp["n"]))
    want = O.postsolve(rec, *point, original=lp)
    got = gp_ffi.postsolve(rec, *point, original=lp)
    for name, a, b in zip("xyz", got, want):
        assert_same_array(name, a, b)


@pytest.mark.parametrize("kind", ["simple", "line", "in-turn"])
def test_chains_of_single_records(kind):
    lp = disjoint_rows(50, 4)
    rng = np.random.default_rng(81)
    line = [(12, np.r_[q % 4, 0], np.r_[0.0, INF, 1.0, INF]) for q in range(700)]
    simple = [(10, np.r_[0], np.r_[rng.standard_normal()]) for _ in range(700)]
    records = {"simple": simple, "line": line, "in-turn": [r for pair in zip(line, simple) for r in pair]}[kind]
    rec = record_of(lp["m"], lp["n"], records, 82)
    rec.update(n1=lp["n"], col_red2org=np.arange(lp["n"], dtype=np.int32), fixed_idx=np.zeros(0, np.int32),
               fixed_val=np.zeros(0))
    point = (np.ones(lp["n"]), rng.standard_normal(50), rng.standard_normal(lp["n"]))
    want = O.postsolve(rec, *point, original=lp)
    got = gp_ffi.postsolve(rec, *point, original=lp)
    for name, a, b in zip("xyz", got, want):
        assert_same_array(name, a, b)


def test_records_without_rows():
    """No rows and no original model: every record is a lane's, but for the
    substituted columns' primal."""
    n = 3000
    rng = np.random.default_rng(91)
    f = lambda size=None: rng.choice([-2.0, -1.0, -0.5, 0.5, 1.0, 2.0], size) * (1 + rng.random(size) * 2.0 ** -20)
    records = []
    for _ in range(900):
        t, cols = int(rng.choice([0, 1, 2, 3, 13, 14])), rng.choice(n, size=20, replace=False)
        if t == 0:
            records.append((0, cols[:1], np.r_[1.0, f()]))
        elif t == 1:
            records.append((1, np.r_[0, cols[0], 2, cols[:2]], np.r_[1.0, 0.5, 1.0, f(2)]))
        elif t == 2:
            records.append((2, np.r_[cols[0], -1, 17, cols[3:]], np.r_[f(), 1.0, 0.0, 0.0, f(), 1.0, f(17) / 64]))
        elif t == 3:
            records.append((3, cols[:2], np.r_[f(), 0.0, 1.0, -1.0, INF]))
        elif t == 13:
            records.append((13, np.r_[cols[:2], -1], np.r_[4.0, f(), 1.0, 0.0, 0.0, 0.0, 4.0, 0.5, 2.0, f()]))
        else:
            records.append((14, np.r_[0, cols[0], 0, cols[1:3]], np.r_[1.0, f(), 2.0, 0.25, rng.standard_normal(2) / 64]))
    rec = record_of(0, n, records, 92)
    point = (rng.integers(0, 2, rec["n1"]).astype(float), np.zeros(0), rng.standard_normal(rec["n1"]))
    with np.errstate(all="ignore"):
        want = O.postsolve(rec, *point)
    assert all(np.isfinite(w).all() for w in want)
    got = gp_ffi.postsolve(rec, *point)
    for name, a, b in zip("xyz", got, want):
        assert_same_array(name, a, b)
