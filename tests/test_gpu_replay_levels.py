"""Tapes written by hand for the postsolve replay, against the oracle's
record-by-record replay, bit for bit: lines around the 16 and 32 entries that
are loaded ahead, every record type in one level, levels around the 64 slots
of the workgroup and around the size that takes a launch of its own."""
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


def test_levels_around_the_slots_and_the_launch_of_their_own():
    lp = original(700, 900, 51)
    rng = np.random.default_rng(52)
    sizes = [1, 3, 4, 5, 15, 16, 17, 63, 64, 65, 127, 128, 129, 510, 511, 512, 513, 600]
    records = [(10, np.r_[row], np.r_[rng.standard_normal()]) for size in sizes for row in range(size)]
    check(lp, records, 53)
    rec = record_of(700, 900, records, 53)
    plan = gp_ffi.PostsolvePlan(rec, original=lp)
    assert plan.shape()["dual_levels"] == len(sizes)
    plan.free()
