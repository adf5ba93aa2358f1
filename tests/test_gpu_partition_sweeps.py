"""GPU tests of the partitioned solve's sweeps and of both ways its tails are
joined: walked (blocks that damp their history, or few of them) and scanned.

Sizes: a last record and a last block of one row, rows of more than one
segment (16, 32 and 48 entries), rows of no entries, duplicated entries past
what a record holds, and blocks that are made longer because they damp too
little.  Bars: relative max-norm 1e-12 against the oracle's sequential forward
substitution, as for every FP64 partitioned solve; for a right-hand side that
is zero but for one row, whose solution falls off by hundreds of orders of
magnitude, each value that is a normal number is not lost (the sums' order
differs, so the bar is on its size: a factor of 2).
"""
import numpy as np
import pytest

import oracle
from capellinisptrsv_amd import api
from conftest import rel_maxnorm

pytestmark = pytest.mark.gpu

FP64_TOL = 1e-12


def _band(n, w, p, seed, positive=False):
    """Entries of each row's previous w columns with probability p, values
    U[-1,1] or U[0,1], diagonal 1 + the sum of their magnitudes."""
    rng = np.random.default_rng(seed)
    keep = rng.random((n, w)) < p
    keep &= np.arange(n)[:, None] - 1 - np.arange(w) >= 0
    count = keep.sum(1)
    rp = np.r_[0, np.cumsum(count + 1)].astype(np.int32)
    ci = np.empty(rp[-1], np.int32)
    v = np.empty(rp[-1])
    last = rp[1:] - 1
    off = np.ones(rp[-1], bool)
    off[last] = False
    rows, back = np.nonzero(keep[:, ::-1])
    ci[off] = rows - w + back
    v[off] = rng.uniform(0.0 if positive else -1.0, 1.0, off.sum())
    ci[last] = np.arange(n)
    v[last] = 0.0
    v[last] = 1.0 + np.add.reduceat(np.abs(v), rp[:-1])
    return rp, ci, v


def _many_duplicates(n):
    """Rows whose one column is stored 400 times."""
    rng = np.random.default_rng(3)
    rp, ci, v = [0], [], []
    for i in range(n):
        if i % 50 == 7:
            ci += [i - 3] * 400
            v += list(rng.uniform(-1, 1, 400) / 400)
        elif i:
            ci.append(i - 1)
            v.append(0.3)
        ci.append(i)
        v.append(1.5)
        rp.append(len(ci))
    return np.array(rp, np.int32), np.array(ci, np.int32), np.array(v)


CASES = {
    "walk_last_row_alone": lambda: _band(16 * 512 + 1, 40, 0.3, 1),   # a last block of one row
    "walk_16_entries": lambda: _band(9001, 32, 0.5, 2),
    "walk_one_segment_or_two": lambda: _band(20_003, 96, 0.34, 4),     # about 32 entries
    "walk_wide": lambda: _band(12_000, 250, 0.2, 5),
    "walk_no_entries": lambda: _band(15_000, 30, 0.02, 6),
    "walk_longer_blocks": lambda: _band(40_000, 128, 0.15, 7),
    "scan": lambda: _band(30_000, 120, 0.3, 8, positive=True),
    "scan_wide": lambda: _band(24_000, 200, 0.1, 9, positive=True),
    "duplicates": lambda: _many_duplicates(6000),
}


def _plan(cuda, mat):
    import torch
    from capellinisptrsv_amd import Plan
    return Plan(*(torch.from_numpy(a).to(cuda) for a in mat), algo="partition")


@pytest.mark.parametrize("name", CASES)
def test_sweeps_match_the_oracle(cuda, name):
    import torch
    mat = CASES[name]()
    n = len(mat[0]) - 1
    plan = _plan(cuda, mat)
    one = None
    for k in (1, 8, 12):
        b = api.uniform(50, n * 12).reshape(n, 12)[:, :k].copy()
        bt = torch.from_numpy(b[:, 0].copy() if k == 1 else b).to(cuda)
        x = plan.solve(bt).cpu().numpy().reshape(n, k)
        ref = oracle.csr_forward(*mat, b.reshape(-1), rhs=k, fused=True).reshape(n, k)
        for q in range(k):
            assert rel_maxnorm(x[:, q], ref[:, q]) <= FP64_TOL, (k, q)
        one = x[:, 0] if one is None else one
        assert np.array_equal(x[:, 0], one), k  # the same bits whatever is solved beside it
        assert torch.equal(plan.solve(bt, out=bt).cpu(), torch.from_numpy(x.reshape(bt.shape)))  # x in b's place
    plan.close()


def _reached(rp, ci, row):
    """Which rows depend on `row` (itself among them)."""
    hit = np.zeros(len(rp) - 1, bool)
    hit[row] = True
    for i in range(row + 1, len(hit)):
        hit[i] = hit[ci[rp[i]:rp[i + 1] - 1]].any()
    return hit


@pytest.mark.parametrize("name", ["walk_16_entries", "scan"])
@pytest.mark.parametrize("value", [np.inf, np.nan])
def test_an_infinity_reaches_the_rows_that_depend_on_it(cuda, name, value):
    import torch
    mat = CASES[name]()
    n = len(mat[0]) - 1
    plan = _plan(cuda, mat)
    row = n // 3
    b = api.uniform(51, n)
    want = oracle.csr_forward(*mat, b, fused=True)
    b[row] = value
    x = plan.solve(torch.from_numpy(b).to(cuda)).cpu().numpy()
    hit = _reached(mat[0], mat[1], row)
    assert rel_maxnorm(x[:row], want[:row]) <= FP64_TOL
    assert not np.isfinite(x[hit]).any()
    plan.close()


@pytest.mark.parametrize("name", ["walk_16_entries", "walk_one_segment_or_two"])
def test_one_nonzero_row(cuda, name):
    """No part of the solution is dropped: the tails are followed as far back
    as a double reaches."""
    import torch
    mat = CASES[name]()
    n = len(mat[0]) - 1
    plan = _plan(cuda, mat)
    b = np.zeros(n)
    b[100] = 1.0
    want = oracle.csr_forward(*mat, b, fused=True)
    x = plan.solve(torch.from_numpy(b).to(cuda)).cpu().numpy()
    assert rel_maxnorm(x, want) <= FP64_TOL
    far = 0
    for lo in range(0, n - 512, 512):  # a stretch's size, where it is a normal number
        a, w = np.abs(x[lo:lo + 512]).max(), np.abs(want[lo:lo + 512]).max()
        if w > 1e-290:
            assert 0.5 * w <= a <= 2.0 * w, lo
            far = lo
    assert far > 2000
    # beside others, dense ones and ones with nonzeros elsewhere: the same bits
    beside = np.zeros((n, 8))
    beside[:, 2] = beside[:, 7] = api.uniform(52, n)
    beside[[n // 2, n // 2 + 300, n - 5], 3] = 1.0
    beside[5, 4] = 1e-200
    for at, col in ((0, 0), (6, 0), (1, 1)):
        beside[100 + col, at] = 1.0
    xs = plan.solve(torch.from_numpy(beside).to(cuda)).cpu().numpy()
    assert np.array_equal(xs[:, 0], x) and np.array_equal(xs[:, 6], x)
    for q in range(8):
        alone = plan.solve(torch.from_numpy(beside[:, q].copy()).to(cuda)).cpu().numpy()
        assert np.array_equal(xs[:, q], alone), q
        ref = oracle.csr_forward(*mat, beside[:, q].copy(), fused=True)
        assert rel_maxnorm(xs[:, q], ref) <= FP64_TOL, q
    plan.close()


@pytest.mark.parametrize("huge", [1e6, 1e25])
def test_a_huge_row_does_not_reach_rows_that_do_not_depend_on_it(cuda, huge):
    """Even and odd rows are systems of their own, and even rows of b at the
    blocks' ends are huge: the odd rows keep the accuracy they have without."""
    import torch
    n, w = 100_000, 50
    rng = np.random.default_rng(5)
    rows = np.repeat(np.arange(n), 2)
    cols = rows - 2 * rng.integers(w - 10, w + 1, len(rows))
    key = np.unique(rows[cols >= 0] * np.int64(n) + cols[cols >= 0])
    rp = np.r_[0, np.cumsum(np.bincount(key // n, minlength=n) + 1)].astype(np.int32)
    ci, v = np.empty(rp[-1], np.int32), np.empty(rp[-1])
    at = np.arange(len(key)) + key // n
    ci[at], v[at] = key % n, rng.uniform(0.5, 1.0, len(key))
    ci[rp[1:] - 1], v[rp[1:] - 1] = np.arange(n), 4.5
    plan = _plan(cuda, (rp, ci, v))
    b = api.uniform(3, n)
    b[np.arange(500, n, 1000) // 2 * 2] = huge
    x = plan.solve(torch.from_numpy(b).to(cuda)).cpu().numpy()
    want = oracle.csr_forward(rp, ci, v, b, fused=True)
    assert rel_maxnorm(x, want) <= FP64_TOL
    assert rel_maxnorm(x[1::2], want[1::2]) <= FP64_TOL
    plan.close()


def test_a_system_whose_right_hand_side_ends_is_not_cut_off(cuda):
    """Even and odd rows are systems of their own; the odd rows of b are zero
    after the first 500, those of x fall off from there.  Off-diagonals are
    negative and b is not, so every sum is of one sign and each value is held
    by itself: down to 1e-290, 4 roundings a row over a chain of 660 and sums of
    64 in each of 106 blocks (of 500 rows or more) are below 2e-12."""
    import torch
    n, w = 100_000, 50
    rng = np.random.default_rng(5)
    rows = np.repeat(np.arange(n), 2)
    cols = rows - 2 * rng.integers(w - 10, w + 1, len(rows))
    key = np.unique(rows[cols >= 0] * np.int64(n) + cols[cols >= 0])
    rp = np.r_[0, np.cumsum(np.bincount(key // n, minlength=n) + 1)].astype(np.int32)
    ci, v = np.empty(rp[-1], np.int32), np.empty(rp[-1])
    at = np.arange(len(key)) + key // n
    ci[at], v[at] = key % n, -rng.uniform(0.5, 1.0, len(key))
    ci[rp[1:] - 1], v[rp[1:] - 1] = np.arange(n), 4.5
    plan = _plan(cuda, (rp, ci, v))
    b = 0.1 + np.abs(api.uniform(3, n))
    b[501::2] = 0.0
    x = plan.solve(torch.from_numpy(b).to(cuda)).cpu().numpy()
    want = oracle.csr_forward(rp, ci, v, b, fused=True)
    seen = want > 1e-290
    assert seen[1::2].sum() > 5_000 and (want[1::2] < 1e-100).any()
    assert (np.abs(x - want)[seen] <= 2 * FP64_TOL * want[seen]).all()
    plan.close()
