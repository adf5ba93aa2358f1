"""GPU parity of the look-through solve (CAP_ALGO_HOP, k_hop).

Every row, also one computed a second time by a row that looks through it,
is the stored-order chain of the thread-per-row kernels, so x must equal the
oracle's bits and the plain write-first plan's, in both arithmetics and both
precisions.  The number of waits is restated here from the rows.
"""
import numpy as np
import pytest

import oracle
from capellinisptrsv_amd import api, _native
from conftest import drop_diagonal, random_lower, upper_from_lower

pytestmark = pytest.mark.gpu


def hops_of(rp, ci):
    """hop(i) = 1 + max over entries c of min(hop(c), max of hop over c's entries)."""
    n = len(rp) - 1
    hop, look = [0] * n, [0] * n
    for i in range(n):
        cs = ci[rp[i]:rp[i + 1] - 1]
        hop[i] = 1 + max((min(hop[c], look[c]) for c in cs), default=0)
        look[i] = max((hop[c] for c in cs), default=0)
    return max(hop)


def _mats():
    # edges of the wavefront and of both workgroup sizes' tickets; 2, 3 and 4
    # entries per row; duplicates, unsorted rows
    for n in (1, 2, 63, 64, 65, 127, 128, 129, 255, 256, 257, 1000):
        yield f"n{n}", random_lower(n, max_off=2 + n % 3, band=40, seed=n, dup=False)
    yield "dup", random_lower(3000, max_off=3, band=500, seed=2, dup=True)
    yield "shuffled", random_lower(3000, max_off=4, band=90, seed=3, shuffle=True)
    yield "diagonal", random_lower(300, max_off=0, seed=4)
    yield "chain", api.generate("band", n=700, offdiag=1, band=1, seed=5)
    yield "wide", api.make_config(1, seed=6, scale=0.05)
    yield "level_o4", api.generate("level", n=30000, levels=30, width=1000, depth=3, offdiag=4, seed=7)


MATS = [(name, m) for name, m in _mats() if np.diff(m[0]).max() <= 5]


def _plan(cuda, rp, ci, v, **kw):
    import torch
    from capellinisptrsv_amd import Plan
    return Plan(*(torch.from_numpy(np.ascontiguousarray(a)).to(cuda) for a in (rp, ci, v)), **kw)


def _run(plan, cuda, b):
    import torch
    x = plan.solve(torch.from_numpy(np.ascontiguousarray(b)).to(cuda))
    torch.cuda.synchronize()
    assert plan.status() == 0
    return x.cpu().numpy()


@pytest.mark.parametrize("threads", [128, 256])
@pytest.mark.parametrize("name,mat", MATS, ids=[m[0] for m in MATS])
def test_hop_bit_exact(cuda, name, mat, threads):
    rp, ci, v = mat
    n = len(rp) - 1
    for dtype, bits in ((np.float64, np.uint64), (np.float32, np.uint32)):
        vt, b = v.astype(dtype), api.uniform(21, n).astype(dtype)
        for arith, fused in (("fused", True), ("reference", False)):
            plan = _plan(cuda, rp, ci, vt, algo="hop", row_threads=threads, arith=arith)
            assert plan.hops() == hops_of(rp, ci)
            x = _run(plan, cuda, b)
            assert np.array_equal(x.view(bits), oracle.csr_forward(rp, ci, vt, b, fused=fused).view(bits)), (name, dtype)
            assert np.array_equal(_run(plan, cuda, b).view(bits), x.view(bits))  # again on the same plan
            plan.close()


@pytest.mark.parametrize("kind", ["upper", "unit", "upper_unit"])
def test_hop_triangular_kinds(cuda, kind):
    """Rows are reversed inside the kernel (no copies of b and x): the
    oracle's bits, also through reset / launch."""
    import torch
    rp, ci, v = random_lower(2500, max_off=4, band=300, seed=8, dup=False)
    upper, unit = kind != "unit", kind != "upper"
    if upper:
        rp, ci, v = upper_from_lower(rp, ci, v)
    if unit:
        rp, ci, v = drop_diagonal(rp, ci, v, upper=upper)
    n = len(rp) - 1
    plan = _plan(cuda, rp, ci, v, algo="hop", upper=upper, unit_diagonal=unit)
    b = api.uniform(22, n)
    ref = oracle.csr_solve(rp, ci, v, b, upper=upper, unit=unit, fused=True)
    assert np.array_equal(_run(plan, cuda, b).view(np.uint64), ref.view(np.uint64))
    d, x = torch.from_numpy(b).to(cuda), torch.zeros(n, dtype=torch.float64, device=cuda)
    plan.reset(x)
    plan.launch(d, x)
    assert plan.status() == 0
    assert np.array_equal(x.cpu().numpy().view(np.uint64), ref.view(np.uint64))
    # several right-hand sides go through the write-first kernel
    bk = api.uniform(23, n * 3).reshape(n, 3)
    xk = _run(plan, cuda, bk)
    for q in range(3):
        refq = oracle.csr_solve(rp, ci, v, np.ascontiguousarray(bk[:, q]), upper=upper, unit=unit, fused=True)
        assert np.array_equal(xk[:, q], refq)
    plan.close()


def test_upper_launch_without_reset_is_refused(cuda):
    """As for the other kernels of upper-triangular plans: a launch that no
    reset or solve came before is an argument error."""
    import torch
    rp, ci, v = upper_from_lower(*random_lower(500, max_off=3, band=100, seed=12, dup=False))
    b = torch.from_numpy(api.uniform(28, 500)).to(cuda)
    x = torch.zeros_like(b)
    for algo in ("wrtfst", "hop"):
        plan = _plan(cuda, rp, ci, v, algo=algo, upper=True)
        with pytest.raises(_native.CapError, match=str(_native.CAP_ERR_ARG)):
            plan.launch(b, x)
        plan.reset(x)
        plan.launch(b, x)
        assert np.array_equal(x.cpu().numpy(), oracle.csr_solve(rp, ci, v, b.cpu().numpy(), upper=True, fused=True))
        plan.close()


def test_hop_reads_the_callers_values_and_special_values(cuda):
    """The tables hold the pattern only: values changed in place between two
    solves count.  Infinities, NaN and the sentinel's own bits in b spread
    like in the write-first kernel."""
    import torch
    from capellinisptrsv_amd import Plan
    rp, ci, v = random_lower(2000, max_off=3, band=200, seed=9)
    d = [torch.from_numpy(a).to(cuda) for a in (rp, ci, v)]
    plan = Plan(*d, algo="hop")
    b = api.uniform(24, 2000)
    assert np.array_equal(_run(plan, cuda, b), oracle.csr_forward(rp, ci, v, b, fused=True))
    d[2].mul_(1.5)
    assert np.array_equal(_run(plan, cuda, b), oracle.csr_forward(rp, ci, v * 1.5, b, fused=True))
    b[3], b[700], b[1400] = np.inf, np.nan, np.array([0xFFF0000000000001], np.uint64).view(np.float64)[0]
    plain = Plan(*d, algo="wrtfst")
    x, ref = _run(plan, cuda, b), _run(plain, cuda, b)
    assert np.array_equal(x, ref, equal_nan=True) and np.isnan(x).any() and np.isinf(x).any()
    plan.close()
    plain.close()


def test_hop_refusals_and_replay(cuda):
    import torch
    rp, ci, v = random_lower(400, max_off=5, band=100, seed=10)
    assert np.diff(rp).max() == 6
    for kw in (dict(), dict(sync="flag"), dict(readiness="in_place"), dict(lds_window=True), dict(row_tiles=True)):
        with pytest.raises(_native.CapError):
            m = (rp, ci, v) if not kw else random_lower(400, max_off=3, band=100, seed=10)
            _plan(cuda, *m, algo="hop", **kw)
    rp, ci, v = api.make_config(1, seed=11, scale=0.02)
    n = len(rp) - 1
    plan = _plan(cuda, rp, ci, v, algo="hop")
    b = torch.from_numpy(api.uniform(25, n)).to(cuda)
    eager = plan.solve(b).clone()
    out = torch.empty_like(b)
    from test_gpu_capture import _replays
    _replays(lambda: plan.solve(b, out=out, stream=torch.cuda.current_stream()), out, eager)
    assert plan.status() == 0
    plan.close()


@pytest.mark.parametrize("threads", [128, 256])
@pytest.mark.parametrize("name,mat", MATS, ids=[m[0] for m in MATS])
def test_refined_sweep_bit_exact(cuda, name, mat, threads):
    """The refinement's first two steps over the same tables: the oracle's
    two-step result bit for bit (a looked-through row's pair is worked out
    again with the row's own operations)."""
    import torch
    rp, ci, v = mat
    n = len(rp) - 1
    plan = _plan(cuda, rp, ci, v, algo="hop", row_threads=threads)
    b = api.uniform(9, n)
    _, _, want = oracle.refine2(rp, ci, v, b, rhs=1, rcp=True)
    bt = torch.from_numpy(b).to(cuda)
    out = torch.empty_like(bt)
    for rep in range(2):  # the second call replays the captured graph
        x, iters, rel = plan.solve_refined(bt, tol=1e-9, out=out)
        torch.cuda.synchronize()
        assert plan.status() == 0
        assert iters == 2, (rep, iters, rel)
        assert np.array_equal(x.cpu().numpy(), want), rep
    plan.close()


def _same_samples(a, b):
    """Equal in what the autotuner's cache key holds of the pattern."""
    at = [[(len(x) - 1) * s // 256 for s in range(257)] for x in a[:2]]
    return (all(len(x) == len(y) and np.array_equal(x[i], y[i]) for x, y, i in zip(a, b, at)) and
            oracle.row_levels(len(a[0]) - 1, *a[:2]).max() == oracle.row_levels(len(b[0]) - 1, *b[:2]).max())


def _longer_row(rp, ci, v):
    """Four neighbouring rows of two entries each become rows of 5, 1, 1, 1."""
    n = len(rp) - 1
    used = {(n) * s // 256 for s in range(257)}
    for i in range(n // 2, n - 4):
        if (np.diff(rp[i:i + 5]) == 3).all() and not used & set(range(i, i + 5)):
            rows = [list(ci[rp[r]:rp[r + 1] - 1]) for r in range(i, i + 4)]
            five = sorted(rows[0] + rows[1][1:] + rows[2][1:] + rows[3][1:])
            new = [five + [i]] + [[rows[t][0], i + t] for t in (1, 2, 3)]
            rp2, ci2 = rp.copy(), ci.copy()
            ci2[rp[i]:rp[i + 4]] = np.concatenate(new)
            rp2[i + 1:i + 5] = rp[i] + np.cumsum([len(r) for r in new])
            v2 = v.copy()
            v2[rp2[i + 1:i + 5] - 1] = 6.0
            if five[-1] < i and len(set(five)) == 5 and _same_samples((rp, ci, v), (rp2, ci2, v2)):
                return rp2, ci2, v2
    raise AssertionError("no place found")


def _far_column(rp, ci, v):
    """One entry of a row in the last tenth moves to the first column."""
    n = len(rp) - 1
    for i in range(n * 9 // 10, n):
        if rp[i + 1] - rp[i] == 4:
            ci2 = ci.copy()
            ci2[rp[i]] = 0
            if _same_samples((rp, ci, v), (rp, ci2, v)):
                return rp, ci2, v
    raise AssertionError("no place found")


@pytest.mark.parametrize("kind", ["hop", "level"])
def test_cached_pick_that_does_not_fit_is_tuned_afresh(cuda, kind):
    """The autotuner's cache knows a pattern by samples: a matrix with a row
    too long for the look-through tables, or with an entry beyond the steps'
    ring, may be taken for one that has neither."""
    if kind == "hop":
        first = api.generate("level", n=100_000, levels=20, width=5000, depth=3, offdiag=2, seed=31)
        second = _longer_row(*first)
        assert np.diff(first[0]).max() == 3 and np.diff(second[0]).max() == 6
    else:
        first = api.generate("band", n=100_000, offdiag=3, band=1000, seed=32)
        second = _far_column(*first)
    n = len(first[0]) - 1
    b = api.uniform(26, n)
    plan = _plan(cuda, *first)
    assert plan.hops() > 0 if kind == "hop" else plan.info()["algo"] == "level"
    for m in (second, first):
        other = _plan(cuda, *m)
        assert np.array_equal(_run(other, cuda, b), oracle.csr_forward(*m, b, fused=True))
        other.close()
    plan.close()


@pytest.mark.parametrize("call", ["solve", "refined"])
def test_spin_limit_counts_polls_without_progress(cuda, call):
    """A chain whose rows also read the rows at 1/4, 1/2 and 3/4 of the way
    sees a value arrive in every quarter of its wait; one whose other entries
    are the first rows waits all along for the last.  Bounded in polls without
    progress, the first needs about a quarter of the second's limit (bar: 0.6,
    between the 0.25 and the 1 of a bound on all of a row's polls)."""
    import torch
    n = 1536

    def chain(spread):
        rp, ci = [0], []
        for i in range(n):
            cs = {i - 1, 3 * i // 4, i // 2, i // 4} if spread else {i - 1, 0, 1, 2}
            ci += sorted(c for c in cs if 0 <= c < i) + [i]
            rp.append(len(ci))
        rp, ci = np.array(rp, np.int32), np.array(ci, np.int32)
        return rp, ci, np.where(ci == np.repeat(np.arange(n), np.diff(rp)), 4.0, 0.5)

    b = torch.from_numpy(api.uniform(27, n)).to(cuda)

    def ends(mat, limit):
        plan = _plan(cuda, *mat, algo="hop", spin_limit=limit)
        ok = []
        for _ in range(3):
            if call == "solve":
                plan.solve(b)
            else:
                try:
                    plan.solve_refined(b, tol=1e-9)
                except _native.CapError:
                    pass
            ok.append(plan.status() == 0)
        plan.close()
        return all(ok)

    def least(mat):
        lo, hi = 1.0, 2.0 ** 17
        assert ends(mat, int(hi))
        while hi > 1.1 * lo:
            mid = (lo * hi) ** 0.5
            lo, hi = (lo, mid) if ends(mat, int(mid)) else (mid, hi)
        return hi

    assert least(chain(True)) <= 0.6 * least(chain(False))


def test_refined_solves_of_many_plans_keep_their_norms_apart(cuda):
    """The pinned words that the norms are read from pass from freed plans to
    new ones, and more plans than are kept hold words at once."""
    import torch
    mats = [random_lower(300 + 7 * i, max_off=3, band=100, seed=60 + i) for i in range(20)]
    for _ in range(2):
        plans = [_plan(cuda, *m, algo="hop") for m in mats]
        for rep in range(2):
            for i, (plan, m) in enumerate(zip(plans, mats)):
                b = api.uniform(70 + i + 20 * rep, len(m[0]) - 1)
                x0, d, want = oracle.refine2(*m, b, rhs=1, rcp=True)
                x, iters, rel = plan.solve_refined(torch.from_numpy(b).to(cuda), tol=1e-9)
                assert iters == 2 and np.array_equal(x.cpu().numpy(), want)
                assert rel == float(np.abs(d).max()) / float(np.abs(x0).max())
        for plan in plans:
            plan.close()
