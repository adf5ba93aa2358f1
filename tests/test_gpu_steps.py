"""GPU parity of the step solve (steps.hip) where the level rule of explicit
CAP_ALGO_LEVEL plans does not reach: autotuned plans over matrices whose
first levels lie all over the rows, rows longer than the 16 entries a step
carries, any number of right-hand sides, batches, and the division by a
table reciprocal at the ends of its range.  Bar: the oracle's bits.
"""
import numpy as np
import pytest

import oracle
from capellinisptrsv_amd import api
from conftest import random_lower

pytestmark = pytest.mark.gpu


def _plan(cuda, rp, ci, v, **kw):
    import torch
    from capellinisptrsv_amd import Plan
    return Plan(*(torch.from_numpy(np.ascontiguousarray(a)).to(cuda) for a in (rp, ci, v)), **kw)


def _solve(plan, cuda, b):
    import torch
    x = plan.solve(torch.from_numpy(np.ascontiguousarray(b)).to(cuda))
    torch.cuda.synchronize()
    assert plan.status() == 0
    return x.cpu().numpy()


def _ragged(n=6001, off=16, band=400, seed=3):
    return api.generate("band_rowcount", n=n, offdiag=off, band=band, seed=seed)


@pytest.mark.parametrize("dtype,bits", [(np.float64, np.uint64), (np.float32, np.uint32)])
@pytest.mark.parametrize("off", [4, 8, 16, 40])
def test_autotuned_steps_bit_exact(cuda, off, dtype, bits):
    """4, 8 and 16 carried entries, and rows of up to 39 (the rest read from
    the overflow table); thread-per-row kernels take about 5 x as long here."""
    rp, ci, v = _ragged(off=off, seed=off)
    v = v.astype(dtype)
    n = len(rp) - 1
    for arith, fused in (("fused", True), ("reference", False)):
        plan = _plan(cuda, rp, ci, v, arith=arith)
        if off != 40:
            assert plan.info()["algo"] == "level"
        for k in (1, 2, 3, 16):
            b = api.uniform(5 + k, n * k).astype(dtype).reshape(n, k) if k > 1 else api.uniform(5, n).astype(dtype)
            x = _solve(plan, cuda, b)
            ref = oracle.csr_forward(rp, ci, v, b.reshape(-1), rhs=k, fused=fused)
            assert np.array_equal(x.reshape(-1).view(bits), ref.view(bits)), (off, arith, k)
        plan.close()


def test_autotuned_steps_read_the_callers_values(cuda):
    """Where the explicit rule refuses the matrix the autotuned plan used to
    run kernels that read the caller's values on every solve; its steps do so
    too."""
    import torch
    from capellinisptrsv_amd import Plan
    rp, ci, v = _ragged(n=20001, seed=21)  # empty rows near the end: beyond that rule's ring
    d = [torch.from_numpy(a).to(cuda) for a in (rp, ci, v)]
    plan = Plan(*d)
    b = api.uniform(6, len(rp) - 1)
    assert np.array_equal(_solve(plan, cuda, b), oracle.csr_forward(rp, ci, v, b, fused=True))
    d[2].mul_(0.75)
    assert np.array_equal(_solve(plan, cuda, b), oracle.csr_forward(rp, ci, v * 0.75, b, fused=True))
    plan.close()


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_autotuned_steps_read_values_where_the_rule_accepts(cuda, dtype):
    """The same on bands that explicit level plans take, for every number of
    right-hand sides, and through the module whose values an optimizer
    changes."""
    import torch
    from capellinisptrsv_amd import Plan
    from capellinisptrsv_amd.torch_ops import TriangularSolve
    rp, ci, v = api.generate("band", n=5000, offdiag=8, band=400, seed=23)  # beyond the partition's bandwidth
    v = v.astype(dtype)
    n = len(rp) - 1
    _plan(cuda, rp, ci, v, algo="level").close()  # accepted
    d = [torch.from_numpy(a).to(cuda) for a in (rp, ci, v)]
    plan = Plan(*d)
    assert plan.info()["algo"] == "level"
    module = TriangularSolve(d[0], d[1], d[2].clone())
    assert module.plan.info()["algo"] == "level"
    scale = 1.0
    for _ in range(2):
        vs = v * dtype(scale)
        for k in (1, 2, 3, 8):
            b = api.uniform(30 + k, n * k).astype(dtype).reshape(n, k) if k > 1 else api.uniform(30, n).astype(dtype)
            ref = oracle.csr_forward(rp, ci, vs, b.reshape(-1), rhs=k, fused=True)
            assert np.array_equal(_solve(plan, cuda, b).reshape(-1), ref), (scale, k)
        x = module(torch.from_numpy(b[:, 0].copy()).to(cuda))
        ref = oracle.csr_forward(rp, ci, vs, b[:, 0].copy(), fused=True)
        assert np.array_equal(x.detach().cpu().numpy(), ref), scale
        d[2].mul_(0.75)
        with torch.no_grad():
            module.values.mul_(0.75)
        scale *= 0.75
    plan.close()


@pytest.mark.parametrize("width", [40, 150, 240])
def test_cached_pick_keeps_its_rows_per_step(cuda, width):
    """A second plan of a pattern schedules for the first one's rows per step
    alone; a matrix taken for it by the cache's samples solves all the same."""
    rp, ci, v = api.generate("level", n=6000, levels=6000 // width, width=width, depth=2, offdiag=9, seed=width)
    n = len(rp) - 1
    b = api.uniform(9, n)
    ref = oracle.csr_forward(rp, ci, v, b, fused=True)
    widths = []
    for _ in range(3):
        plan = _plan(cuda, rp, ci, v)
        info = plan.info()
        assert info["algo"] == "level"
        widths.append(info["row_threads"])
        assert np.array_equal(_solve(plan, cuda, b), ref)
        plan.close()
    assert len(set(widths)) == 1
    assert _plan(cuda, rp, ci, v, algo="level").info()["row_threads"] == widths[0]


def test_autotuned_short_chains_follow_the_callers_values(cuda):
    """The partition holds the values of plan creation: on short chains, where
    it wins by little, auto keeps a kernel that reads them."""
    import torch
    from capellinisptrsv_amd import Plan
    rp, ci, v = api.generate("band_rowcount", n=20000, offdiag=3, band=120, seed=20120)  # 89 levels
    d = [torch.from_numpy(a).to(cuda) for a in (rp, ci, v)]
    plan = Plan(*d)
    assert plan.info()["algo"] != "partition"
    d[2].mul_(0.75)
    b = api.uniform(7, 20000)
    assert np.array_equal(_solve(plan, cuda, b), oracle.csr_forward(rp, ci, v * 0.75, b, fused=True))
    plan.close()


def test_autotuned_pick_is_timed_with_a_dense_right_hand_side(cuda):
    """A partitioned solve of b = 0 has no tails to join and takes half of
    what a dense b does (67 us here, against 36 by steps)."""
    rp, ci, v = api.generate("band", n=2000, offdiag=8, band=250, seed=2250)
    plan = _plan(cuda, rp, ci, v)
    assert plan.info()["algo"] == "level"
    b = api.uniform(8, 2000)
    assert np.array_equal(_solve(plan, cuda, b), oracle.csr_forward(rp, ci, v, b, fused=True))
    plan.close()


def _grid(nx, ny, nz):
    """The lower half of a 7-point stencil, natural order."""
    i = np.arange(nx * ny * nz)
    x, y, z = i % nx, i // nx % ny, i // (nx * ny)
    rows = np.concatenate([i[z > 0], i[y > 0], i[x > 0]])
    cols = np.concatenate([i[z > 0] - nx * ny, i[y > 0] - nx, i[x > 0] - 1])
    order = np.lexsort((cols, rows))
    rows, cols = rows[order], cols[order]
    rp = np.r_[0, np.cumsum(np.bincount(rows, minlength=len(i)) + 1)].astype(np.int32)
    ci = np.empty(rp[-1], np.int32)
    ci[np.arange(len(rows)) + rows], ci[rp[1:] - 1] = cols, i
    v = api.uniform(60, len(ci))
    v[rp[1:] - 1] = 4.0
    return rp, ci, v


SEVERAL = {
    "hop": lambda: _grid(30, 25, 20),                                                             # look-through, then rows
    "near_tie": lambda: api.generate("level", n=30_000, levels=50, width=600, depth=2, offdiag=9, seed=61),
    "steps": lambda: api.generate("band", n=5000, offdiag=8, band=400, seed=62),
}


@pytest.mark.parametrize("name", SEVERAL)
@pytest.mark.parametrize("upper", [False, True])
def test_several_right_hand_sides_of_hop_and_level_picks(cuda, name, upper):
    """Where one right-hand side goes by look-through tables or steps, several
    are timed as steps (near ties) and thread-per-row shapes: the oracle's
    bits from each, and after them."""
    from conftest import upper_from_lower
    rp, ci, v = SEVERAL[name]()
    if upper:
        rp, ci, v = upper_from_lower(rp, ci, v)
    n = len(rp) - 1
    plan = _plan(cuda, rp, ci, v, upper=upper)
    for k in (2, 3, 16, 64, 1, 16):
        b = api.uniform(70 + k, n * k).reshape(n, k) if k > 1 else api.uniform(70, n)
        x = _solve(plan, cuda, b).reshape(n, k)
        for q in range(0, k, 7):
            bq = np.ascontiguousarray(b.reshape(n, k)[:, q])
            assert np.array_equal(x[:, q], oracle.csr_solve(rp, ci, v, bq, upper=upper, fused=True)), (k, q)
    if not upper:
        b = api.uniform(71, n * 4).reshape(n, 4)
        import torch
        xr, _, _ = plan.solve_refined(torch.from_numpy(b).to(cuda), tol=1e-12)
        ref = oracle.csr_forward(rp, ci, v, b.reshape(-1), rhs=4, fused=True).reshape(n, 4)
        assert np.max(np.abs(xr.cpu().numpy() - ref)) <= 1e-12 * np.max(np.abs(ref))
    plan.close()


def test_level_pick_captures_a_first_solve(cuda):
    """The first solve with a number of right-hand sides may be a captured
    one: nothing is timed then, the steps run."""
    import torch
    rp, ci, v = SEVERAL["near_tie"]()
    n = len(rp) - 1
    plan = _plan(cuda, rp, ci, v)
    if plan.info()["algo"] != "level":
        pytest.skip("the tuner's pick is not the steps here")
    b = torch.from_numpy(api.uniform(72, n * 8).reshape(n, 8)).to(cuda)
    out = torch.zeros_like(b)
    side = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        plan.solve(b, out=out, stream=torch.cuda.current_stream())
    ref = oracle.csr_forward(rp, ci, v, b.cpu().numpy().reshape(-1), rhs=8, fused=True).reshape(n, 8)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(out.cpu().numpy(), ref)
        assert np.array_equal(plan.solve(b).cpu().numpy(), ref)  # timed now; the graph keeps what it holds
    plan.close()


@pytest.mark.parametrize("dtype,bits,span", [(np.float64, np.uint64, 620), (np.float32, np.uint32, 80)])
def test_step_division_range(cuda, dtype, bits, span):
    """Diagonals and right-hand sides over powers of two beyond both ends of
    the reciprocal's range, negative diagonals, zeros of both signs, the
    smallest numbers: the division's bits; infinities and NaN as the
    write-first kernel spreads them."""
    rng = np.random.default_rng(7)
    rp, ci, v = random_lower(4000, max_off=2, band=60, seed=8)
    n = len(rp) - 1
    v = v.astype(dtype)
    last = rp[1:] - 1
    off = np.ones(len(v), bool)
    off[last] = False
    v[off] = (rng.random(off.sum()) < 0.1) * v[off] * dtype(2.0) ** -3  # mostly independent rows
    v[last] = (rng.choice([-1, 1], n) * (1 + rng.random(n)) * 2.0 ** rng.integers(-span, span, n)).astype(dtype)
    b = ((1 + rng.random(n)) * 2.0 ** rng.integers(-span, span, n) * rng.choice([-1, 1], n)).astype(dtype)
    b[::17] = 0.0
    b[5::17] = -0.0
    b[9::17] = np.finfo(dtype).smallest_subnormal
    plan = _plan(cuda, rp, ci, v, algo="level")
    with np.errstate(all="ignore"):
        ref = oracle.csr_forward(rp, ci, v, b, fused=True)
    x = _solve(plan, cuda, b)
    ok = np.isfinite(ref)
    assert ok.sum() > n // 2
    assert np.array_equal(x[ok].view(bits), ref[ok].view(bits))
    assert np.array_equal(x, ref, equal_nan=True)
    b[3], b[500] = np.inf, np.nan
    plain = _plan(cuda, rp, ci, v, algo="wrtfst")
    assert np.array_equal(_solve(plan, cuda, b), _solve(plain, cuda, b), equal_nan=True)
    plan.close()
    plain.close()


@pytest.mark.parametrize("dtype,bits", [(np.float64, np.uint64), (np.float32, np.uint32)])
@pytest.mark.parametrize("extra", [0, 4, 8])
def test_unused_entries_keep_the_sign_of_a_zero_sum(cuda, extra, dtype, bits):
    """A product that underflows to -0 leaves the sum -0, and -0 - (-0) is +0:
    the entries a row does not have must not turn the sum into +0.  4, 8 and
    16 entries carried (`extra` more in the last row)."""
    n = 40
    tiny = np.finfo(dtype).tiny
    rp, ci, v = [0], [], []
    for i in range(n):
        cols = [i - 1] if i % 2 else []
        if i == n - 1:
            cols = list(range(i - 1 - extra, i))
        ci += cols + [i]
        v += [-float(tiny)] * len(cols) + [1.0 if i % 4 else -2.0]
        rp.append(len(ci))
    rp, ci, v = np.array(rp, np.int32), np.array(ci, np.int32), np.array(v, dtype)
    b = np.full(n, tiny, dtype)  # even rows: x = +-tiny, whose products with tiny underflow
    b[1::2] = dtype(-0.0)
    ref = oracle.csr_forward(rp, ci, v, b, fused=True)
    assert np.signbit(ref[1::2]).any() and not np.signbit(ref[1::2]).all()
    plan = _plan(cuda, rp, ci, v, algo="level")
    assert np.array_equal(_solve(plan, cuda, b).view(bits), ref.view(bits))
    plan.close()


def _batch(seed, sizes, off, band):
    mats = [api.generate("band_rowcount", n=n, offdiag=off, band=band, seed=seed + i) if n else
            (np.zeros(1, np.int32), np.zeros(0, np.int32), np.zeros(0)) for i, n in enumerate(sizes)]
    row_off = np.cumsum([0] + [len(m[0]) - 1 for m in mats]).astype(np.int32)
    nnz_off = np.cumsum([0] + [len(m[1]) for m in mats])
    rp = np.concatenate([m[0][:-1] + o for m, o in zip(mats, nnz_off)] + [[nnz_off[-1]]]).astype(np.int32)
    return mats, row_off, rp, np.concatenate([m[1] for m in mats]).astype(np.int32), np.concatenate([m[2] for m in mats])


@pytest.mark.parametrize("dtype,arith", [(np.float64, "fused"), (np.float32, "fused"), (np.float64, "reference")])
@pytest.mark.parametrize("k", [1, 3, 4, 16])
def test_batch_steps_bit_exact(cuda, k, dtype, arith):
    """Matrices from empty to 9,000 rows (fewer and more than the eight of a
    group), solved twice, and captured into a graph."""
    import torch
    from capellinisptrsv_amd import Batch
    from test_gpu_capture import _replays
    for sizes in ((9000, 0, 700, 1), tuple(2000 + 37 * i for i in range(19))):
        mats, row_off, rp, ci, v = _batch(50 + k, sizes, 16, 300)
        v = v.astype(dtype)
        N = int(row_off[-1])
        b = api.uniform(9 + k, N * k).astype(dtype)
        bt = Batch(*(torch.from_numpy(a).to(cuda) for a in (row_off, rp, ci, v)), k=k, arith=arith)
        assert bt.step_matrices == sum(n > 0 for n in sizes) and bt.partitioned == 0
        bd = torch.from_numpy(b.reshape(N, k)).to(cuda)
        x = bt.solve(bd)
        flat = x.cpu().numpy().reshape(-1)
        for m, (mrp, mci, mv) in enumerate(mats):
            lo, hi = row_off[m] * k, row_off[m + 1] * k
            if hi > lo:
                ref = oracle.csr_forward(mrp, mci, mv.astype(dtype), b[lo:hi], rhs=k, fused=arith == "fused")
                assert np.array_equal(flat[lo:hi], ref), m
        out = torch.empty_like(bd)
        _replays(lambda: bt.solve(bd, out=out, stream=torch.cuda.current_stream()), out, x)
        bt.close()


@pytest.mark.parametrize("dtype,bits", [(np.float64, np.uint64), (np.float32, np.uint32)])
@pytest.mark.parametrize("n,width", [(1, 1), (2, 1), (9, 1), (10, 1), (11, 1), (12, 1), (13, 1), (21, 1), (640, 63),
                                     (650, 65), (2000, 130), (3003, 250), (3000, 600)])
def test_loads_in_their_own_wavefronts(cuda, n, width, dtype, bits):
    """Up to 4 entries a row: step counts around the 10 steps that the loading
    wavefronts are ahead, odd and even, and steps of one to four wavefronts
    (rows of level l read level l - 1)."""
    rng = np.random.default_rng(n)
    rp, ci, v = [0], [], []
    for i in range(n):
        first = i // width * width
        if first:
            ci += sorted(rng.choice(np.arange(first - width, first), size=min(width, 1 + i % 4), replace=False))
        ci.append(i)
        v += list(rng.uniform(-1, 1, len(ci) - 1 - rp[-1])) + [3.0]
        rp.append(len(ci))
    rp, ci, v = np.array(rp, np.int32), np.array(ci, np.int32), np.array(v).astype(dtype)
    plan = _plan(cuda, rp, ci, v, algo="level")
    b = api.uniform(6, n).astype(dtype)
    for x in (_solve(plan, cuda, b) for _ in range(2)):
        ref = oracle.csr_forward(rp, ci, v, b, rhs=1, fused=True)
        assert np.array_equal(x.view(bits), ref.view(bits))
    plan.close()


def _long_rows(n, longest, seed):
    """Rows of 17 to `longest` entries in the 60 rows before them, and between
    them rows of one, so that levels follow the row order."""
    rng = np.random.default_rng(seed)
    rp, ci, v = [0], [], []
    for i in range(n):
        want = int(rng.integers(17, longest + 1)) if i % 3 == 0 else 1
        cols = sorted(i - 1 - rng.choice(min(60, i), size=min(want, i), replace=False)) if i else []
        ci += list(cols) + [i]
        v += list(rng.uniform(-1, 1, len(cols))) + [1.0 + longest]
        rp.append(len(ci))
    return np.array(rp, np.int32), np.array(ci, np.int32), np.array(v)


@pytest.mark.parametrize("dtype,bits", [(np.float64, np.uint64), (np.float32, np.uint32)])
@pytest.mark.parametrize("arith", ["fused", "reference"])
def test_rows_beyond_the_carried_entries(cuda, arith, dtype, bits):
    """Rows of 17 to 39 entries: 16 in the step's pieces, the rest from the
    overflow table, read behind them in the stored order."""
    rp, ci, v = _long_rows(3000, 39, 80)
    v = v.astype(dtype)
    assert np.diff(rp).max() > 30
    plan = _plan(cuda, rp, ci, v, algo="level", arith=arith)
    b = api.uniform(81, 3000).astype(dtype)
    ref = oracle.csr_forward(rp, ci, v, b, fused=arith == "fused")
    for _ in range(2):
        assert np.array_equal(_solve(plan, cuda, b).view(bits), ref.view(bits))
    plan.close()


@pytest.mark.parametrize("k", [6, 16])  # two and four right-hand sides per thread
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("arith", ["fused", "reference"])
@pytest.mark.parametrize("off", [4, 8, 16, 30])
def test_several_right_hand_sides_per_thread(cuda, off, arith, dtype, k):
    """200 equal matrices: more workgroups of one right-hand side than the
    compute units take at once, so a thread solves as many as divide k."""
    import torch
    from capellinisptrsv_amd import Batch
    mats, n = 200, 1200
    rp1, ci1, v1 = api.generate("level", n=n, levels=60, width=20, depth=2, offdiag=off, seed=83 + off)
    assert off - 4 < np.diff(rp1).max() - 1 <= off
    nnz = len(ci1)
    rp = np.concatenate([rp1[:-1] + m * nnz for m in range(mats)] + [[mats * nnz]]).astype(np.int32)
    ci = np.tile(ci1, mats)
    v = (np.tile(v1, mats) * np.repeat(1.0 + 0.001 * np.arange(mats), nnz)).astype(dtype)
    row_off = (np.arange(mats + 1) * n).astype(np.int32)
    bt = Batch(*(torch.from_numpy(a).to(cuda) for a in (row_off, rp, ci, v)), k=k, arith=arith)
    assert bt.step_matrices == mats
    b = api.uniform(84 + k, mats * n * k).astype(dtype)
    x = bt.solve(torch.from_numpy(b.reshape(mats * n, k)).to(cuda)).cpu().numpy().reshape(mats, -1)
    for m in range(0, mats, 13):
        ref = oracle.csr_forward(rp1, ci1, v[m * nnz:(m + 1) * nnz], b[m * n * k:(m + 1) * n * k], rhs=k,
                                 fused=arith == "fused")
        assert np.array_equal(x[m], ref), m
    bt.close()
