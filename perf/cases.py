"""The work whose speed this library is judged by: solves, refined solves,
gradients and batches over the matrices users bring, through the public
entry points (Plan, Batch, sptrsv, sptrsv_csr_solve).

Matrix kinds (all lower triangular, diagonal last in each row, off-diagonal
values U[-1,1], diagonal 1 + sum|off-diagonal|):
  level      rows in `levels` groups of about n / levels; a row draws 1 to
             `offdiag` columns from the previous 1 to 3 groups (graphs and
             circuits with wide, shallow dependencies)
  band       up to `offdiag` columns in the previous `band` rows
  dense_band every column of the previous `band` rows kept with probability p
             (factors of banded and one-dimensional problems: few rows per
             level, tens of entries per row)
  ragged     row i draws 0 to `offdiag` columns in the previous `band` rows
             (row lengths that vary, as in the batched workload)
  grid       the lower half of a 7-point stencil on an nx x ny x nz grid, in
             natural order (incomplete factorizations, Gauss-Seidel sweeps)

Operations:
  solve      plan.solve(b) of one matrix that a program holds a plan of
  precond    y = L^-1 b, then x = U^-1 y with U the upper factor and L unit
             lower: one application of an ILU preconditioner
  refined    plan.solve_refined(b): FP32 solves inside FP64 refinement
  train      x = sptrsv(values, b, plan) and its gradients
  batch      Batch.solve: many matrices, several right-hand sides each
  oneshot    api.sptrsv_csr_solve on host arrays: check, copies and solve
"""
import functools
import json
import math
import zlib

import numpy as np
import torch

from capellinisptrsv_amd import Batch, Plan, api
from capellinisptrsv_amd.torch_ops import sptrsv

# ---------------------------------------------------------------------- cases


def listed():
    return [
        # a small system inside an outer loop: latency and launches
        dict(name="small_band_2k", op="solve", kind="band", n=2000, offdiag=3, band=64, k=1, dtype="f64"),
        # narrow levels: hundreds of levels of a hundred rows
        dict(name="band_100k", op="solve", kind="band", n=100_000, offdiag=3, band=1000, k=1, dtype="f64"),
        # rows of varying length, a few tens of rows per level, an odd size
        dict(name="ragged_60k", op="solve", kind="ragged", n=60_001, offdiag=15, band=2500, k=1, dtype="f64"),
        # a preconditioner application on a structured grid, both directions
        dict(name="ilu_grid_720k", op="precond", kind="grid", nx=100, ny=90, nz=80, k=1, dtype="f64"),
        # the largest single solve: wide levels, 2 M rows
        dict(name="wide_2m", op="solve", kind="level", n=2_000_000, levels=200, offdiag=2, k=1, dtype="f64"),
        # the same kind in single precision, an odd size
        dict(name="wide_f32_777k", op="solve", kind="level", n=777_001, levels=120, offdiag=3, k=1, dtype="f32"),
        # a block of right-hand sides on wide levels (block Krylov, several loads)
        dict(name="wide_1m_rhs16", op="solve", kind="level", n=1_000_000, levels=100, offdiag=2, k=16, dtype="f64"),
        # a deep, narrow, dense band: one row after another
        dict(name="deep_band_500k", op="solve", kind="dense_band", n=500_000, band=128, p=0.3, k=1, dtype="f64"),
        # the same kind with several right-hand sides
        dict(name="deep_band_200k_rhs8", op="solve", kind="dense_band", n=200_000, band=96, p=0.3, k=8, dtype="f64"),
        # mixed precision: single-precision solves refined to double
        dict(name="refined_1m", op="refined", kind="level", n=1_000_000, levels=100, offdiag=2, k=1, dtype="f64"),
        # training through the solve: forward and gradients
        dict(name="train_1m", op="train", kind="level", n=1_000_000, levels=100, offdiag=2, k=1, dtype="f64"),
        # many matrices of mixed sizes with several right-hand sides each
        dict(name="batch_40x16", op="batch", kind="ragged", matrices=40, n_lo=2000, n_hi=40_000, offdiag=15,
             band_lo=64, band_hi=4096, k=16, dtype="f64"),
    ]


def _size(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["small", "band", "ragged", "precond", "wide", "wide", "wide_rhs", "deep", "deep_rhs", "refined",
                     "train", "batch", "oneshot"])
    if op == "small":
        return dict(op="solve", kind=rng.choice(["band", "ragged"]), n=_size(rng, 500, 20_000),
                    offdiag=rng.randint(2, 8), band=_size(rng, 32, 500), k=rng.choice([1, 1, 2, 4]),
                    dtype=rng.choice(["f64", "f64", "f32"]))
    if op == "band":
        return dict(op="solve", kind="band", n=_size(rng, 20_000, 200_000), offdiag=rng.randint(2, 4),
                    band=_size(rng, 500, 2000), k=1, dtype=rng.choice(["f64", "f64", "f32"]))
    if op == "ragged":
        return dict(op="solve", kind="ragged", n=_size(rng, 20_000, 100_000), offdiag=rng.randint(6, 15),
                    band=_size(rng, 1000, 4096), k=1, dtype="f64")
    if op == "precond":
        return dict(op="precond", kind="grid", nx=rng.randint(40, 110), ny=rng.randint(40, 100),
                    nz=rng.randint(20, 80), k=1, dtype=rng.choice(["f64", "f64", "f32"]))
    if op in ("deep", "deep_rhs"):
        return dict(op="solve", kind="dense_band", n=_size(rng, 50_000, 400_000 if op == "deep" else 150_000),
                    band=rng.randint(32, 128), p=round(rng.uniform(0.1, 0.3), 3),
                    k=1 if op == "deep" else rng.choice([2, 4, 8]), dtype="f64")
    if op == "batch":
        return dict(op="batch", kind="ragged", matrices=rng.randint(10, 40), n_lo=2000,
                    n_hi=_size(rng, 8000, 40_000), offdiag=rng.randint(5, 15), band_lo=64,
                    band_hi=_size(rng, 500, 4096), k=rng.choice([4, 8, 16]), dtype="f64")
    if op == "oneshot":
        return dict(op="oneshot", kind="level", n=_size(rng, 10_000, 300_000), levels=rng.randint(10, 40), offdiag=2,
                    k=1, dtype=rng.choice(["f64", "f32"]))
    n = _size(rng, 100_000, 1_900_000 if op == "wide" else 900_000)
    case = dict(op="solve", kind="level", n=n, levels=max(10, n // rng.randint(6000, 12_000)),
                offdiag=rng.randint(2, 3), k=1, dtype="f64")
    if op == "wide":
        case["dtype"] = rng.choice(["f64", "f32"])
    elif op == "wide_rhs":
        case["k"] = rng.choice([3, 4, 8, 16])
    else:
        case["op"] = op
    return case


# ------------------------------------------------------------------- matrices
def _csr(n, rows, cols, distinct=False):
    """row_ptr and col_idx: the off-diagonals (rows, cols), each once and
    sorted (distinct: they come that way), and the diagonal."""
    if not distinct:
        key = np.unique(rows * np.int64(n) + cols)
        rows, cols = key // n, key % n
    rp = np.zeros(n + 1, np.int64)
    np.cumsum(np.bincount(rows, minlength=n) + 1, out=rp[1:])
    ci = np.empty(rp[-1], np.int32)
    ci[np.arange(len(rows)) + rows] = cols  # one diagonal slot per earlier row
    ci[rp[1:] - 1] = np.arange(n)
    return rp.astype(np.int32), ci


def _band(n, count, band, rng):
    """count[i] draws per row from the previous `band` rows."""
    count = np.minimum(count, np.arange(n))
    rows = np.repeat(np.arange(n, dtype=np.int64), count)
    width = np.minimum(rows, band)
    return rows, rows - 1 - (rng.random(len(rows)) * width).astype(np.int64)


def _pattern(case, rng):
    kind = case["kind"]
    if kind == "grid":
        nx, ny, nz = case["nx"], case["ny"], case["nz"]
        n = nx * ny * nz
        i = np.arange(n, dtype=np.int64)
        x, y, z = i % nx, i // nx % ny, i // (nx * ny)
        pairs = [(i[m], i[m] - s) for m, s in ((z > 0, nx * ny), (y > 0, nx), (x > 0, 1))]
        rows, cols = (np.concatenate(a) for a in zip(*pairs))
        return _csr(n, rows, cols)
    n = case["n"]
    if kind == "level":
        width = -(-n // case["levels"])
        count = rng.integers(1, case["offdiag"] + 1, n)
        count[:width] = 0
        rows = np.repeat(np.arange(n, dtype=np.int64), count)
        first = rows // width * width
        lo = np.maximum(0, first - 3 * width)
        cols = lo + (rng.random(len(rows)) * (first - lo)).astype(np.int64)
    elif kind == "band":
        rows, cols = _band(n, np.full(n, case["offdiag"]), case["band"], rng)
    elif kind == "ragged":
        rows, cols = _band(n, rng.integers(0, case["offdiag"] + 1, n), case["band"], rng)
    else:  # dense_band
        w = case["band"]
        keep = rng.integers(0, 65536, (n, w), dtype=np.uint16) < int(case["p"] * 65536)
        keep[:w] &= np.arange(w) >= (w - np.arange(min(w, n)))[:, None]  # columns below 0
        at = np.flatnonzero(keep)
        rows = at // w
        return _csr(n, rows, at - rows * (w - 1) - w, distinct=True)
    return _csr(n, rows, cols)


@functools.lru_cache(maxsize=4)
def _patterns(key):
    """The case's sparsity patterns: a program solves with many matrices of
    one pattern (time steps, training steps), so the seed changes values."""
    case = json.loads(key)
    rng = np.random.default_rng(zlib.crc32(key.encode()))
    if case["op"] != "batch":
        return [_pattern(case, rng)]
    out = []
    for _ in range(case["matrices"]):
        n = int(np.exp(rng.uniform(np.log(case["n_lo"]), np.log(case["n_hi"]))))
        band = int(rng.integers(case["band_lo"], case["band_hi"] + 1))
        out.append(_pattern(dict(case, n=n, band=band), rng))
    return out


def _inputs(case, seed):
    """Host arrays of the case: matrices, right-hand sides, and the gradient
    of x (train) -- the same for a seed on every side."""
    rng = np.random.default_rng([seed, 20240])
    dt = np.float32 if case["dtype"] == "f32" else np.float64
    mats = []
    for rp, ci in _patterns(json.dumps({k: v for k, v in case.items() if k != "name"}, sort_keys=True)):
        v = rng.uniform(-1.0, 1.0, len(ci))
        last = rp[1:] - 1
        v[last] = 0.0
        v[last] = 1.0 + np.add.reduceat(np.abs(v), rp[:-1])
        mats.append((rp, ci, v.astype(dt)))
    total = sum(len(m[0]) - 1 for m in mats)
    b = rng.uniform(-1.0, 1.0, total if case["k"] == 1 else (total, case["k"])).astype(dt)
    if case["op"] == "batch":
        return dict(mats=mats, b=b)
    (rp, ci, v), n = mats[0], total
    out = dict(rp=rp, ci=ci, v=v, b=b)
    if case["op"] == "train":
        out["g"] = rng.uniform(-1.0, 1.0, b.shape)
    if case["op"] == "precond":
        # the unit lower factor's strict part, and the upper factor: the
        # transposed pattern with values of its own, diagonal first
        diag = np.zeros(len(ci), bool)
        diag[rp[1:] - 1] = True
        rows = np.repeat(np.arange(n), np.diff(rp))
        out["l"] = (rp - np.arange(n + 1, dtype=np.int32), ci[~diag], 0.3 * v[~diag].astype(dt))
        order = np.argsort(ci, kind="stable")  # column c: its diagonal, then the rows below in order
        urp = np.zeros(n + 1, np.int32)
        np.cumsum(np.bincount(ci, minlength=n), out=urp[1:])
        out["u"] = (urp, rows[order].astype(np.int32), v[order].astype(dt))
    return out


# ------------------------------------------------------------------ the calls
def prepare(case, seed):
    h = _inputs(case, seed)
    dev = torch.device("cuda:0")

    def put(a):
        return torch.from_numpy(np.ascontiguousarray(a)).to(dev)

    op = case["op"]
    if op == "oneshot":
        return dict(op=op, **h)
    b = put(h["b"])
    if op == "batch":
        off = np.cumsum([0] + [len(m[0]) - 1 for m in h["mats"]]).astype(np.int32)
        nz = np.cumsum([0] + [len(m[1]) for m in h["mats"]])
        rp = np.concatenate([m[0][:-1] + o for m, o in zip(h["mats"], nz)] + [[nz[-1]]]).astype(np.int32)
        ci = np.concatenate([m[1] for m in h["mats"]])
        v = np.concatenate([m[2] for m in h["mats"]])
        batch = Batch(*(put(a) for a in (off, rp, ci, v)), k=case["k"])
        return dict(op=op, plan=batch, b=b, x=torch.empty_like(b))
    if op == "precond":
        return dict(op=op, lower=Plan(*(put(a) for a in h["l"]), unit_diagonal=True),
                    upper=Plan(*(put(a) for a in h["u"]), upper=True), b=b, y=torch.empty_like(b),
                    x=torch.empty_like(b))
    values = put(h["v"])
    plan = Plan(put(h["rp"]), put(h["ci"]), values)
    if op == "train":
        return dict(op=op, plan=plan, values=values.requires_grad_(), b=b.requires_grad_(), g=put(h["g"]))
    return dict(op=op, plan=plan, b=b, x=torch.empty_like(b))


def run(state):
    op = state["op"]
    if op == "oneshot":
        return api.sptrsv_csr_solve(state["rp"], state["ci"], state["v"], state["b"])
    if op == "precond":
        state["lower"].solve(state["b"], out=state["y"])
        return state["upper"].solve(state["y"], out=state["x"])
    if op == "refined":
        return state["plan"].solve_refined(state["b"], tol=1e-12, out=state["x"])[0]
    if op == "train":
        x = sptrsv(state["values"], state["b"], state["plan"])
        gv, gb = torch.autograd.grad(x, (state["values"], state["b"]), state["g"])
        return x.detach(), gb, gv
    return state["plan"].solve(state["b"], out=state["x"])


def _rows_and_entries(case):
    """Rows and (expected) stored entries of a case's matrices."""
    kind = case["kind"]
    if case["op"] == "batch":
        lo, hi = case["n_lo"], case["n_hi"]
        n = case["matrices"] * (hi - lo) / math.log(hi / lo)  # n is log-uniform
        return n, n * (1 + case["offdiag"] / 2)
    if kind == "grid":
        nx, ny, nz = case["nx"], case["ny"], case["nz"]
        n = nx * ny * nz
        return n, 4 * n - nx * ny - ny * nz - nx * nz
    n = case["n"]
    per_row = {"level": (1 + case.get("offdiag", 0)) / 2, "band": case.get("offdiag", 0),
               "ragged": case.get("offdiag", 0) / 2, "dense_band": case.get("p", 0) * case.get("band", 0)}[kind]
    return n, n * (1 + per_row)


def work(case):
    n, nnz = _rows_and_entries(case)
    vb = 4 if case["dtype"] == "f32" else 8
    matrix, vec = 4 * (n + 1) + (4 + vb) * nnz, vb * n * case["k"]
    if case["op"] == "precond":  # both factors; the intermediate vector is written and read
        return dict(bytes=2 * matrix + 4 * vec, flops=4 * nnz)
    if case["op"] == "train":  # forward (b, x) and backward (matrix, g, x; both gradients)
        return dict(bytes=2 * matrix + 5 * vec + vb * nnz, flops=5 * nnz)
    return dict(bytes=matrix + 2 * vec, flops=2 * nnz * case["k"])


# ------------------------------------------------------------- 64-bit results
def _by_rows(rp, ci, v, b):
    """Forward substitution row by row (diagonal last)."""
    x = np.zeros_like(b)
    ptr = rp.tolist()
    for i in range(len(ptr) - 1):
        s, e = ptr[i], ptr[i + 1] - 1
        x[i] = (b[i] - v[s:e] @ x[ci[s:e]]) / v[e]
    return x


def _spans(start, count):
    """The positions start[i] .. start[i] + count[i] - 1 of all i, in a row."""
    ends = np.cumsum(count)
    return np.arange(ends[-1] if len(ends) else 0) + np.repeat(start - (ends - count), count)


def _by_levels(rp, ci, v, b):
    """Forward substitution a level at a time, for matrices of few levels."""
    n = len(rp) - 1
    rows = np.repeat(np.arange(n), np.diff(rp))
    off = np.flatnonzero(ci != rows)
    order = off[np.argsort(ci[off], kind="stable")]
    out_ptr = np.zeros(n + 1, np.int64)
    np.cumsum(np.bincount(ci[off], minlength=n), out=out_ptr[1:])
    out_row = rows[order]
    waiting = np.diff(rp).astype(np.int64) - 1
    s = np.zeros_like(b)
    x = np.zeros_like(b)
    front = np.flatnonzero(waiting == 0)
    while len(front):
        x[front] = ((b[front] - s[front]).T / v[rp[front + 1] - 1]).T
        at = _spans(out_ptr[front], out_ptr[front + 1] - out_ptr[front])
        to, e = out_row[at], order[at]
        np.add.at(s, to, (x[ci[e]].T * v[e]).T)
        np.subtract.at(waiting, to, 1)
        to = np.unique(to)
        front = to[waiting[to] == 0]
    return x


def _solve(case, rp, ci, v, b):
    few = case["kind"] in ("level", "grid")
    return (_by_levels if few else _by_rows)(rp.astype(np.int64), ci, v.astype(np.float64), b.astype(np.float64))


def exact(case, seed):
    h = _inputs(case, seed)
    op = case["op"]
    if op == "batch":
        parts, lo = [], 0
        for rp, ci, v in h["mats"]:
            hi = lo + len(rp) - 1
            parts.append(_solve(case, rp, ci, v, h["b"][lo:hi]))
            lo = hi
        return torch.from_numpy(np.concatenate(parts))
    if op == "precond":
        rp, ci, v = h["l"]
        n = len(rp) - 1
        # append the unit diagonal
        at = np.arange(len(ci)) + np.repeat(np.arange(n), np.diff(rp))
        frp = (rp + np.arange(n + 1)).astype(np.int64)
        fci, fv = np.empty(frp[-1], np.int64), np.ones(frp[-1])
        fci[at], fv[at] = ci, v
        fci[frp[1:] - 1] = np.arange(n)
        y = _solve(case, frp, fci, fv, h["b"])
        # backward substitution is forward substitution on reversed rows and columns
        rp, ci, v = h["u"]
        x = _solve(case, rp[-1] - rp[::-1], n - 1 - ci[::-1], v[::-1], y[::-1])
        return torch.from_numpy(x[::-1].copy())
    rp, ci, v, b = h["rp"], h["ci"], h["v"], h["b"]
    x = _solve(case, rp, ci, v, b)
    if op == "train":
        n = len(rp) - 1
        rows = np.repeat(np.arange(n), np.diff(rp))
        # L^T with rows and columns reversed is lower triangular, diagonal last
        order = np.lexsort((-rows, n - 1 - ci))
        rows_t, cols_t = (n - 1 - ci)[order], (n - 1 - rows)[order]
        ptr = np.zeros(n + 1, np.int64)
        np.cumsum(np.bincount(rows_t, minlength=n), out=ptr[1:])
        gb = _solve(case, ptr, cols_t, v[order], h["g"][::-1])[::-1].copy()
        return torch.from_numpy(x), torch.from_numpy(gb), torch.from_numpy(-gb[rows] * x[ci])
    if op == "oneshot":
        return x
    return torch.from_numpy(x)
