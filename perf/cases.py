"""Performance cases of the HSMU SpGEMM library: C = A * B, CSR in and CSR out, through the
Python binding of the C ABI (hsmu.Context), as a program that keeps its matrices in device
memory calls it.

A case names a matrix family with its sizes, the entry point (mode), the precision and the
width of C's row pointers.  Options are those of the autotuner table for the case's shape
class where the table holds it, else the defaults, with stage timing off (a program in
production asks for none).  C stays with the state until its next pass, which releases it
first, as a loop over products does.

Families (made on the GPU; structures belong to the case, values to the seed):
  laplace2d, laplace3d  5- and 7-point stencils with variable coefficients, A * A
  banded                FEM-like: 40..88 distinct columns per row within +-400, A * A
  random                rectangular, ragged rows, A * B
  rmat                  skewed graph (a, b, c = .57, .19, .19), edge factor 5..16, A * A
  zipf                  a panel of rows of A times A^T, A with 8 Zipf(1.2) columns per row
  batch                 many uneven Laplacians, C_i = A_i * A_i
"""
import functools
import math
import os
import random
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PKG = os.path.join(_ROOT, "hsmu-spgemm_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)
_TABLE = os.path.join(_PKG, "tuning", "gfx950.tsv")
_DEV = "cuda" if torch.cuda.is_available() else "cpu"

_ZIPF_ROWS, _ZIPF_COLS, _ZIPF_PER_ROW, _ZIPF_S = 500000, 100000, 8, 1.2
_BAND_LO, _BAND_HI, _BAND_HALF = 40, 88, 400


def listed():
    return [
        # the smallest call: a coarse multigrid level; all latency
        dict(name="lap2d-16", family="laplace2d", n=16, mode="call", precision="fp64", rowptr64=False),
        # the 128 x 128 grid Laplacian, squared
        dict(name="lap2d-128", family="laplace2d", n=128, mode="call", precision="fp64", rowptr64=False),
        # a 3D stencil of odd side: rows whose span is mostly empty
        dict(name="lap3d-47", family="laplace3d", n=47, mode="call", precision="fp64", rowptr64=False),
        # rectangular, ragged: a Galerkin-like product of unstructured operators
        dict(name="random-30k", family="random", m=30011, k=20029, n=25013, per_row=24, mode="call", precision="fp64",
             rowptr64=False),
        # the banded FEM-like matrix of the benchmark
        dict(name="banded-62k", family="banded", m=62451, mode="call", precision="fp64", rowptr64=False),
        # a smaller one of odd size in compensated FP32
        dict(name="banded-20k-fp32c", family="banded", m=20011, mode="call", precision="fp32c", rowptr64=False),
        # graph squaring, skewed rows: compensated FP32 at a middle size, FP64 at a large one
        # whose nnz(C) asks for 64-bit row pointers
        dict(name="rmat-16-fp32c", family="rmat", scale=16, edges=16, mode="call", precision="fp32c", rowptr64=False),
        dict(name="rmat-18", family="rmat", scale=18, edges=16, mode="call", precision="fp64", rowptr64=True),
        # a co-occurrence product streamed in row panels, both precisions
        dict(name="zipf-2000", family="zipf", rows=2000, mode="rows", precision="fp64", rowptr64=True),
        dict(name="zipf-777-fp32c", family="zipf", rows=777, mode="rows", precision="fp32c", rowptr64=True),
        # many uneven products in one call, and a replayed plan of a smaller set (a time
        # loop with fixed structure)
        dict(name="batch-512", family="batch", count=512, mode="batch", precision="fp64", rowptr64=False),
        dict(name="batch-96-plan", family="batch", count=96, mode="plan", precision="fp64", rowptr64=False),
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    family = rng.choice(("laplace2d", "laplace3d", "random", "banded", "rmat", "zipf", "batch"))
    case = dict(family=family, mode="call", precision=rng.choice(("fp64", "fp64", "fp32c")),
                rowptr64=rng.random() < 0.25)
    if family == "laplace2d":
        case.update(n=log(16, 400), mode=rng.choice(("call", "call", "plan")))
    elif family == "laplace3d":
        case.update(n=log(8, 64), mode=rng.choice(("call", "call", "plan")))
    elif family == "random":
        case.update(m=log(300, 60000), k=log(300, 40000), n=log(300, 50000), per_row=rng.randint(4, 32))
    elif family == "banded":
        case.update(m=log(3000, 62451), mode=rng.choice(("call", "call", "plan")))
    elif family == "rmat":
        case.update(scale=rng.randint(10, 17), edges=rng.randint(5, 16))
        case["rowptr64"] = rng.random() < 0.5
    elif family == "zipf":
        case.update(rows=log(100, 1500), mode="rows")
        case["rowptr64"] = True
    else:
        case.update(count=log(8, 400), mode=rng.choice(("batch", "plan")))
    return case


# ---- inputs ------------------------------------------------------------------------------

class _Csr:
    """A CSR matrix in torch tensors (int32 row pointers and columns) with the struct the
    library takes."""

    def __init__(self, M, N, rowptr, col, val):
        self.M, self.N, self.nnz = int(M), int(N), int(col.numel())
        self.rowptr, self.col = rowptr.to(torch.int32, copy=True), col.to(torch.int32, copy=True)
        self.val = val
        hsmu = _hsmu()
        self.csr = hsmu.Csr(self.M, self.N, self.nnz, self.rowptr.data_ptr(), self.col.data_ptr(),
                            self.val.data_ptr(), 0, 1 if val.dtype == torch.float32 else 0)


@functools.lru_cache(maxsize=None)
def _hsmu():
    import hsmu
    return hsmu


@functools.lru_cache(maxsize=None)
def _context():
    return _hsmu().Context(0)


def _gen(seed):
    g = torch.Generator(device=_DEV)
    g.manual_seed(int(seed))
    return g


def _rand(g, *shape, dtype=torch.float64):
    return torch.rand(*shape, generator=g, device=_DEV, dtype=dtype)


def _rowptr(rows, M):
    rp = torch.zeros(M + 1, dtype=torch.int64, device=_DEV)
    rp[1:] = torch.cumsum(torch.bincount(rows, minlength=M), 0)
    return rp


@functools.lru_cache(maxsize=1024)
def _stencil(dim, n):
    """Row pointers, columns and the diagonal's places of the (2 dim + 1)-point stencil on
    an n^dim grid."""
    M = n ** dim
    i = torch.arange(M, device=_DEV)
    steps = [n ** d for d in range(dim - 1, -1, -1)]
    offs, ok = [], []
    for s in steps:
        offs.append(-s)
        ok.append((i // s) % n > 0)
    offs.append(0)
    ok.append(torch.ones(M, dtype=torch.bool, device=_DEV))
    for s in reversed(steps):
        offs.append(s)
        ok.append((i // s) % n < n - 1)
    ok = torch.stack(ok, 1)
    col = (i[:, None] + torch.tensor(offs, device=_DEV)[None, :])[ok]
    rows = i[:, None].expand(-1, len(offs))[ok]
    return _rowptr(rows, M).to(torch.int32), col.to(torch.int32), rows == col


def _laplace_values(dim, diag, g):
    off = -(0.5 + _rand(g, diag.numel()))
    return torch.where(diag, 2.0 * dim + _rand(g, diag.numel()), off)


def _banded(m, g):
    width = 2 * _BAND_HALF + 1
    base = torch.arange(m, device=_DEV)[:, None] - _BAND_HALF + torch.arange(width, device=_DEV)[None, :]
    inside = (base >= 0) & (base < m)
    key = _rand(g, m, width, dtype=torch.float32).masked_fill_(~inside, 2.0)
    want = torch.randint(_BAND_LO, _BAND_HI + 1, (m, 1), generator=g, device=_DEV)
    want = torch.minimum(want, inside.sum(1, keepdim=True))
    order = torch.argsort(key, dim=1)
    rank_ok = torch.arange(width, device=_DEV)[None, :] < want
    take = torch.zeros(m, width, dtype=torch.bool, device=_DEV).scatter_(1, order, rank_ok)
    rows = torch.arange(m, device=_DEV)[:, None].expand(-1, width)[take]
    return m, m, _rowptr(rows, m), base[take]


def _merge(rows, col, M, N):
    """Sorted distinct (row, column) pairs as row pointers and columns."""
    key = torch.unique(rows * N + col)
    return M, N, _rowptr(key // N, M), key % N


def _random(m, n, per_row, g):
    want = torch.randint(0, per_row + 1, (m,), generator=g, device=_DEV)
    rows = torch.repeat_interleave(torch.arange(m, device=_DEV), want)
    return _merge(rows, torch.randint(0, n, (rows.numel(),), generator=g, device=_DEV), m, n)


def _rmat(scale, factor, g):
    M = 1 << scale
    edges = factor * M
    row = torch.zeros(edges, dtype=torch.int64, device=_DEV)
    col = torch.zeros(edges, dtype=torch.int64, device=_DEV)
    for _ in range(scale):
        u = _rand(g, edges)
        row = 2 * row + (u >= 0.76)
        col = 2 * col + (((u >= 0.57) & (u < 0.76)) | (u >= 0.95))
    return _merge(row, col, M, M)


def _zipf(g):
    w = torch.arange(1, _ZIPF_COLS + 1, device=_DEV, dtype=torch.float64) ** -_ZIPF_S
    cdf = torch.cumsum(w, 0) / w.sum()

    def pick(k):
        return torch.searchsorted(cdf, _rand(g, k)).clamp_(max=_ZIPF_COLS - 1)

    c = pick(_ZIPF_ROWS * _ZIPF_PER_ROW).view(_ZIPF_ROWS, _ZIPF_PER_ROW)
    while True:  # redraw the repeated columns of a row
        c = torch.sort(c, 1).values
        rep = torch.zeros_like(c, dtype=torch.bool)
        rep[:, 1:] = c[:, 1:] == c[:, :-1]
        k = int(rep.sum())
        if k == 0:
            break
        c[rep] = pick(k)
    rp = torch.arange(0, c.numel() + 1, _ZIPF_PER_ROW, device=_DEV)
    return _ZIPF_ROWS, _ZIPF_COLS, rp, c.reshape(-1)


def _transposed(M, N, rp, col):
    """The transposed structure, and the order of A's values in it."""
    rows = torch.repeat_interleave(torch.arange(M, device=_DEV), (rp[1:] - rp[:-1]).long())
    order = torch.argsort(col.long() * M + rows)
    return (N, M, _rowptr(col.long(), N), rows[order]), order


@functools.lru_cache(maxsize=16)
def _batch_sides(count):
    """Half 2D with sides log-uniform in [16, 256], half 3D in [8, 48]."""
    r = random.Random(3)
    two = [(2, int(math.exp(r.uniform(math.log(16), math.log(256))))) for _ in range(count // 2)]
    return two + [(3, int(math.exp(r.uniform(math.log(8), math.log(48))))) for _ in range(count - count // 2)]


def _zipf_start(case):
    return (_ZIPF_ROWS - case["rows"]) // 2


@functools.lru_cache(maxsize=2)
def _structure(key):
    """The structures of the case's matrices, drawn from the case alone: (M, N, rowptr, col)
    each, with what places their values."""
    case, g = dict(key), _gen(2)
    f = case["family"]
    if f == "rmat":
        return _rmat(case["scale"], case["edges"], g), None
    if f == "banded":
        return _banded(case["m"], g), None
    if f == "random":
        return _random(case["m"], case["k"], case["per_row"], g), _random(case["k"], case["n"], case["per_row"], g)
    if f == "zipf":
        a = _zipf(g)
        return a, _transposed(*a)
    raise ValueError(f)


def _key(case):
    return tuple(sorted((k, v) for k, v in case.items() if k != "name"))


def _inputs(case, seed):
    """The case's pairs (A, B) as (M, N, rowptr, col, val) with FP64 values (rounded to FP32
    where the case runs in FP32).  The structure belongs to the case, the values to the
    seed: N(0,1) for the banded matrix, U(0,1) for the graphs, U(-1,1) for the others."""
    g = _gen(seed)
    f = case["family"]
    if f in ("batch", "laplace2d", "laplace3d"):
        sides = _batch_sides(case["count"]) if f == "batch" else [(2 if f == "laplace2d" else 3, case["n"])]
        pairs = []
        for dim, n in sides:
            rp, col, diag = _stencil(dim, n)
            a = (n ** dim, n ** dim, rp, col, _laplace_values(dim, diag, g))
            pairs.append((a, a))
    else:
        a, b = _structure(_key(case))
        nnz = a[3].numel()
        if f == "banded":
            a += (torch.randn(nnz, generator=g, device=_DEV, dtype=torch.float64),)
        elif f == "rmat":
            a += (_rand(g, nnz),)
        else:
            a += (2.0 * _rand(g, nnz) - 1.0,)
        if f == "random":
            b += (2.0 * _rand(g, b[3].numel()) - 1.0,)
        elif f == "zipf":
            b = b[0] + (a[4][b[1]],)
        else:
            b = a
        pairs = [(a, b)]
    if case["precision"] == "fp32c":
        pairs = [tuple(x[:4] + (x[4].float().double(),) for x in p) for p in pairs]
    return pairs


# ---- the program ---------------------------------------------------------------------------

class _State:
    """The operands, the options and the last result (released before the next pass and
    when the state goes)."""

    def __init__(self, case, seed):
        hsmu, self.ctx, self.case = _hsmu(), _context(), case
        val = torch.float32 if case["precision"] == "fp32c" else torch.float64
        self.As, self.Bs = [], []
        for a, b in _inputs(case, seed):
            self.As.append(_Csr(*a[:4], a[4].to(val)))
            two = case["family"] in ("random", "zipf")
            self.Bs.append(_Csr(*b[:4], b[4].to(val)) if two else self.As[-1])
        torch.cuda.synchronize()
        base = hsmu.default_opts(timing=0, rowptr64=case["rowptr64"],
                                 precision=hsmu.HSMU_FP32_COMP if case["precision"] == "fp32c" else hsmu.HSMU_FP64)
        shapes = self.As
        if case["mode"] == "rows":  # the class of a panel
            self.r0 = _zipf_start(case)
            shapes = [_Panel(case["rows"], self.As[0].N, case["rows"] * _ZIPF_PER_ROW)]
        self.opts, _ = self.ctx.autotune(shapes, self.Bs, base=base, table=_TABLE if os.path.exists(_TABLE) else None,
                                         search=False)
        self.plan = self.ctx.plan(self.As, self.Bs, self.opts) if case["mode"] == "plan" else None
        self.result = None

    def release(self):
        if self.result is not None:
            if self.case["mode"] == "batch":
                self.ctx.free_batch(self.result)
            else:
                self.ctx.free_result(self.result)
            self.result = None

    def __del__(self):
        try:
            self.release()
            if self.plan is not None:
                self.plan.destroy()
        except Exception:
            pass


class _Panel:
    def __init__(self, M, N, nnz):
        self.csr = _hsmu().Csr(M, N, nnz, 0, 0, 0, 0, 0)


class _View:
    def __init__(self, ptr, n, kind):
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": kind, "data": (ptr, False), "version": 2}


def _view(ptr, n, kind):
    if n == 0:
        return torch.empty(0, dtype={"<i4": torch.int32, "<i8": torch.int64, "<f4": torch.float32,
                                     "<f8": torch.float64}[kind], device=_DEV)
    return torch.as_tensor(_View(ptr, n, kind), device=_DEV)


def prepare(case, seed):
    return _State(case, seed)


def run(state):
    ctx, mode = state.ctx, state.case["mode"]
    state.release()
    if mode == "plan":
        state.plan.execute()
        cs = state.plan.results
    elif mode == "batch":
        cs, _ = ctx.spgemm_batched_device(state.As, state.Bs, state.opts)
        state.result = cs
    elif mode == "rows":
        c, _ = ctx.spgemm_rows_device(state.As[0], state.r0, state.r0 + state.case["rows"], state.Bs[0], state.opts)
        state.result = c
        cs = [c]
    else:
        c, _ = ctx.spgemm_device(state.As[0], state.Bs[0], state.opts)
        state.result = c
        cs = [c]
    # the C_i of a batch lie one after another in three arrays
    c0, last = cs[0], cs[len(cs) - 1]
    wide, val = c0.rowptr64, "<f4" if c0.val32 else "<f8"
    esz, vsz = 8 if wide else 4, 4 if c0.val32 else 8
    nrp = (last.rowptr - c0.rowptr) // esz + last.M + 1
    nnz = (last.val - c0.val) // vsz + last.nnz
    return {"rowptr": _view(c0.rowptr, nrp, "<i8" if wide else "<i4"), "col": _view(c0.col, nnz, "<i4"),
            "val": _view(c0.val, nnz, val)}


# ---- what the product is -------------------------------------------------------------------

def _stacked(case, seed):
    """The case as one product: A's columns index B's rows, C's columns are local to their
    instance.  (rows of each instance, A rowptr/col/val, B rowptr/col/val, columns)"""
    pairs = _inputs(case, seed)
    if case["family"] == "zipf":
        (M, N, rp, col, val), b = pairs[0]
        r0 = _zipf_start(case)
        lo, hi = int(rp[r0]), int(rp[r0 + case["rows"]])
        pairs = [((case["rows"], N, rp[r0:r0 + case["rows"] + 1] - lo, col[lo:hi], val[lo:hi]), b)]

    def stack(mats, shift):
        rps, cols, vals, e, k = [], [], [], 0, 0
        for (M, N, rp, col, val), s in zip(mats, shift):
            rps.append(rp[:-1].long() + e)
            cols.append(col.long() + s)
            vals.append(val)
            e += col.numel()
        rps.append(torch.tensor([e], device=_DEV))
        return torch.cat(rps), torch.cat(cols), torch.cat(vals)

    As, Bs = [p[0] for p in pairs], [p[1] for p in pairs]
    starts = np.concatenate([[0], np.cumsum([b[0] for b in Bs])])[:-1].tolist()
    return [a[0] for a in As], stack(As, starts), stack(Bs, [0] * len(Bs)), max(b[1] for b in Bs)


_CHUNK = 1 << 28


def _chunks(A, B):
    """Row ranges of A of at most about _CHUNK products, with the products of each entry."""
    rpa, ca, _ = A
    rpb = B[0]
    per = rpb[ca + 1] - rpb[ca]
    cum = torch.zeros(per.numel() + 1, dtype=torch.int64, device=_DEV)
    cum[1:] = torch.cumsum(per, 0)
    ends = cum[rpa]
    M = rpa.numel() - 1
    r = 0
    while r < M:
        stop = int(torch.searchsorted(ends, ends[r] + _CHUNK, right=True)) - 1
        stop = min(max(stop, r + 1), M)
        yield r, stop, int(rpa[r]), int(rpa[stop]), per
        r = stop


def _keys(A, B, N, r, stop, lo, hi, per, values):
    """(row, column) keys of the products of rows [r, stop), and their values."""
    rpa, ca, va = A
    rpb, cb, vb = B
    n = per[lo:hi]
    if int(n.sum()) == 0:
        return None, None
    first = torch.cumsum(n, 0) - n
    at = torch.arange(int(n.sum()), device=_DEV)
    at += torch.repeat_interleave(rpb[ca[lo:hi]] - first, n)
    rows = torch.repeat_interleave(torch.arange(stop - r, device=_DEV), rpa[r + 1:stop + 1] - rpa[r:stop])
    key = torch.repeat_interleave(rows * N, n)
    key += cb[at]
    return key, torch.repeat_interleave(va[lo:hi], n) * vb[at] if values else None


@functools.lru_cache(maxsize=None)
def _size(items):
    case = dict(items)
    rows, A, B, N = _stacked(case, 1)
    products = nnz = 0
    for r, stop, lo, hi, per in _chunks(A, B):
        key, _ = _keys(A, B, N, r, stop, lo, hi, per, False)
        if key is not None:
            products += key.numel()
            key = torch.sort(key).values
            nnz += 1 + int((key[1:] != key[:-1]).sum())
    nnz_b = B[1].numel()
    rows_b = B[0].numel() - 1
    return products, nnz, sum(rows), A[1].numel(), rows_b, nnz_b


def work(case):
    """Each input array read once (a self-product's once in all) and C written once; two
    operations per product."""
    products, nnz, M, nnz_a, K, nnz_b = _size(_key(case))
    v = 4 if case["precision"] == "fp32c" else 8
    count = case.get("count", 1)
    nbytes = 4 * (M + count) + (4 + v) * nnz_a + (8 if case["rowptr64"] else 4) * (M + count) + (4 + v) * nnz
    if case["family"] in ("random", "zipf"):
        nbytes += 4 * (K + 1) + (4 + v) * nnz_b
    return {"bytes": nbytes, "flops": 2 * products}


def exact(case, seed):
    """C in 64 bits: every product formed, sorted by (row, column) and summed in FP64."""
    rows, A, B, N = _stacked(case, seed)
    counts, cols, vals = [], [], []
    for r, stop, lo, hi, per in _chunks(A, B):
        key, v = _keys(A, B, N, r, stop, lo, hi, per, True)
        if key is None:
            counts.append(torch.zeros(stop - r, dtype=torch.int64, device=_DEV))
            continue
        key, order = torch.sort(key)
        head = torch.ones_like(key, dtype=torch.bool)
        head[1:] = key[1:] != key[:-1]
        place = torch.cumsum(head, 0) - 1
        out = torch.zeros(int(place[-1]) + 1, dtype=torch.float64, device=_DEV)
        out.index_add_(0, place, v[order])
        del place, order, v
        key = key[head]
        counts.append(torch.bincount(key // N, minlength=stop - r))
        cols.append((key % N).to(torch.int32))
        vals.append(out)
    rp = torch.zeros(sum(rows) + 1, dtype=torch.int64, device=_DEV)
    rp[1:] = torch.cumsum(torch.cat(counts), 0)
    parts, at = [], 0
    for m in rows:
        parts.append(rp[at:at + m + 1] - rp[at])
        at += m
    empty = torch.empty(0, device=_DEV)
    return {"rowptr": torch.cat(parts).to(torch.int64 if case["rowptr64"] else torch.int32),
            "col": torch.cat(cols) if cols else empty.to(torch.int32),
            "val": torch.cat(vals) if vals else empty.double()}
