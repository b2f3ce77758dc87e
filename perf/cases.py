"""Measured cases: what a user of the local SpGEMM path has it do.

Every case goes through the Python entry points of trident_amd.device (one
call each of the C-ABI behind them) on operands that are in device memory,
as a stage loop, an AMG setup or a request server keeps them.  The kinds:

  product     C = A*A (LocalMatrix::spgemm), Erdos-Renyi or R-MAT operand
  galerkin    C = P^T (A P), the AMG coarse operator, P^T made once
  accumulate  C += A*B of one tile pair of a 4x4 grid (LocalMatrix::sp_mma)
  add         C += X, sorted partial-C tiles (LocalMatrix::spadd)
  exchange    SpaComm's step before a multiply: masks of A's columns and B's
              rows, their intersection, both tiles compressed by it
  convert     CSC tile to CSR (the form A's tiles arrive in)
  stage       one stage of 16 tile products as one graph launch (Batch)
  serve       a burst of mixed requests through the request server

Sizes are those of the repository's own configurations, tests and benchmark
(ER n = 1024, R-MAT scales 12-20, edge factors 8-16, 4x4 grids, 27-point
Laplacians 16^3-96^3) or generic ones between them.
"""
from __future__ import annotations

import ctypes
import functools
import gc
import math

import torch

import trident_amd.device as td
from trident_amd import gen
from trident_amd._lib import TR_COLS, TR_ROWS, tr_csx_t

DEV = "cuda:0"


# --------------------------------------------------------------------- cases
def listed():
    return [
        # the smallest product in use (a unit test, a coarse level): latency
        dict(name="product_er_1024", kind="product", graph="er", n=1024, degree=8, panels=False),
        # a small graph request, odd dimension
        dict(name="product_rmat_15013", kind="product", graph="rmat", n=15013, degree=11, panels=False),
        # an ordinary graph product
        dict(name="product_rmat_17", kind="product", graph="rmat", n=1 << 17, degree=16, panels=False),
        # the largest: a product beyond one int32 tile, returned as panels
        dict(name="product_rmat_19", kind="product", graph="rmat", n=1 << 19, degree=16, panels=True),
        # AMG setup on a small and on a large grid
        dict(name="galerkin_19", kind="galerkin", n=19),
        dict(name="galerkin_96", kind="galerkin", n=96),
        # one rank's multiply-and-accumulate of a small tile pair
        dict(name="accumulate_rmat_16", kind="accumulate", scale=16, degree=16, i=1, j=2, k=1),
        # the partial-C add alone, at the size of a large stage's tile
        dict(name="add_262144", kind="add", n=1 << 18, x_degree=100, y_degree=400),
        # the exchange step of a stage and the conversion that follows it
        dict(name="exchange_rmat_18", kind="exchange", n=1 << 18, degree=16),
        dict(name="convert_rmat_19", kind="convert", n=500009, degree=16),
        # a whole stage as one launch
        dict(name="stage_rmat_18", kind="stage", scale=18, degree=16, k=1),
        # requests of mixed sizes that arrive together
        dict(name="serve_16", kind="serve", requests=16, scale_lo=12, scale_hi=16, grid_lo=16, grid_hi=48),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["product", "product", "galerkin", "accumulate", "add", "exchange", "convert", "stage", "serve"])
    if kind == "product":
        if rng.random() < 0.3:
            return dict(kind=kind, graph="er", n=_log_int(rng, 256, 200000), degree=rng.randint(3, 16), panels=False)
        return dict(kind=kind, graph="rmat", n=_log_int(rng, 1500, 260000), degree=rng.randint(6, 16),
                    panels=rng.random() < 0.3)
    if kind == "galerkin":
        return dict(kind=kind, n=_log_int(rng, 10, 96))
    if kind == "accumulate":
        k = rng.randint(1, 3)
        return dict(kind=kind, scale=rng.randint(12, 19), degree=rng.randint(8, 16), i=rng.randint(0, 3),
                    j=rng.randint(0, 3), k=k)
    if kind == "add":
        return dict(kind=kind, n=_log_int(rng, 1000, 1 << 18), x_degree=_log_int(rng, 4, 100),
                    y_degree=_log_int(rng, 16, 400))
    if kind in ("exchange", "convert"):
        return dict(kind=kind, n=_log_int(rng, 4000, 1 << 20), degree=rng.randint(4, 16))
    if kind == "stage":
        return dict(kind=kind, scale=rng.randint(13, 18), degree=rng.randint(8, 16), k=rng.randint(1, 3))
    lo = rng.randint(12, 14)
    glo = rng.randint(10, 24)
    return dict(kind=kind, requests=rng.randint(4, 20), scale_lo=lo, scale_hi=lo + rng.randint(0, 2), grid_lo=glo,
                grid_hi=glo + rng.randint(1, 24))


# -------------------------------------------------------------------- inputs
class Host:
    """A CSR matrix as torch tensors on the GPU (int64 ptr, int64 idx, fp64)."""

    def __init__(self, nrows, ncols, ptr, idx, val):
        self.nrows, self.ncols, self.ptr, self.idx, self.val = nrows, ncols, ptr, idx, val

    @property
    def nnz(self):
        return int(self.idx.numel())

    def rows(self):
        return torch.repeat_interleave(torch.arange(self.nrows, device=DEV), self.ptr[1:] - self.ptr[:-1])

    def transposed(self):
        key = self.idx * self.nrows + self.rows()
        key, order = torch.sort(key)
        return _from_keys(key, self.val[order], self.ncols, self.nrows)


def _from_keys(key, val, nrows, ncols):
    """CSR of sorted unique keys row * ncols + column."""
    rows = torch.div(key, ncols, rounding_mode="floor")
    ptr = torch.zeros(nrows + 1, dtype=torch.int64, device=DEV)
    ptr[1:] = torch.cumsum(torch.bincount(rows, minlength=nrows), 0)
    return Host(nrows, ncols, ptr, key - rows * ncols, val)


def _pattern(seed):
    """Generator of a workload's sparsity pattern: fixed, as the sizes of its
    results are; what changes with the inputs' seed is the numbering
    (_renumbered) and the values."""
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _renumbered(v, n, flip):
    """Vertices renumbered inside aligned groups of 16 (all but a last,
    incomplete group): another pattern with the same degrees and locality."""
    return torch.where((v | 15) < n, v ^ flip, v)


def _uniform(g, n):
    return torch.rand(n, generator=g, device=DEV, dtype=torch.float64) * 2 - 1


def _er(g, n, degree, flip, pattern=1):
    """Erdos-Renyi: `degree` uniform columns per row, duplicates merged."""
    c = torch.randint(0, n, (n * degree,), generator=_pattern(pattern), device=DEV)
    r = torch.arange(n, device=DEV).repeat_interleave(degree)
    key = torch.unique(_renumbered(r, n, flip) * n + _renumbered(c, n, flip))
    return _from_keys(key, _uniform(g, key.numel()), n, n)


def _rmat(g, n, degree, flip, pattern=1):
    """R-MAT of the smallest scale that holds n vertices, cut to n x n (a =
    0.57, b = c = 0.19), duplicates merged, values U[-1, 1]."""
    scale = max(1, (n - 1).bit_length())
    m = degree << scale
    r = torch.zeros(m, dtype=torch.int64, device=DEV)
    c = torch.zeros(m, dtype=torch.int64, device=DEV)
    edges = _pattern(pattern)
    for _ in range(scale):
        u = torch.rand(m, generator=edges, device=DEV)
        down = u >= 0.76
        r = r * 2 + down
        c = c * 2 + torch.where(down, u >= 0.95, u >= 0.57)
    key = _renumbered(r, n, flip) * n + _renumbered(c, n, flip)
    if n < 1 << scale:
        key = key[(r < n) & (c < n)]
    del r, c
    key = torch.unique(key)
    return _from_keys(key, _uniform(g, key.numel()), n, n)


def _tile(m, i, j, grid):
    """Tile (i, j) of the square matrix m cut grid x grid."""
    t = m.nrows // grid
    rows = m.rows()
    keep = (rows >= i * t) & (rows < (i + 1) * t) & (m.idx >= j * t) & (m.idx < (j + 1) * t)
    key = (rows[keep] - i * t) * t + (m.idx[keep] - j * t)
    return _from_keys(key, m.val[keep], t, t)


@functools.lru_cache(maxsize=4)
def _grid_operators(n):
    return gen.laplace27(n), gen.sa_prolongator(n)


def _galerkin_inputs(g, n):
    """27-point operator and its smoothed prolongator, coefficients varied by
    up to 10% from point to point (a problem's own coefficients)."""
    out = []
    for m in _grid_operators(n):
        scale = 1.0 + 0.1 * _uniform(g, m.nnz)
        out.append(Host(m.nrows, m.ncols, torch.from_numpy(m.ptr).to(DEV).long(), torch.from_numpy(m.idx).to(DEV).long(),
                        torch.from_numpy(m.val).to(DEV) * scale))
    return out


def _multiply(a, b, budget=100_000_000):
    """a * b by expansion, sort and segment sums in fp64 (torch only)."""
    blen = b.ptr[1:] - b.ptr[:-1]
    ends = torch.cat([torch.zeros(1, dtype=torch.int64, device=DEV), torch.cumsum(blen[a.idx], 0)])
    row_end = ends[a.ptr].cpu()
    keys, vals = [], []
    r0 = 0
    while r0 < a.nrows:
        r1 = int(torch.searchsorted(row_end, int(row_end[r0]) + budget, right=True)) - 1
        r1 = min(max(r1, r0 + 1), a.nrows)
        p0, p1 = int(a.ptr[r0]), int(a.ptr[r1])
        if int(row_end[r1]) > int(row_end[r0]):
            k = a.idx[p0:p1]
            ln = blen[k]
            src = torch.repeat_interleave(torch.arange(p1 - p0, device=DEV), ln)
            q = torch.arange(src.numel(), device=DEV) - (ends[p0:p1] - ends[p0])[src] + b.ptr[k][src]
            arow = torch.repeat_interleave(torch.arange(r0, r1, device=DEV), a.ptr[r0 + 1:r1 + 1] - a.ptr[r0:r1])
            key, order = torch.sort(arow[src] * b.ncols + b.idx[q])
            prod = (a.val[p0:p1][src] * b.val[q])[order]
            del src, q, order
            _sum_equal(key, prod, keys, vals)
        r0 = r1
    key = torch.cat(keys) if keys else torch.zeros(0, dtype=torch.int64, device=DEV)
    val = torch.cat(vals) if vals else torch.zeros(0, dtype=torch.float64, device=DEV)
    return _from_keys(key, val, a.nrows, b.ncols)


def _sum_equal(key, val, keys, vals):
    """Appends the unique keys of the sorted `key` and the sums of their values."""
    uk, inv = torch.unique_consecutive(key, return_inverse=True)
    keys.append(uk)
    vals.append(torch.zeros(uk.numel(), dtype=torch.float64, device=DEV).index_add_(0, inv, val))


def _partial(g, a, b):
    """A partial C with the pattern of a * b (a stage's before) and values of
    its own."""
    c = _multiply(a, b)
    c.val = _uniform(g, c.nnz)
    return c


def _add(x, y):
    key, order = torch.sort(torch.cat([x.rows() * x.ncols + x.idx, y.rows() * y.ncols + y.idx]))
    keys, vals = [], []
    _sum_equal(key, torch.cat([x.val, y.val])[order], keys, vals)
    return _from_keys(keys[0], vals[0], x.nrows, x.ncols)


def _serve_plan(case):
    """(requests, scales, grids): 60% products of R-MATs, 40% Galerkin."""
    scales = sorted({case["scale_lo"], (case["scale_lo"] + case["scale_hi"]) // 2, case["scale_hi"]})
    grids = sorted({case["grid_lo"], (case["grid_lo"] + case["grid_hi"]) // 2, case["grid_hi"]})
    reqs = []
    for i in range(case["requests"]):
        if i % 5 in (0, 2, 4):
            reqs.append(("product", scales[(i // 2) % len(scales)]))
        else:
            reqs.append(("galerkin", grids[(i // 2) % len(grids)]))
    return reqs, scales, grids


def _inputs(case, seed):
    """The case's operands as Host matrices, made from the seed alone."""
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    flip = int(torch.randint(0, 16, (1,), generator=g, device=DEV))
    kind = case["kind"]
    if kind == "product":
        if case["panels"]:
            flip = 0  # where panels are cut depends on the order of the rows
        make = _er if case["graph"] == "er" else _rmat
        return {"A": make(g, case["n"], case["degree"], flip)}
    if kind == "galerkin":
        A, P = _galerkin_inputs(g, case["n"])
        return {"A": A, "P": P}
    if kind == "accumulate":
        m = _rmat(g, 1 << case["scale"], case["degree"], flip)
        i, j, k = case["i"], case["j"], case["k"]
        # the partial C of the stage before: the tile pair of inner index k - 1 or k + 1
        kc = k + 1 if k < 3 else 2
        return {"A": _tile(m, i, k, 4), "B": _tile(m, k, j, 4),
                "C": _partial(g, _tile(m, i, kc, 4), _tile(m, kc, j, 4))}
    if kind == "add":
        return {"X": _rmat(g, case["n"], case["x_degree"], flip), "Y": _rmat(g, case["n"], case["y_degree"], flip, 2)}
    if kind == "exchange":
        return {"A": _rmat(g, case["n"], case["degree"], flip), "B": _rmat(g, case["n"], case["degree"], flip, 2)}
    if kind == "convert":
        return {"A": _rmat(g, case["n"], case["degree"], flip)}
    if kind == "stage":
        m = _rmat(g, 1 << case["scale"], case["degree"], flip)
        k = case["k"]
        kc = k + 1 if k < 3 else 2
        t = {}
        for x in range(4):
            t["A%d" % x], t["B%d" % x] = _tile(m, x, k, 4), _tile(m, k, x, 4)
        la, lb = [_tile(m, x, kc, 4) for x in range(4)], [_tile(m, kc, x, 4) for x in range(4)]
        for i in range(4):
            for j in range(4):
                t["C%d%d" % (i, j)] = _partial(g, la[i], lb[j])
        return t
    if kind == "serve":
        _, scales, grids = _serve_plan(case)
        t = {}
        for s in scales:
            t["R%d" % s] = _rmat(g, 1 << s, 8 if s % 2 else 16, flip)
        for n in grids:
            t["A%d" % n], t["P%d" % n] = _galerkin_inputs(g, n)
        return t
    raise ValueError(kind)


# ------------------------------------------------------------------ prepare
class _Memory:
    """__cuda_array_interface__ of device memory that `owner` keeps alive."""

    def __init__(self, owner, ptr, n, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": typestr, "data": (ptr, False), "version": 2}


class _Owner:
    """Device matrices freed together (operands, or the last results), the
    tensors that operands borrow and the handles that use them."""

    def __init__(self):
        self.held, self.closers, self.kept = [], [], []

    def free(self):
        for m in self.held:
            m.free()
        self.held = []

    def __del__(self):
        try:
            for f in self.closers:
                f()
            self.free()
            _ctx.synchronize()  # before the borrowed tensors go
        except Exception:
            pass


class State:
    def __init__(self, case):
        self.case, self.own, self.out, self.views = case, _Owner(), _Owner(), {}

    def tensors(self, m):
        """ptr, idx, val of a device matrix as tensors on its memory."""
        d = m.d if isinstance(m, td.DeviceCsx) else m
        p = (d.nrows if d.majordim == TR_ROWS else d.ncols) + 1
        key = (d.ptr_vec, d.idx_vec, d.val, p, d.nnz)
        v = self.views.get(key)
        if v is None:
            if len(self.views) > 64:
                self.views.clear()
            v = [self._view(d.ptr_vec, p, "<i4"), self._view(d.idx_vec, d.nnz, "<i4"), self._view(d.val, d.nnz, "<f8")]
            self.views[key] = v
        return v

    def _view(self, ptr, n, typestr):
        if n == 0:
            return torch.empty(0, dtype=torch.int32 if typestr == "<i4" else torch.float64, device=DEV)
        address = ctypes.cast(ptr, ctypes.c_void_p).value
        return torch.as_tensor(_Memory((self.own, self.out), address, int(n), typestr), device=DEV)


_ctx = None  # the program's context: one stream, one pool
_last = None


def _context(case):
    global _ctx, _last
    if _ctx is None:
        _ctx = td.Context(0)
    if case != _last:  # another workload: a program's pools start empty
        gc.collect()
        _ctx.pool_trim()
        torch.cuda.empty_cache()
        _last = dict(case)
    return _ctx


def _device(ctx, x, major=TR_ROWS):
    """x as a device matrix over tensors of the program's own (the library
    borrows operands); returns it with the tensors to keep."""
    m = x if major == TR_ROWS else x.transposed()
    keep = (m.ptr.to(torch.int32), m.idx.to(torch.int32), m.val.contiguous())
    d = tr_csx_t(majordim=major, nrows=x.nrows, ncols=x.ncols, nnz=x.nnz)
    d.ptr_vec, d.idx_vec, d.val = (t.data_ptr() for t in keep)
    return td.DeviceCsx(ctx, d), keep


def prepare(case, seed):
    ctx = _context(case)
    s = State(case)
    m = _inputs(case, seed)
    kind = case["kind"]

    def up(x, major=TR_ROWS):
        d, keep = _device(ctx, x, major)
        s.own.kept.append(keep)
        return d

    if kind == "product":
        s.A = up(m["A"])
    elif kind == "galerkin":
        s.A, s.P = up(m["A"]), up(m["P"])
        torch.cuda.synchronize()  # the context's stream reads what torch's wrote
        s.Pt = s.P.transpose()
        s.own.held.append(s.Pt)
    elif kind == "accumulate":
        s.A, s.B, s.C = up(m["A"]), up(m["B"]), up(m["C"])
    elif kind == "add":
        s.X, s.Y = up(m["X"]), up(m["Y"])
    elif kind == "exchange":
        s.A, s.B = up(m["A"], TR_COLS), up(m["B"])
    elif kind == "convert":
        s.A = up(m["A"], TR_COLS)
    elif kind == "stage":
        A = [up(m["A%d" % i]) for i in range(4)]
        B = [up(m["B%d" % j]) for j in range(4)]
        C = [up(m["C%d%d" % (i, j)]) for i in range(4) for j in range(4)]
        torch.cuda.synchronize()
        s.batch = td.Batch(ctx, [A[t // 4] for t in range(16)], [B[t % 4] for t in range(16)], C, compress=True)
        s.own.closers.append(s.batch.close)
    elif kind == "serve":
        s.requests, scales, grids = _serve_plan(case)
        mats = {name: up(x) for name, x in m.items()}
        torch.cuda.synchronize()
        s.server = td.Server(mem_budget=8 << 30, workers=1, max_batch=32)
        s.own.closers.append(s.server.close)
        s.ops = {}
        for r in scales:
            op = s.server.register(mats["R%d" % r])
            s.ops["product", r] = (td.TR_REQ_SPGEMM, op, op)
        for n in grids:
            s.ops["galerkin", n] = (td.TR_REQ_GALERKIN, s.server.register(mats["A%d" % n]),
                                    s.server.register(mats["P%d" % n]))
        s.done = []
    torch.cuda.synchronize()
    return s


# ---------------------------------------------------------------------- run
def _borrowed(m):
    """The descriptor of m as an accumulator that the call leaves intact."""
    d = tr_csx_t()
    ctypes.memmove(ctypes.byref(d), ctypes.byref(m.d), ctypes.sizeof(tr_csx_t))
    return d


def run(s):
    kind = s.case["kind"]
    s.out.free()  # the results of the pass before
    if kind == "product":
        if s.case["panels"]:
            panels, _ = td.spgemm_panels(s.A, s.A)
            s.out.held = panels
            return [s.tensors(p) for p in panels]
        c = td.spgemm(s.A, s.A)
        s.out.held = [c]
        return s.tensors(c)
    if kind == "galerkin":
        ap = td.spgemm(s.A, s.P)
        c = td.spgemm(s.Pt, ap)
        ap.free()
        s.out.held = [c]
        return s.tensors(c)
    if kind == "accumulate":
        c = td.DeviceCsx(s.A.ctx, _borrowed(s.C))
        td.sp_mma(s.A, s.B, c)
        s.out.held = [c]
        return s.tensors(c)
    if kind == "add":
        c = td.DeviceCsx(s.X.ctx, _borrowed(s.Y))
        td.spadd(s.X, c)
        s.out.held = [c]
        return s.tensors(c)
    if kind == "exchange":
        ctx, n = s.A.ctx, s.case["n"]
        ma = td.SpaComm.gen_bitmask(ctx, ctypes.cast(s.A.d.ptr_vec, ctypes.c_void_p).value, n)
        mb = td.SpaComm.gen_bitmask(ctx, ctypes.cast(s.B.d.ptr_vec, ctypes.c_void_p).value, n)
        both = td.SpaComm.intersect(ctx, ma, mb, (n + 63) // 64)
        a, b = td.SpaComm.compress(s.A, both), td.SpaComm.compress(s.B, both)
        for mask in (ma, mb, both):
            ctx.free(mask)
        s.out.held = [a, b]
        return [s.tensors(a), s.tensors(b)]
    if kind == "convert":
        c = s.A.csc_to_csr()
        s.out.held = [c]
        return s.tensors(c)
    if kind == "stage":
        s.batch.run()
        return [s.tensors(s.batch.result(t)) for t in range(16)]
    if kind == "serve":
        for rid in s.done:
            s.server.release(rid)
        s.done = [s.server.submit(*s.ops[r]) for r in s.requests]
        return [s.tensors(s.server.wait(rid)[0]) for rid in s.done]
    raise ValueError(kind)


# --------------------------------------------------------------------- work
def _csx_bytes(rows, nnz):
    return 12.0 * nnz + 4.0 * (rows + 1)


def work(case):
    """Operands read once, results written once; 2 flops a multiplication."""
    ctx = _context(case)
    m = _inputs(case, 1)
    kind = case["kind"]

    def size(x):
        return _csx_bytes(x.nrows, x.nnz)

    def product(a, b):
        (da, _a), (db, _b) = _device(ctx, a), _device(ctx, b)
        torch.cuda.synchronize()
        return td.symbolic(da, db)[0], td.spgemm_flops(da, db)

    def galerkin(A, P):
        (da, _a), (dp, _p) = _device(ctx, A), _device(ctx, P)
        torch.cuda.synchronize()
        pt, ap = dp.transpose(), td.spgemm(da, dp)
        nnz, _ = td.symbolic(pt, ap)
        flops = 2.0 * (td.spgemm_flops(da, dp) + td.spgemm_flops(pt, ap))
        # A and P^T read (P is P^T's entries), AP written and read, C written
        nbytes = size(A) + 2 * size(P) + 2 * _csx_bytes(A.nrows, ap.nnz) + _csx_bytes(P.ncols, nnz)
        pt.free(), ap.free()
        return nbytes, flops

    if kind == "product":
        A = m["A"]
        nnz, mults = product(A, A)
        return {"bytes": size(A) + _csx_bytes(A.nrows, nnz), "flops": 2.0 * mults}
    if kind == "galerkin":
        b, f = galerkin(m["A"], m["P"])
        return {"bytes": b, "flops": f}
    if kind in ("accumulate", "stage"):
        pairs = [("A", "B", "C")] if kind == "accumulate" else [("A%d" % i, "B%d" % j, "C%d%d" % (i, j))
                                                               for i in range(4) for j in range(4)]
        nbytes, flops = 0.0, 0.0
        seen = set()
        for a, b, c in pairs:
            nnz, mults = product(m[a], m[b])
            flops += 2.0 * mults
            for name in (a, b, c):
                if name not in seen:
                    seen.add(name)
                    nbytes += size(m[name])
            nbytes += _csx_bytes(m[c].nrows, max(nnz, m[c].nnz))  # the new partial C holds both patterns
        return {"bytes": nbytes, "flops": flops}
    if kind == "add":
        return {"bytes": 2 * (size(m["X"]) + size(m["Y"])), "flops": 0.0}
    if kind == "exchange":
        return {"bytes": 2 * (size(m["A"]) + size(m["B"])), "flops": 0.0}
    if kind == "convert":
        return {"bytes": 2 * size(m["A"]), "flops": 0.0}
    if kind == "serve":
        nbytes, flops = 0.0, 0.0
        cost = {}
        for r in _serve_plan(case)[0]:
            if r not in cost:
                if r[0] == "product":
                    A = m["R%d" % r[1]]
                    nnz, mults = product(A, A)
                    cost[r] = (size(A) + _csx_bytes(A.nrows, nnz), 2.0 * mults)
                else:
                    cost[r] = galerkin(m["A%d" % r[1]], m["P%d" % r[1]])
            nbytes += cost[r][0]
            flops += cost[r][1]
        return {"bytes": nbytes, "flops": flops}
    raise ValueError(kind)


# -------------------------------------------------------------------- exact
def exact(case, seed):
    """What run() returns, from torch alone in 64 bits; None for the largest."""
    kind = case["kind"]

    def out(h):
        return [h.ptr.to(torch.int32), h.idx.to(torch.int32), h.val]

    if kind == "product" and (case["panels"] or case["n"] > 300000):
        return None
    m = _inputs(case, seed)
    if kind == "product":
        return out(_multiply(m["A"], m["A"]))
    if kind == "galerkin":
        return out(_multiply(m["P"].transposed(), _multiply(m["A"], m["P"])))
    if kind == "accumulate":
        return out(_add(m["C"], _multiply(m["A"], m["B"])))
    if kind == "add":
        return out(_add(m["Y"], m["X"]))
    if kind == "exchange":
        A, B = m["A"], m["B"]
        At = A.transposed()
        keep = (At.ptr[1:] > At.ptr[:-1]) & (B.ptr[1:] > B.ptr[:-1])
        got = []
        for x in (At, B):
            sel = keep[x.rows()]
            ptr = torch.zeros_like(x.ptr)
            ptr[1:] = torch.cumsum((x.ptr[1:] - x.ptr[:-1]) * keep, 0)
            got.append(out(Host(x.nrows, x.ncols, ptr, x.idx[sel], x.val[sel])))
        return got
    if kind == "convert":
        return out(m["A"])
    if kind == "stage":
        return [out(_add(m["C%d%d" % (i, j)], _multiply(m["A%d" % i], m["B%d" % j]))) for i in range(4)
                for j in range(4)]
    if kind == "serve":
        done = {}
        for r in _serve_plan(case)[0]:
            if r not in done:
                if r[0] == "product":
                    A = m["R%d" % r[1]]
                    done[r] = out(_multiply(A, A))
                else:
                    A, P = m["A%d" % r[1]], m["P%d" % r[1]]
                    done[r] = out(_multiply(P.transposed(), _multiply(A, P)))
        return [done[r] for r in _serve_plan(case)[0]]
    raise ValueError(kind)
