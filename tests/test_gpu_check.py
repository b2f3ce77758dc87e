"""Operand checks and flop sums at the edges of their work units (2048 segment
ends plus entries): a fault planted at each entry around a unit's edge is
found, a descent between rows is not one, and rows that span units or empty
runs have the oracle's flops."""
import numpy as np
import pytest

import oracle
from trident_amd import gen
from trident_amd._lib import TR_ERR_INVALID, TridentError
from trident_amd.device import spgemm, spgemm_flops
from trident_amd.gen import Csr

pytestmark = pytest.mark.gpu


def _rows(lens, ncols):
    lens = np.asarray(lens, np.int64)
    ptr = np.zeros(len(lens) + 1, np.int64)
    np.cumsum(lens, out=ptr[1:])
    idx = np.concatenate([np.arange(n) * (ncols // max(n, 1)) for n in lens] + [np.zeros(0, np.int64)])
    return Csr(len(lens), ncols, ptr.astype(np.int32), idx.astype(np.int32), np.ones(int(ptr[-1])))


def _status(ctx, m):
    d = ctx.upload(m)
    s = d.validate()
    d.free()
    return s


SHAPES = {"one_row": [9000], "rows": [3] * 2000, "gap": [5] + [0] * 3000 + [4000] + [0] * 70 + [1]}


@pytest.mark.parametrize("shape", sorted(SHAPES))
def test_faults_at_unit_edges(ctx, shape):
    m = _rows(SHAPES[shape], 1 << 20)
    assert _status(ctx, m) == 0
    first = np.zeros(m.nnz, bool)
    first[m.ptr[:-1][np.diff(m.ptr) > 0]] = True
    places = [p for p in (1, 63, 64, 511, 512, 513, 1534, 1536, 2046, 2047, 2048, 4094, m.nnz - 1) if p < m.nnz]
    for p in places:
        for bad, bit in ((m.idx[p - 1], 4), (-1, 2), (1 << 20, 2)):
            c = m.idx.copy()
            c[p] = bad
            s = _status(ctx, Csr(m.nrows, m.ncols, m.ptr, c, m.val))
            if bit == 2:
                assert s & 2, (p, bad)
            else:
                assert s == (0 if first[p] and (p + 1 == m.nnz or first[p + 1] or bad < m.idx[p + 1]) else 4), (p, bad)
    for r, v in ((0, 1), (len(m.ptr) // 2, m.nnz + 1), (len(m.ptr) - 1, m.nnz - 1), (len(m.ptr) // 2, -1)):
        q = m.ptr.copy()
        q[r] = v
        assert _status(ctx, Csr(m.nrows, m.ncols, q, m.idx, m.val)) & 1, (r, v)


def test_checks_start_clean_after_a_rejection(ctx):
    m = _rows([4] * 700, 5000)
    c = m.idx.copy()
    c[1000], c[1001] = c[1001], c[1000]
    bad, good = ctx.upload(Csr(m.nrows, m.ncols, m.ptr, c, m.val)), ctx.upload(_rows([3] * 5000, 40))
    for _ in range(2):
        with pytest.raises(TridentError) as e:
            spgemm(bad, good)
        assert e.value.code == TR_ERR_INVALID and "A has unsorted" in str(e.value)
        sq = ctx.upload(gen.erdos_renyi(300, 5, seed=3))
        spgemm(sq, sq).free()
        sq.free()
    bad.free()
    good.free()


@pytest.mark.parametrize("shape", sorted(SHAPES))
def test_flops_of_rows_over_units(ctx, shape):
    rng = np.random.default_rng(7)
    a = _rows(SHAPES[shape], 20000)
    lens = rng.integers(0, 4, 20000)
    lens[::5000] = 2500
    b = _rows(lens, 2500)
    da, db = ctx.upload(a), ctx.upload(b)
    assert spgemm_flops(da, db) == oracle.spgemm_flops(a, b)
    c = spgemm(da, db)
    h = c.download()
    p, i, v = oracle.spgemm(a, b)
    assert np.array_equal(h.ptr, p) and np.array_equal(h.idx, i) and np.array_equal(h.val, v)
    for x in (c, da, db):
        x.free()


def _status_by_definition(m):
    n, nnz, p = m.nrows, m.nnz, m.ptr.astype(np.int64)
    bad = (p < 0).any() or (p > nnz).any() or p[0] != 0 or p[-1] != nnz or (np.diff(p) < 0).any()
    start = {v for i, v in enumerate(p[:-1]) if 0 <= v < p[i + 1] and (i > 0 or v == 0)}
    order = any(m.idx[q] <= m.idx[q - 1] and q not in start for q in range(1, nnz))
    return int(bad) | 2 * bool((m.idx < 0).any() or (m.idx >= m.ncols).any()) | 4 * order


@pytest.mark.parametrize("shape", sorted(SHAPES))
@pytest.mark.parametrize("fault", ["short", "long", "descent", "negative", "first"])
def test_entries_under_malformed_pointers(ctx, shape, fault):
    """A tile's entries are judged all the same where its pointers are wrong."""
    m = _rows(SHAPES[shape], 1 << 20)
    at, v = {"short": (-1, m.nnz // 2), "long": (-1, m.nnz + 5), "descent": (len(m.ptr) // 2, 1),
             "negative": (len(m.ptr) // 2, -7), "first": (0, 2)}[fault]
    q = m.ptr.copy()
    q[at] = v
    for place, value in ((None, 0), (m.nnz - 1, 1 << 20), (m.nnz - 1, -1), (m.nnz - 2, 1 << 19)):
        c = m.idx.copy()
        if place is not None:
            c[place] = value
        t = Csr(m.nrows, m.ncols, q, c, m.val)
        assert _status(ctx, t) == _status_by_definition(t), (place, value)
