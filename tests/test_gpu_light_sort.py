"""Light rows at the edges of their classes (sorted up to 256, 512 and 1024
products a row): bit-exact against the oracle with values over 2^+-20, so
that a sum in another order shows; rows that meet few columns often, rows of
many A entries whose B rows are mostly empty, narrow outputs, and outputs too
wide for a 32-bit (column, position) key."""
import numpy as np
import pytest

import oracle
from trident_amd.device import spgemm
from trident_amd.gen import Csr

pytestmark = pytest.mark.gpu

PRODUCTS = [128, 129, 130, 255, 256, 257, 511, 512, 513, 1000, 1023, 1024]


def _values(rng, n):
    return rng.uniform(-1, 1, n) * np.exp2(rng.integers(-20, 21, n))


def _csr(rows, ncols, rng):
    ptr = np.zeros(len(rows) + 1, np.int64)
    np.cumsum([len(r) for r in rows], out=ptr[1:])
    idx = np.concatenate([np.asarray(r, np.int64) for r in rows] + [np.zeros(0, np.int64)])
    return Csr(len(rows), ncols, ptr.astype(np.int32), idx.astype(np.int32), _values(rng, int(ptr[-1])))


def _check(ctx, a, b):
    da, db = ctx.upload(a), ctx.upload(b)
    c = spgemm(da, db)
    h = c.download()
    p, i, v = oracle.spgemm(a, b)
    assert np.array_equal(h.ptr, p) and np.array_equal(h.idx, i) and np.array_equal(h.val, v)
    for x in (c, da, db):
        x.free()


@pytest.mark.parametrize("ncols", [131, 300, 1100, 1 << 18, (1 << 22) - 1, 1 << 22, (1 << 22) + 1])
@pytest.mark.parametrize("row_len", [1, 3, 40, 128])
def test_class_edges(ctx, row_len, ncols):
    """A rows of exactly n products for each n, over B rows of about row_len."""
    rng = np.random.default_rng(row_len * 7 + ncols)
    rows_b, rows_a = [], []
    span = min(ncols, max(2 * row_len, 200))  # columns met again and again
    for n in PRODUCTS:
        row = []
        while n > 0:
            m = min(n, row_len)
            row.append(len(rows_b))
            cols = np.sort(rng.choice(span, m, replace=False))
            if ncols >= 2 * span:  # the same few columns, spread to the far end
                cols = np.sort(np.where(cols % 5 == 0, ncols - 1 - cols, cols))
            rows_b.append(cols)
            n -= m
        rows_a.append(row)
    a, b = _csr(rows_a, len(rows_b), rng), _csr(rows_b, ncols, rng)
    _check(ctx, a, b)


def test_many_entries_few_products(ctx):
    """Rows of thousands of A entries, nearly all over empty B rows."""
    rng = np.random.default_rng(5)
    nb = 6000
    rows_b = [np.sort(rng.choice(5000, 2, replace=False)) if k % 13 == 0 else [] for k in range(nb)]
    rows_a = [np.sort(rng.choice(nb, m, replace=False)) for m in (900, 1700, 3000, 6000 // 2, 5999)] + [[0], []]
    _check(ctx, _csr(rows_a, nb, rng), _csr(rows_b, 5000, rng))


@pytest.mark.parametrize("nrows", [32767, 32768, 32775, 33001])
@pytest.mark.parametrize("span", [6, 32, 33, 64, 5000])
def test_short_rows(ctx, nrows, span):
    """Eight rows to a wave, in products of 32768 rows and more: many A entries
    over B rows of 2 to 10 entries on average (some empty, some over eight), at
    most 128 products, over about `span` columns (sorted beyond 32 entries),
    rows of other classes between them."""
    rng = np.random.default_rng(nrows * 100 + span)
    nb = 400
    lens = rng.choice([0, 1, 2, 4, 5, 7, 8, 9, 16, 17], nb)
    rows_b = [np.sort(rng.choice(span, min(m, span), replace=False)) * 7 for m in lens]
    rows_a = []
    for r in range(600):
        row, f = [], 0
        target = int(rng.choice([8, 40, 100, 127, 128, 128, 200]))
        for k in rng.permutation(nb):
            if f + len(rows_b[k]) <= target:
                row.append(k)
                f += len(rows_b[k])
            if len(row) >= 60 or f == target:
                break
        rows_a.append(np.sort(row))
    pick = rng.integers(0, 600, nrows)
    _check(ctx, _csr([rows_a[i] for i in pick], nb, rng), _csr(rows_b, 7 * span + 1, rng))


@pytest.mark.parametrize("repeats", [1, 3000])
@pytest.mark.parametrize("ncols", [300, (1 << 22) + 1])
def test_classes_together(ctx, repeats, ncols):
    """Every light class in one product: few rows share a launch, many do not."""
    rng = np.random.default_rng(repeats + ncols)
    cols = np.sort(rng.choice(ncols, 200, replace=False)) if ncols > 1000 else np.arange(50, 250)
    rows_b = [np.sort(rng.choice(cols, n, replace=False)) for n in (1, 2, 7, 31, 64, 150)]
    sizes = [1, 31, 32, 33, 64, 65, 128, 129, 256, 257, 512, 513, 1024]
    spread = [r for _ in range(120) for r in rows_b]  # B's rows again and again
    rows_a = []
    for n in sizes:
        row, i = [], 0
        while n > 0:
            if len(spread[i]) <= n:
                row.append(i)
                n -= len(spread[i])
            i += 1
        rows_a.append(row)
    a, b = _csr(rows_a * repeats, len(spread), rng), _csr(spread, ncols, rng)
    _check(ctx, a, b)
