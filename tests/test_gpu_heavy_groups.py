"""Heavy rows whose products meet in the same columns: bit-exact against the
oracle with values over 2^+-20, so that a sum in another order shows.  Products
of one A entry fall in groups of 64 of every wave, columns are met once, by two
entries, or by every entry, next to each other or rounds apart, and a batch
holds more products than a round of marks (4096)."""
import numpy as np
import pytest

import oracle
from trident_amd.device import Context, spgemm, tuning_default
from trident_amd.gen import Csr

pytestmark = pytest.mark.gpu


def _csr(rows, ncols, rng):
    ptr = np.zeros(len(rows) + 1, np.int64)
    np.cumsum([len(r) for r in rows], out=ptr[1:])
    idx = np.concatenate([np.asarray(r, np.int64) for r in rows])
    n = int(ptr[-1])
    return Csr(len(rows), ncols, ptr.astype(np.int32), idx.astype(np.int32),
               rng.uniform(-1, 1, n) * np.exp2(rng.integers(-20, 21, n)))


@pytest.mark.parametrize("table", [2048, 4096])
@pytest.mark.parametrize("kind", ["one_column", "pairs", "all_equal", "few_columns", "spread"])
@pytest.mark.parametrize("entries", [65, 255, 256, 257, 513, 700])
def test_shared_slots(kind, entries, table):
    rng = np.random.default_rng(entries)
    ncols = 60000
    if kind == "one_column":  # every entry meets column 7, and columns of its own
        rows = [np.r_[7, 100 + 40 * k + np.arange(40)] for k in range(entries)]
    elif kind == "pairs":  # entry k and k + 1 share half of their columns
        rows = [100 + 32 * k + np.arange(64) for k in range(entries)]
    elif kind == "all_equal":
        rows = [np.arange(0, 1800, 2)] * entries
    elif kind == "few_columns":
        rows = [np.sort(rng.choice(90, 33, replace=False)) + 1000 for _ in range(entries)]
    else:
        rows = [np.sort(rng.choice(ncols, 50, replace=False)) for _ in range(entries)]
    b = _csr(rows, ncols, rng)
    a = _csr([np.arange(entries), np.arange(0, entries, 2), np.arange(entries)], entries, rng)
    p, i, v = oracle.spgemm(a, b)
    with Context(0) as ctx:
        if table == 4096:
            ctx.set_tuning(dict(tuning_default(), heavy_table=4096, window_entries=1920, dense_width=4096))
        c = spgemm(ctx.upload(a), ctx.upload(b)).download()
    assert np.array_equal(c.ptr, p) and np.array_equal(c.idx, i) and np.array_equal(c.val, v)


@pytest.mark.parametrize("ncols", [400, 300000, 600000])
def test_b_row_lengths(ctx, ncols):
    """Heavy rows over B rows of every length around those that are taken four
    at a time (up to 128 columns), in any order, empty ones between them."""
    rng = np.random.default_rng(ncols)
    lens = [n for n in (0, 1, 15, 16, 17, 32, 33, 63, 64, 65, 112, 113, 127, 128, 129, 191, 255, 256, 257, 300) for _ in range(40)]
    rng.shuffle(lens)
    b = _csr([np.sort(rng.choice(ncols, n, replace=False)) for n in lens], ncols, rng)
    some = [np.sort(rng.choice(len(lens), k, replace=False)) for k in (20, 63, 64, 65, 500, 513, 800)]
    only = [np.flatnonzero(np.array(lens) == n) for n in (128, 129, 300)]
    a = _csr(some + only, len(lens), rng)
    p, i, v = oracle.spgemm(a, b)
    da, db = ctx.upload(a), ctx.upload(b)
    d = spgemm(da, db)
    c = d.download()
    assert np.array_equal(c.ptr, p) and np.array_equal(c.idx, i) and np.array_equal(c.val, v)
    for x in (d, da, db):
        x.free()
