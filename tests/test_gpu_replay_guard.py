"""Replays of a batch whose operands no longer have the planned sparsity
pattern: the run stays inside the plan's buffers, tr_batch_check reports it,
and the planned pattern makes runs valid again."""
import numpy as np
import pytest

import oracle
from trident_amd import gen
from trident_amd._lib import TR_ERR_INVALID, TridentError
from trident_amd.device import Batch

pytestmark = pytest.mark.gpu


def _rows(rows, ncols, rng):
    ptr = np.concatenate([[0], np.cumsum([len(r) for r in rows])])
    return gen.from_arrays(len(rows), ncols, ptr, np.concatenate(rows), rng.uniform(-1, 1, ptr[-1]))


def _exact(batch, a, b):
    p, i, v = oracle.spgemm(a, b)
    h = batch.result(0).download()
    return np.array_equal(h.ptr, p) and np.array_equal(h.idx, i) and np.array_equal(h.val, v)


def _put_columns(ctx, d, idx):
    idx = np.ascontiguousarray(idx, np.int32)
    ctx.check(ctx.lib.tr_memcpy_h2d(ctx.h, d.d.idx_vec, idx.ctypes.data, idx.nbytes))


def _refused_then_valid(ctx, batch, da, a, b, changed_idx):
    try:
        assert _exact(batch, a, b)
        _put_columns(ctx, da, changed_idx)
        batch.run()
        with pytest.raises(TridentError) as e:
            batch.check()
        assert e.value.code == TR_ERR_INVALID
        _put_columns(ctx, da, a.idx)
        batch.run()
        batch.check()
        assert _exact(batch, a, b)
    finally:
        batch.close()


@pytest.mark.parametrize("graph", [True, False])
def test_more_windows_than_planned(ctx, graph):
    """Heavy rows that met B rows of 3 entries meet B rows of 2000 instead:
    their windows and items are ten times what the work lists hold, so that
    most rows are refused and what the lists hold must not be used."""
    rng = np.random.default_rng(1)
    ncols, rows, entries = 100000, 64, 400
    b = _rows([np.sort(rng.choice(ncols, 3 if k < entries else 2000, replace=False)) for k in range(2 * entries)],
              ncols, rng)
    a = _rows([np.arange(entries) for _ in range(rows)], 2 * entries, rng)
    da, db = ctx.upload(a), ctx.upload(b)
    batch = Batch(ctx, [da], [db], None, graph=graph)
    _refused_then_valid(ctx, batch, da, a, b, np.tile(np.arange(entries, 2 * entries), rows))
    da.free()
    db.free()


@pytest.mark.parametrize("graph", [True, False])
def test_rows_that_no_planned_launch_takes(ctx, graph):
    """Short rows of 32 entries, the most that their kernel takes; then one row
    of 48, which the plan has no launch for, and one of 16, so that every size
    of the plan still fits."""
    rng = np.random.default_rng(2)
    rows, sets = 32768, 16  # B rows 4 s .. 4 s + 3 hold the columns of set s
    b = _rows([4 * (k // 4) + np.arange(4) for k in range(4 * sets)], 4 * sets, rng)
    planned = np.concatenate([[4 * s, 4 * s + 1] for s in range(8)])
    a = _rows([planned] * rows, 4 * sets, rng)
    more = np.concatenate([[4 * s, 4 * s + 1] for s in range(4)] + [[4 * s] for s in range(4, 12)])
    less = np.arange(16)
    da, db = ctx.upload(a), ctx.upload(b)
    batch = Batch(ctx, [da], [db], None, graph=graph)
    _refused_then_valid(ctx, batch, da, a, b, np.concatenate([more, less, a.idx[32:]]))
    da.free()
    db.free()
