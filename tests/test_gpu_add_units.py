"""The sorted add at the edges of its work units (512 row ends plus merged
entries): rows that span units, runs of empty rows longer than a unit, pairs of
equal columns that a unit's edge parts, and faults planted at each entry around
an edge, against the oracle, bit for bit."""
import ctypes

import numpy as np
import pytest

import oracle
from trident_amd._lib import TR_ERR_INVALID, TR_ERR_OOM, TridentError, tr_csx_t
from trident_amd.device import spadd
from trident_amd.gen import Csr

pytestmark = pytest.mark.gpu


def _csr(rows, ncols, rng):
    ptr = np.zeros(len(rows) + 1, np.int64)
    np.cumsum([len(r) for r in rows], out=ptr[1:])
    idx = np.concatenate([np.asarray(r, np.int64) for r in rows] + [np.zeros(0, np.int64)])
    val = rng.uniform(-1, 1, int(ptr[-1])) * np.exp2(rng.integers(-20, 21, int(ptr[-1])))
    return Csr(len(rows), ncols, ptr.astype(np.int32), idx.astype(np.int32), val)


def _check(ctx, a, c):
    da, dc = ctx.upload(a), ctx.upload(c)
    spadd(da, dc)
    h = dc.download()
    p, i, v = oracle.spadd(a, c)
    assert np.array_equal(h.ptr, p) and np.array_equal(h.idx, i) and np.array_equal(h.val, v)
    da.free()
    dc.free()


@pytest.mark.parametrize("lead", [0, 1, 2, 3, 4, 5, 1021, 1022, 1023])
@pytest.mark.parametrize("kind", ["same", "one_sided", "alternating", "mixed"])
def test_pairs_at_unit_edges(ctx, kind, lead):
    """One row over many units after `lead` single entries or empty rows, so
    that every unit edge falls at each place of a pair; more rows behind it."""
    rng = np.random.default_rng(lead * 5 + len(kind))
    n = 3000
    cols = np.arange(n) * 2
    x, y = {"same": (cols, cols), "one_sided": (cols, cols[:0]), "alternating": (cols, cols + 1),
            "mixed": (np.sort(rng.choice(8000, n, replace=False)), np.sort(rng.choice(8000, n, replace=False)))}[kind]
    tail = [np.sort(rng.choice(8000, k, replace=False)) for k in (1, 0, 7, 0, 0, 300, 2)]
    single = [rng.integers(0, 8000, 1) if r % 3 else [] for r in range(lead)]
    none = [[] for _ in range(lead)]
    _check(ctx, _csr(single + [x] + tail, 8000, rng), _csr(none + [y] + tail[::-1], 8000, rng))
    _check(ctx, _csr(none + [y] + tail, 8000, rng), _csr(single + [x] + tail, 8000, rng))


@pytest.mark.parametrize("ncols", [4000, 1 << 21, (1 << 21) + 1, (1 << 31) - 1])
@pytest.mark.parametrize("shape", ["short", "empty_runs", "all_empty", "one_entry"])
def test_rows_and_gaps(ctx, shape, ncols):
    """Also at the widest tile of 32-bit merge keys and beyond it."""
    rng = np.random.default_rng(len(shape))
    if shape == "short":
        lens = rng.integers(0, 9, (2, 5000))
    elif shape == "empty_runs":
        lens = np.zeros((2, 9000), np.int64)
        lens[0, [0, 2100, 8999]] = [1500, 3, 1]
        lens[1, [0, 5000, 8999]] = [1500, 2000, 1]
    else:
        lens = np.zeros((2, 1024), np.int64)
        if shape == "one_entry":
            lens[1, 1023] = 1
    mk = lambda ls: _csr([np.sort(rng.choice(4000, k, replace=False)) * (ncols - 1) // 3999 for k in ls], ncols, rng)
    _check(ctx, mk(lens[0]), mk(lens[1]))


def test_merged_in_parts(ctx):
    """With room for the merge of a part of the units only, they are merged
    again part by part, with the same result."""
    from trident_amd.device import Context

    rng = np.random.default_rng(9)
    lens = rng.integers(0, 3000, (2, 7500))
    a, b = (_csr([np.sort(rng.choice(6000, k, replace=False)) for k in ls], 6000, rng) for ls in lens)
    p, i, v = oracle.spadd(a, b)
    units = (a.nrows + a.nnz + b.nnz) // 512 + 1  # 128 bytes of merge and 20 of places each
    granule = 2 << 20                              # of the pool
    out = -(-(12 * len(i) + 4 * (a.nrows + 1)) // granule) * granule
    for room in (out + 5 * granule, out + 2 * granule, out // 2):
        with Context(0) as c:
            da, db = c.upload(a), c.upload(b)
            c.set_pool_limit(c.pool_stats()[0] + room)
            if room < out:
                with pytest.raises(TridentError) as e:
                    spadd(da, db)
                assert e.value.code == TR_ERR_OOM
                continue
            spadd(da, db)
            h = db.download()
            assert np.array_equal(h.ptr, p) and np.array_equal(h.idx, i) and np.array_equal(h.val, v)
    with Context(0) as c:  # into caller arrays: the merge itself has too little room
        da, db = c.upload(a), c.upload(b)
        d = tr_csx_t()
        d.ptr_vec, d.idx_vec, d.val = c.malloc(4 * (a.nrows + 1)), c.malloc(4 * len(i)), c.malloc(8 * len(i))
        need = ctypes.c_int64(-1)
        c.set_pool_limit(c.pool_stats()[0] + 100 * units)
        rc = c.lib.tr_spadd_into(c.h, ctypes.byref(da.d), ctypes.byref(db.d), ctypes.byref(d), len(i), ctypes.byref(need))
        c.check(rc, "tr_spadd_into")
        assert need.value == len(i)
        assert np.array_equal(c.to_host(d.ptr_vec, a.nrows + 1, np.int32), p)
        assert np.array_equal(c.to_host(d.idx_vec, len(i), np.int32), i)
        assert np.array_equal(c.to_host(d.val, len(i), np.float64), v)


@pytest.mark.parametrize("side", [0, 1])
def test_faults_at_unit_edges(ctx, side):
    rng = np.random.default_rng(side)
    cols = np.arange(4000) * 2
    m = [_csr([cols, cols[:5]], 9000, rng), _csr([cols + 1, cols[:5]], 9000, rng)]
    for p in (1, 510, 511, 512, 513, 1023, 1024, 2047, 2048, 3999):
        for bad in (m[side].idx[p - 1], -1, 9000):
            c = m[side].idx.copy()
            c[p] = bad
            t = list(m)
            t[side] = Csr(2, 9000, m[side].ptr, c, m[side].val)
            d = [ctx.upload(k) for k in t]
            with pytest.raises(TridentError) as e:
                spadd(d[0], d[1])
            assert e.value.code == TR_ERR_INVALID, (p, bad)
            for k in d:
                k.free()
    _check(ctx, m[0], m[1])  # a descent between rows is none
