"""Transposition at the edges of its passes (one digit up to 2^10
destinations, two up to 2^20, three beyond) and tiles (4096 entries), with hub
destinations, long runs of empty source segments and entries in any order
inside a segment; exact against a stable sort."""
import numpy as np
import pytest

from trident_amd._lib import TR_COLS, TridentError
from trident_amd.gen import Csr

pytestmark = pytest.mark.gpu


def _entries(nseg, other, nnz, seed, hub=0.0):
    """A matrix with `nnz` entries in random segments, in random order inside
    them, a share of them in one destination."""
    rng = np.random.default_rng(seed)
    seg = np.sort(rng.integers(0, nseg, nnz))
    ptr = np.zeros(nseg + 1, np.int64)
    np.cumsum(np.bincount(seg, minlength=nseg), out=ptr[1:])
    idx = rng.integers(0, other, nnz)
    idx[rng.random(nnz) < hub] = other // 2
    return Csr(nseg, other, ptr.astype(np.int32), idx.astype(np.int32), rng.standard_normal(nnz))


def _want(m):
    order = np.argsort(m.idx, kind="stable")
    ptr = np.zeros(m.ncols + 1, np.int64)
    np.cumsum(np.bincount(m.idx, minlength=m.ncols), out=ptr[1:])
    return ptr, m.row_ids()[order], m.val[order]


def _check(h, m):
    p, i, v = _want(m)
    assert np.array_equal(h.ptr, p) and np.array_equal(h.idx, i) and np.array_equal(h.val, v)


@pytest.mark.parametrize("nseg,other,nnz,hub", [
    (1, 1, 1, 0.0), (7, 2, 4095, 0.0), (300, 1023, 4096, 0.5), (300, 1024, 4097, 0.0), (300, 1025, 20000, 0.9),
    (1, 5000, 9000, 0.0), (9000, 1, 9000, 0.0), (60000, 40, 5000, 0.0), (300000, 70000, 30000, 0.3),
    (1000, 1 << 20, 50000, 0.2), (1000, (1 << 20) + 1, 50000, 0.2), (5, (1 << 30) // 8, 12345, 0.0), (10, 10, 0, 0.0),
])
def test_transpose_edges(ctx, nseg, other, nnz, hub):
    m = _entries(nseg, other, nnz, nnz + other, hub)
    d = ctx.upload(m)
    t = d.transpose()
    assert t.shape == (other, nseg)
    _check(t.download(), m)
    t.free()
    d.free()
    # the same arrays as the CSC form of an other x nseg matrix
    c = ctx.upload(Csr(other, nseg, m.ptr, m.idx, m.val), TR_COLS)
    r = c.csc_to_csr()
    assert r.shape == (other, nseg)
    _check(r.download(), m)
    r.free()
    c.free()


@pytest.mark.parametrize("other", [3000, 70000])
def test_transpose_within_a_pool_limit(other):
    """Without room for the records the destinations are taken 1024 at a time,
    with the same result; without room for that either the call fails."""
    from trident_amd.device import Context
    m = _entries(500, other, 400000, other, 0.3)
    with Context(0) as c:
        d = c.upload(m)
        held = c.pool_stats()[0]
        tile = 12 * m.nnz + 4 * (other + 1)
        c.set_pool_limit(held + tile + 18 * m.nnz)  # the records alone are 16 bytes an entry
        t = d.transpose()
        _check(t.download(), m)
        t.free()
        c.set_pool_limit(held + tile + m.nnz)
        with pytest.raises(TridentError):
            d.transpose()
        c.set_pool_limit(0)
        t = d.transpose()
        _check(t.download(), m)
        t.free()
        d.free()
