"""Transposition under a pool limit: without room for the records of all
entries it goes by ranges of destinations, few of them if little is missing,
with the same result as without a limit (exact against a stable sort)."""
import numpy as np
import pytest

from trident_amd.device import Context
from trident_amd.gen import Csr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("other,hub,sweeps", [
    # Room for 10 bytes an entry.  Counts and offsets take at most 12 << 10
    # bytes a tile of 4096 entries (3 an entry), an entry of a range 20 (36 of
    # three digits) and its blocks up to a third more in granules: an eighth of
    # the destinations fits, so eight ranges of at most three counts, and one
    # for each halving on the way.
    (1 << 20, 0.0, 8 * 3 + 3),
    # (two digits for 2^20 destinations or fewer, so the eighth holds here too)
    (1 << 22, 0.0, 16 * 3 + 5),
    # 30% in one destination: down to a single digit around it (11 halvings)
    # and up again (as many doublings)
    (1 << 20, 0.3, 8 * 3 + 11 + 11 * 3),
])
def test_ranges_follow_the_missing_room(other, hub, sweeps):
    rng = np.random.default_rng(other)
    nseg, nnz = 500, 2000000
    ptr = np.concatenate([[0], np.cumsum(np.bincount(rng.integers(0, nseg, nnz), minlength=nseg))])
    idx = rng.integers(0, other, nnz)
    idx[rng.random(nnz) < hub] = other // 2
    m = Csr(nseg, other, ptr.astype(np.int32), idx.astype(np.int32), rng.standard_normal(nnz))
    order = np.argsort(idx, kind="stable")
    want_ptr = np.concatenate([[0], np.cumsum(np.bincount(idx, minlength=other))])
    with Context(0) as c:
        d = c.upload(m)
        held = c.pool_stats()[0]
        c.set_pool_limit(held + 12 * nnz + 4 * (other + 1) + 10 * nnz)
        c.set_timing(True)
        c.reset_timing()
        t = d.transpose()
        counts = c.timings()["transpose_count"][0]
        c.set_timing(False)
        h = t.download()
        t.free()
        d.free()
    assert np.array_equal(h.ptr, want_ptr) and np.array_equal(h.idx, m.row_ids()[order])
    assert np.array_equal(h.val, m.val[order])
    assert counts <= sweeps
