"""Compression at the edges of its work units (2048 segment ends plus
entries): segments that span several units, runs of empty segments longer than
a unit, everything or nothing kept; exact against the oracle."""
import numpy as np
import pytest

import oracle
from trident_amd._lib import TR_COLS, TR_ROWS
from trident_amd.device import Batch, SpaComm
from trident_amd.gen import Csr

pytestmark = pytest.mark.gpu


def _matrix(lens, other, seed):
    rng = np.random.default_rng(seed)
    lens = np.asarray(lens, np.int64)
    ptr = np.zeros(len(lens) + 1, np.int64)
    np.cumsum(lens, out=ptr[1:])
    idx = np.concatenate([np.sort(rng.choice(other, n, replace=False)) for n in lens] + [np.zeros(0, np.int64)])
    return Csr(len(lens), other, ptr.astype(np.int32), idx.astype(np.int32), rng.standard_normal(int(ptr[-1])))


SHAPES = {
    "one": [1],
    "unit": [3] * 512,                                     # 512 * (3 + 1) = one unit exactly
    "unit_plus": [3] * 512 + [1],
    "long": [5, 0, 7000, 1, 0, 0, 2047, 2048, 2049, 3],    # segments over several units
    "gap": [4] + [0] * 5000 + [4] + [0] * 4095,            # units of empty segments
    "words": [63, 64, 65, 1, 127, 128, 129, 0, 62] * 20,   # segment edges at 64-entry words
}


@pytest.mark.parametrize("keep", ["all", "none", "some"])
@pytest.mark.parametrize("shape", sorted(SHAPES))
def test_compress_units(ctx, shape, keep):
    m = _matrix(SHAPES[shape], 8000, 1)
    n = m.nrows
    k = {"all": np.ones(n, bool), "none": np.zeros(n, bool),
         "some": np.random.default_rng(2).random(n) < 0.5}[keep]
    mask = np.packbits(np.append(k, np.zeros(-n % 64, bool)), bitorder="little").view(np.uint64)
    p, i, v = oracle.compress(n, m.ptr, m.idx, m.val, mask)
    dm = ctx.to_device(mask)
    for major in (TR_ROWS, TR_COLS):
        x = m if major == TR_ROWS else Csr(m.ncols, m.nrows, m.ptr, m.idx, m.val)
        d = ctx.upload(x, major)
        out = SpaComm.compress(d, dm)
        h = out.download()
        assert np.array_equal(h.ptr, p) and np.array_equal(h.idx, i) and np.array_equal(h.val, v)
        out.free()
        d.free()
    ctx.free(dm)


def test_batch_compress_units(ctx):
    """Tasks that share tiles, have their own, and have empty ones; an A with
    hub columns (one set bit met by every entry) and rows longer than a unit."""
    inner = 4100
    hub = np.zeros(600, np.int64)
    hub[:] = 2
    a0 = _matrix(hub, inner, 3)
    a0.idx[0::2], a0.idx[1::2] = 7, 4099
    a1 = _matrix([0, 3000, 1, 4100, 0], inner, 4)
    empty = Csr(5, inner, np.zeros(6, np.int32), np.zeros(0, np.int32), np.zeros(0))
    b0 = _matrix(np.random.default_rng(5).integers(0, 3, inner), 900, 5)
    b1 = _matrix([0] * 4000 + [5] * 100, 900, 6)
    pairs = [(a0, b0), (a0, b1), (a1, b0), (a1, b1), (empty, b0)]
    dev = {id(m): ctx.upload(m) for m in (a0, a1, empty, b0, b1)}
    batch = Batch(ctx, [dev[id(a)] for a, _ in pairs], [dev[id(b)] for _, b in pairs], compress=True)
    for _ in range(3):
        batch.run()
        batch.check()
        for t, (a, b) in enumerate(pairs):
            h = batch.result(t).download()
            p, i, v = oracle.spgemm(a, b)
            assert np.array_equal(h.ptr, p) and np.array_equal(h.idx, i) and np.array_equal(h.val, v)
    batch.close()
    for d in dev.values():
        d.free()
