"""Row offsets at the edges of the scan's forms: one workgroup (up to 16384
items), tiles that sum the totals before them (up to 2048 tiles of 4096), and
scanned totals beyond.  Seen through tr_compress, whose row pointer is the
scan of the kept segment lengths; exact."""
import numpy as np
import pytest

from trident_amd.device import SpaComm
from trident_amd.gen import Csr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 64, 1023, 1025, 16383, 16384, 16385, 20481, 2048 * 4096, 2048 * 4096 + 1])
def test_row_offsets(ctx, n):
    rng = np.random.default_rng(n)
    ln = (rng.random(n) < min(1.0, 3e5 / n)) * rng.integers(1, 4, n)
    ln[-1] = 2  # the last item counts
    ptr = np.zeros(n + 1, np.int64)
    np.cumsum(ln, out=ptr[1:])
    nnz = int(ptr[-1])
    first = np.repeat(ptr[:-1], ln)
    m = Csr(n, 8, ptr.astype(np.int32), (np.arange(nnz) - first).astype(np.int32), rng.standard_normal(nnz))
    keep = rng.random(n) < 0.7
    keep[-1] = True
    padded = np.append(keep, np.zeros(-n % 64, bool))
    mask = np.packbits(padded, bitorder="little").view(np.uint64)
    d, dm = ctx.upload(m), ctx.to_device(mask)
    out = SpaComm.compress(d, dm)
    got = out.download()
    want = np.zeros(n + 1, np.int64)
    np.cumsum(ln * keep, out=want[1:])
    sel = np.repeat(keep, ln)
    assert np.array_equal(got.ptr, want)
    assert np.array_equal(got.idx, m.idx[sel]) and np.array_equal(got.val, m.val[sel])
    out.free()
    d.free()
    ctx.free(dm)
