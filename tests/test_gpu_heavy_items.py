"""Heavy rows of several column passes cut into items at the ends of the tuning
range: the work lists hold them and the products equal the oracle's."""
import numpy as np
import pytest

import oracle
from trident_amd import gen
from trident_amd.device import Context, spgemm, tuning_default

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b_rows,window_entries,item_windows", [
    (16, 64, 64),    # 16000 multiplications: sixteen passes of 2^19 columns
    (16, 1152, 64),  # sparse passes
    (200, 64, 64),   # 200000: eight passes of 2^20 columns
    (200, 257, 16),
])
def test_items_of_many_passes(b_rows, window_entries, item_windows):
    rng = np.random.default_rng(b_rows)
    ncols, rows = 1 << 23, 4
    bl = [np.unique(rng.integers(0, ncols, 1000)) for _ in range(b_rows)]
    ptr = np.concatenate([[0], np.cumsum([len(x) for x in bl])])
    b = gen.from_arrays(b_rows, ncols, ptr, np.concatenate(bl), rng.uniform(-1, 1, ptr[-1]))
    a = gen.from_arrays(rows, b_rows, np.arange(rows + 1) * b_rows, np.tile(np.arange(b_rows), rows),
                        rng.uniform(-1, 1, rows * b_rows))
    p, i, v = oracle.spgemm(a, b)
    with Context(0) as c:
        c.set_tuning(dict(tuning_default(), window_entries=window_entries, item_windows=item_windows))
        h = spgemm(c.upload(a), c.upload(b)).download()
    assert np.array_equal(h.ptr, p) and np.array_equal(h.idx, i) and np.array_equal(h.val, v)
