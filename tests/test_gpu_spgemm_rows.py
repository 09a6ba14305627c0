"""Sparse products with so many right rows that a wavefront a row passes the
lanes of one launch."""
import numpy as np
import pytest

import bootcmatchg_amd as bc

from common import bits

pytestmark = pytest.mark.gpu


def test_more_than_2_to_the_26_right_rows():
    """One long left row against 2^26 + 100 right rows of an entry each (64
    columns): the column tiles of every right row are found, those past 2^26
    too."""
    n, cols = (1 << 26) + 100, 64
    ctx = bc.Context(0)
    rng = np.random.default_rng(4)
    pick = np.unique(np.concatenate([rng.integers(0, n, 3000), np.arange(n - 60, n)]))
    lv = rng.uniform(-1, 1, len(pick))
    rcol = (np.arange(n, dtype=np.int64) * 37 % cols).astype(np.int32)
    rv = np.full(n, 0.5)
    rv[pick] = rng.uniform(-1, 1, len(pick))
    C = bc.spgemm(ctx, (np.array([0, len(pick)], np.int32), pick.astype(np.int32), lv),
                  (np.arange(n + 1, dtype=np.int32), rcol, rv), cols)
    row, col, val = C.download()
    want = np.zeros(cols)
    for k, l in zip(pick, lv):
        want[rcol[k]] = want[rcol[k]] + l * rv[k]
    assert np.array_equal(row, [0, cols]) and np.array_equal(col, np.arange(cols))
    assert np.array_equal(bits(val), bits(want))
    ctx.close()
