"""Sparse products whose long rows accumulate in LDS, a wavefront per column
tile: pattern, column order and every bit equal the oracle's at the edges of
the tiles, of the column limit and of the rules that choose the form.
"""
import numpy as np
import pytest

import bootcmatchg_amd as bc
from oracle import oracle as orc

from common import bits

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = bc.Context(0)
    yield c
    c.close()


def rows(rng, n, m, lengths, special=False):
    """CSR with the given row lengths, ascending distinct columns; special:
    zeros of both signs, subnormals and large values among the entries."""
    col = [np.sort(rng.choice(m, min(k, m), replace=False)) for k in lengths]
    row = np.concatenate(([0], np.cumsum([len(c) for c in col])))
    val = rng.uniform(-1, 1, row[-1])
    if special:
        pick = np.array([0.0, -0.0, 5e-324, -3e-310, 1e300, 1e-200])
        at = rng.random(row[-1]) < 0.3
        val[at] = rng.choice(pick, at.sum())
    return row.astype(np.int32), np.concatenate(col).astype(np.int32), val


@pytest.mark.parametrize("m", [64, 1000, 1024, 1025, 4160, 16383, 16384, 16385])
@pytest.mark.parametrize("per_pass", [0, 9000])
def test_tiles(ctx, m, per_pass):
    """Right rows of 0 to m entries (segments of 0, 1, 63, 64, 65 and more
    than eight times 64 entries), short and long left rows, few and many
    products per left entry."""
    rng = np.random.default_rng(m)
    k = 150
    R = rows(rng, k, m, [0, m, min(m, 700)] + list(rng.integers(0, min(m, 130), k - 3)), True)
    L = rows(rng, 40, k, [0, 1, 1, 2, 64, 65, 128, 150] + list(rng.integers(1, k, 32)), True)
    row, col, val = bc.spgemm(ctx, L, R, m, slots_per_pass=per_pass).download()
    orow, ocol, oval = orc.spgemm(L, R, m)
    assert np.array_equal(row, orow)
    assert np.array_equal(col, ocol)
    assert np.array_equal(bits(val), bits(oval))


@pytest.mark.parametrize("per_entry", [2, 5, 40])
def test_short_right_rows(ctx, per_entry):
    """Long rows on both sides of the products-per-left-entry rule in one
    product, and right rows too short for tile pointers."""
    rng = np.random.default_rng(per_entry)
    m, k = 10000, 1500
    R = rows(rng, k, m, [per_entry] * (k // 2) + [12 * per_entry] * (k - k // 2))
    L = rows(rng, 20, k, [1400, 1200, 900, 700] * 5)
    row, col, val = bc.spgemm(ctx, L, R, m).download()
    orow, ocol, oval = orc.spgemm(L, R, m)
    assert np.array_equal(row, orow)
    assert np.array_equal(col, ocol)
    assert np.array_equal(bits(val), bits(oval))
