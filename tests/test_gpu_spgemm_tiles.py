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


def same(val, oval):
    nan = np.isnan(oval)
    return np.array_equal(np.isnan(val), nan) and np.array_equal(bits(val[~nan]), bits(oval[~nan]))


@pytest.mark.parametrize("n,k,m,fl,fr,special", [
    (16, 160, 128, 0.5, 0.5, True),       # one tile, one column block
    (17, 161, 129, 0.6, 0.4, True),       # a row and a column beyond them
    (8, 160, 128, 0.5, 0.5, True),        # fewer rows than a tile
    (9, 161, 129, 0.6, 0.4, True),
    (67, 300, 1000, 0.9, 0.2, False),
    (130, 1025, 640, 0.3, 0.35, True),
    (40, 200, 300, 0.05, 0.9, False),     # below the fill that is taken
])
@pytest.mark.parametrize("change", ["", "infinite", "left order", "a short row"])
def test_dense_operands(ctx, n, k, m, fl, fr, special, change):
    """Well-filled operands, and what keeps the other form: a value that is
    not finite, left rows out of order, a short row among long ones."""
    rng = np.random.default_rng(n + k)
    L = rows(rng, n, k, np.maximum(20, rng.binomial(k, fl, n)), special)
    R = rows(rng, k, m, np.maximum(60, rng.binomial(m, fr, k)), special)
    if change == "infinite":
        L[2][len(L[2]) // 2] = np.inf
    elif change == "left order":
        for i in range(0, n, 3):
            s = slice(L[0][i], L[0][i + 1])
            p = rng.permutation(s.stop - s.start)
            L[1][s], L[2][s] = L[1][s][p], L[2][s][p]
    elif change == "a short row":
        L = rows(rng, n, k, np.r_[1, np.maximum(20, rng.binomial(k, fl, n - 1))], special)
    row, col, val = bc.spgemm(ctx, L, R, m).download()
    with np.errstate(all="ignore"):
        orow, ocol, oval = orc.spgemm(L, R, m)
    assert np.array_equal(row, orow)
    assert np.array_equal(col, ocol)
    assert same(val, oval)


@pytest.mark.parametrize("m", [1500, 60000])
@pytest.mark.parametrize("stride", [8, 4, 1])
def test_hashed_rows(ctx, m, stride):
    """Right row k holds the eight columns from stride k on, so a left row of t
    entries has 8 t products and 8 + stride (t - 1) columns: tables just full
    and one entry too small, rows on both sides of each product bound."""
    rng = np.random.default_rng(stride)
    k = (m - 8) // stride + 1
    col = (np.arange(k)[:, None] * stride + np.arange(8)).ravel()
    R = (np.arange(0, 8 * k + 1, 8).astype(np.int32), col.astype(np.int32),
         rng.uniform(-1, 1, 8 * k))
    counts = [t for t in (0, 1, 63, 64, 65, 127, 128, 129, 255, 256, 300, 1017, 1018) if t <= k]
    row = np.concatenate(([0], np.cumsum(counts))).astype(np.int32)
    start = [int(rng.integers(0, k - t + 1)) for t in counts]
    L = (row, np.concatenate([np.arange(s, s + t) for s, t in zip(start, counts)])
         .astype(np.int32), rng.uniform(-1, 1, row[-1]))
    crow, ccol, cval = bc.spgemm(ctx, L, R, m).download()
    orow, ocol, oval = orc.spgemm(L, R, m)
    assert np.array_equal(crow, orow)
    assert np.array_equal(ccol, ocol)
    assert np.array_equal(bits(cval), bits(oval))
