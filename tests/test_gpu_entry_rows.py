"""Row kernels by entries (irregular operators, small levels): products,
residuals and sweeps equal the serial sum - products rounded, added left to
right - bit for bit, at the edges of the row blocks and of the rules.
"""
import numpy as np
import pytest

import bootcmatchg_amd as bc
from bootcmatchg_amd import operators as ops

from common import bits

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = bc.Context(0)
    yield c
    c.close()


def dev(ctx, a):
    return bc.DeviceArray.from_numpy(ctx, a)


def irregular(n, avg, longest):
    """A diagonal and random entries: rows of 1 to about 2 avg entries, every
    97th of `longest` (as far as n allows), columns ascending."""
    rng = np.random.default_rng(n + avg)
    want = rng.integers(0, 2 * avg - 1, n)
    want[::97] = longest - 1
    r = np.repeat(np.arange(n), np.minimum(want, n - 1))
    near = rng.integers(-300, 301, len(r))
    c = np.where(rng.random(len(r)) < 0.8, np.abs(r + near) % n, rng.integers(0, n, len(r)))
    key = np.unique(np.concatenate((r * n + c, np.arange(n) * (n + 1))))
    row = np.concatenate(([0], np.cumsum(np.bincount(key // n, minlength=n))))
    val = rng.uniform(-1, 1, len(key))
    val[key // n == key % n] += 3.0
    return row.astype(np.int32), (key % n).astype(np.int32), val


def serial(A, x):
    row, col, val = A
    n, length = len(row) - 1, np.diff(row)
    t = np.zeros(n)
    with np.errstate(invalid="ignore", over="ignore"):
        for k in range(length.max()):
            i = np.nonzero(length > k)[0]
            e = row[i] + k
            t[i] = t[i] + val[e] * x[col[e]]
    return t


def same(a, b):
    nan = np.isnan(b)
    return np.array_equal(np.isnan(a), nan) and np.array_equal(bits(a[~nan]), bits(b[~nan]))


@pytest.mark.parametrize("n,avg,longest", [
    (1, 1, 1), (63, 5, 40), (64, 5, 40), (65, 5, 40), (1000, 13, 70), (6351, 8, 51),
    (65536, 12, 30), (65537, 12, 30), (65537, 4, 20), (70000, 9, 20), (200003, 13, 24)])
def test_products_and_sweeps(ctx, n, avg, longest):
    A = irregular(n, avg, longest)
    dA = bc.Csr(ctx, A)
    d = np.add.reduceat(np.abs(A[2]), A[0][:-1])
    f, x = ops.uniform_pm1(1, n), ops.uniform_pm1(2, n)
    if n > 1000:
        x[500], x[700], f[3] = np.inf, np.nan, -np.inf
    with np.errstate(invalid="ignore"):
        y = dev(ctx, np.zeros(n))
        bc.spmv(ctx, dA, dev(ctx, x), y)
        assert same(y.numpy(), serial(A, x))
        bc.residual(ctx, dA, dev(ctx, x), dev(ctx, f), y)
        assert same(y.numpy(), f - serial(A, x))
        u = dev(ctx, x)
        bc.relax(ctx, dA, dev(ctx, d), dev(ctx, f), u, dev(ctx, np.zeros(n)), 2)
        want = x
        for _ in range(2):
            want = (f - serial(A, want)) / d + want
        assert same(u.numpy(), want)


@pytest.mark.parametrize("grid", [17, 24, 40])
@pytest.mark.parametrize("precision", [bc.PREC_FP64, bc.PREC_FP32])
def test_fused_prolongation(ctx, grid, precision):
    """A single solve folds the prolongation into a sweep on its small levels,
    a solve of several columns does not: same bits."""
    A = ops.lognormal3d(grid, 4.0, seed=1)
    n = len(A[0]) - 1
    B = bc.Boot(ctx, bc.Csr(ctx, A), bc.make_params())
    B.set_precision(precision)
    b = [ops.uniform_pm1(j, n) for j in range(3)]
    xs = [dev(ctx, np.zeros(n)) for _ in b]
    it, _, _ = B.fcg_multi([dev(ctx, v) for v in b], xs)
    for j in range(3):
        x = dev(ctx, np.zeros(n))
        k, _ = B.fcg(dev(ctx, b[j]), x)
        assert k == it[j]
        assert np.array_equal(bits(x.numpy()), bits(xs[j].numpy()))
    B.free()
