"""Row classes (operators whose rows take few distinct forms, read as one byte
per row) and symmetric stencils (half of the values, by diagonals): every row
kernel gives the bits of the int32-column kernels, at the edges of the
kernels' blocks and of the rules that choose them.

bcmg_csr_set_columns(4) restricts a handle to its int32 columns; the default
uses the classes where they are kept (no more than 256 forms of at most 8
entries), else the symmetric stencil (at most 7 offsets, from 32 768 rows)."""
import ctypes

import numpy as np
import pytest
import scipy.sparse as sp

import bootcmatchg_amd as bc
from bootcmatchg_amd import operators as ops
from oracle import oracle as orc

from common import SETTINGS, bits

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = bc.Context(0)
    yield c
    c.close()


def csr(S):
    S = sp.csr_matrix(S)
    S.sort_indices()
    return (S.indptr.astype(np.int32), S.indices.astype(np.int32), S.data.astype(np.float64))


def tridiagonal(n):
    return csr(sp.diags([np.full(n - 1, -1.0), np.full(n, 2.5), np.full(n - 1, -0.75)],
                        [-1, 0, 1]))


def neumann2d(N):
    """Diagonal = number of neighbours + 1/8: the forms differ in a value, so
    they are classes but no constant stencil."""
    A = ops.poisson2d(N)
    S = ops.to_scipy(A)
    S.setdiag(0.125 + np.diff(A[0]) - 1.0)
    return csr(S)


def diagonals(n, kinds):
    """`kinds` distinct values on the diagonal."""
    return csr(sp.diags(1.0 + (np.arange(n) * 7919 % kinds) / 1024.0))


def eight_entries(N):
    """2D 9-point without one corner: 8 entries in an inner row."""
    T = sp.diags([np.ones(N - 1), np.ones(N), np.ones(N - 1)], [-1, 0, 1])
    U = sp.diags([np.ones(N - 1)], [1])
    return csr(10.0 * sp.eye(N * N) - sp.kron(T, T) + sp.kron(U, U))


def varying2d(N, asymmetric=False):
    """5-point operator with varying symmetric coefficients; asymmetric
    changes one lower entry by an ulp."""
    n = N * N
    rng = np.random.default_rng(N)
    ex, ey = rng.uniform(1, 2, n - 1), rng.uniform(1, 2, n - N)
    ex[np.arange(1, n) % N == 0] = 0.0
    S = sp.csr_matrix(sp.diags([-ey, -ex, -ex, -ey], [-N, -1, 1, N], shape=(n, n)))
    S.eliminate_zeros()
    S = S + sp.diags(0.1 - np.asarray(S.sum(axis=1)).ravel())
    row, col, val = csr(S)
    if asymmetric:
        val[row[n // 2]] = np.nextafter(val[row[n // 2]], 0.0)
    return row, col, val


OPERATORS = {
    "lognormal3d_33": lambda: ops.lognormal3d(33, 4.0, seed=2),   # a symmetric stencil
    "lognormal3d_53": lambda: ops.lognormal3d(53, 4.0, seed=2),   # two rows a thread, ragged
    "varying2d_181": lambda: varying2d(181),                      # just analysed
    "varying2d_401": lambda: varying2d(401),
    "varying2d_401_asymmetric": lambda: varying2d(401, True),
    "poisson3d_17": lambda: ops.poisson3d(17),        # few blocks, all near an end
    "aniso2d_65": lambda: ops.aniso2d(65, 0.01),      # 4225 rows
    "poisson3d_41": lambda: ops.poisson3d(41),        # one row a thread, ragged
    "tridiagonal_4097": lambda: tridiagonal(4097),
    "tridiagonal_524289": lambda: tridiagonal((1 << 19) + 1),  # two rows a thread, one over
    "aniso2d_725": lambda: ops.aniso2d(725, 0.05),
    "poisson3d_81": lambda: ops.poisson3d(81),
    "neumann2d_70": lambda: neumann2d(70),
    "neumann2d_731": lambda: neumann2d(731),
    "diagonals_200": lambda: diagonals(20011, 200),
    "diagonals_257": lambda: diagonals(20011, 257),   # one form too many
    "eight_entries_91": lambda: eight_entries(91),
    "lognormal3d_18": lambda: ops.lognormal3d(18, 4.0, seed=1),  # neither form
}


class At:
    """A device array from its element `o` on."""

    def __init__(self, d, o):
        self.ptr = ctypes.c_void_p(d.ptr.value + 8 * o)


def row_ops(ctx, dA, n, x, f, d, o=0):
    pad = np.zeros(o)
    dx, df, dd = (bc.DeviceArray.from_numpy(ctx, np.concatenate([pad, a])) for a in (x, f, d))
    y, u2 = bc.DeviceArray(ctx, n + o), bc.DeviceArray(ctx, n + o)
    out = []
    bc.spmv(ctx, dA, At(dx, o), At(y, o))
    out.append(y.numpy()[o:])
    bc.residual(ctx, dA, At(dx, o), At(df, o), At(y, o))
    out.append(y.numpy()[o:])
    bc.relax(ctx, dA, At(dd, o), At(df, o), At(dx, o), At(u2, o), 3)
    out.append(dx.numpy()[o:])
    return out


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("name", list(OPERATORS))
def test_row_kernels_same_bits(ctx, name, offset):
    """Products, residuals and sweeps on vectors that start on and off a
    16-byte boundary."""
    A = OPERATORS[name]()
    n = len(A[0]) - 1
    rng = np.random.default_rng(5)
    x, f, d = rng.uniform(-1, 1, n), rng.uniform(-1, 1, n), rng.uniform(7, 8, n)
    dA = bc.Csr(ctx, A)
    got = row_ops(ctx, dA, n, x, f, d, offset)
    dA.set_columns(4)
    want = row_ops(ctx, dA, n, x, f, d, offset)
    for g, w in zip(got, want):
        assert np.array_equal(bits(g), bits(w)), name
    absmv = ops.to_scipy((A[0], A[1], np.abs(A[2]))) @ np.abs(x)
    assert np.all(np.abs(got[0] - orc.spmv(A, x)) <= 1e-13 * absmv + 1e-300)
    dA.free()


@pytest.mark.parametrize("name", ["poisson3d_41", "aniso2d_725", "neumann2d_70",
                                  "lognormal3d_53", "varying2d_181"])
def test_special_values_stay_where_the_rows_read_them(ctx, name):
    """Infinities and NaN in x reach exactly the rows that have an entry
    there; a row without the entry is not touched."""
    A = OPERATORS[name]()
    n = len(A[0]) - 1
    rng = np.random.default_rng(6)
    x, f, d = rng.uniform(-1, 1, n), rng.uniform(-1, 1, n), rng.uniform(7, 8, n)
    N = int(name.split("_")[1])
    x[[0, N - 1, N, 5 * N, n - N, n - 1]] = [np.inf, np.nan, -np.inf, np.nan, np.inf, -np.inf]
    dA = bc.Csr(ctx, A)
    got = row_ops(ctx, dA, n, x, f, d)
    dA.set_columns(4)
    want = row_ops(ctx, dA, n, x, f, d)
    for g, w in zip(got, want):
        assert np.array_equal(np.isnan(g), np.isnan(w))
        m = ~np.isnan(w)
        assert np.array_equal(bits(g[m]), bits(w[m]))
    dA.free()


@pytest.mark.parametrize("prec", [bc.PREC_FP64, bc.PREC_FP32, bc.PREC_BF16])
@pytest.mark.parametrize("setting", ["V_L1_2sweeps", "H_jacobi_1sweep"])
@pytest.mark.parametrize("name", ["poisson3d_41", "neumann2d_70", "aniso2d_725",
                                  "lognormal3d_33", "varying2d_401"])
def test_solves_same_bits(ctx, name, setting, prec):
    """Setup and FCG with level 0 read as classes and as int32 columns (the
    L1 and the diagonal divisor come from the forms in one, from their arrays
    in the other)."""
    A = OPERATORS[name]()
    n = len(A[0]) - 1
    db = bc.DeviceArray.from_numpy(ctx, ops.uniform_pm1(3, n))
    dA = bc.Csr(ctx, A)
    out = []
    for _ in range(2):
        B = bc.Boot(ctx, dA, bc.make_params(**dict(SETTINGS[setting], rtol=1e-6)))
        B.set_precision(prec)
        dx = bc.DeviceArray(ctx, n)
        it, res = B.fcg(db, dx)
        out.append((it, res, dx.numpy()))
        B.free()
        dA.set_columns(4)
    assert out[0][0] == out[1][0] and out[0][1] == out[1][1]
    assert np.array_equal(bits(out[0][2]), bits(out[1][2]))
    dA.free()


@pytest.mark.parametrize("prec", [bc.PREC_FP64, bc.PREC_FP32])
@pytest.mark.parametrize("name,k", [("poisson3d_41", 2), ("aniso2d_65", 5), ("poisson3d_17", 32),
                                    ("eight_entries_91", 11), ("neumann2d_70", 4)])
def test_columns_equal_single_solves(ctx, name, k, prec):
    """Several right-hand sides: whole and partly filled vectors of columns
    a lane, on constant stencils of 5, 7 and 8 entries and on classes."""
    A = OPERATORS[name]()
    n = len(A[0]) - 1
    dA = bc.Csr(ctx, A)
    B = bc.Boot(ctx, dA, bc.make_params(**dict(SETTINGS["V_L1_2sweeps"], itnlim=25)))
    B.set_precision(prec)
    bs = [bc.DeviceArray.from_numpy(ctx, ops.uniform_pm1(j, n)) for j in range(k)]
    xs = [bc.DeviceArray(ctx, n) for _ in range(k)]
    its, res, st = B.fcg_multi(bs, xs)
    dx = bc.DeviceArray(ctx, n)
    for j in range(k):
        it, r = B.fcg(bs[j], dx)
        assert st[j] == bc.OK and its[j] == it and res[j] == r
        assert np.array_equal(bits(xs[j].numpy()), bits(dx.numpy())), j
    B.free()
    dA.free()
