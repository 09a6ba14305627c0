"""The rules that choose a kernel form, seen through the library's queries."""
import numpy as np
import pytest
import scipy.sparse as sp

import bootcmatchg_amd as bc
from bootcmatchg_amd import operators as ops

from common import SETTINGS, bits
from test_gpu_classes import csr, neumann2d, row_ops

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = bc.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("make", [lambda: ops.poisson3d(20), lambda: ops.aniso2d(90, 0.05)])
@pytest.mark.parametrize("prec,k", [(bc.PREC_FP64, 2), (bc.PREC_FP32, 4), (bc.PREC_FP32, 32)])
def test_a_residual_is_formed_once(ctx, make, prec, k):
    """The residual and its restriction share a launch, which forms a residual
    for every entry of R, where R holds a fine row once at most: not with a
    smoothed prolongator."""
    dA = bc.Csr(ctx, make())
    for aggrtype in (0, 1):
        B = bc.Boot(ctx, dA, bc.make_params(**dict(SETTINGS["V_L1_2sweeps"], aggrtype=aggrtype)))
        B.set_precision(prec)
        entries = len(B.level_Pcsr(0, 0)[1])
        assert (entries > dA.n) == (aggrtype == 1)
        assert bool(B.level_multi(0, 0, k) & bc.MULTI_RESTRICT) == (aggrtype == 0)
        B.free()
    dA.free()


def test_query_refuses_what_is_not_there(ctx):
    B = bc.Boot(ctx, bc.Csr(ctx, ops.poisson2d(40)), bc.make_params())
    for k, l, columns in [(1, 0, 4), (-1, 0, 4), (0, 99, 4), (0, 0, 0), (0, 0, 33)]:
        with pytest.raises(bc.BcmgError):
            B.level_multi(k, l, columns)


def test_a_restriction_to_a_column_form_is_lifted(ctx):
    """bcmg_csr_set_columns(4) hides the narrower forms, BCMG_COLUMNS_ANY gives
    them back."""
    dA = bc.Csr(ctx, ops.poisson3d(120))
    assert dA.column_bytes == 0
    dA.set_columns(4)
    assert dA.column_bytes == 4
    dA.set_columns(bc.COLUMNS_ANY)
    assert dA.column_bytes == 0
    dA.free()


def test_the_form_that_the_row_kernels_read(ctx):
    """bcmg_csr_form names the form, restricted and not, also where no narrow
    column copy is kept (below 11.2 M entries bcmg_csr_column_bytes says 4)."""
    for make, form in [(lambda: ops.poisson3d(24), bc.FORM_STENCIL),
                       (lambda: neumann2d(70), bc.FORM_CLASSES),
                       (lambda: ops.lognormal3d(33, 4.0, seed=2), bc.FORM_SYMMETRIC),
                       (lambda: ops.lognormal3d(18, 4.0, seed=1), bc.FORM_COLUMNS)]:
        dA = bc.Csr(ctx, make())
        assert dA.form == form and dA.column_bytes == 4
        dA.set_columns(4)
        assert dA.form == bc.FORM_COLUMNS
        dA.set_columns(bc.COLUMNS_ANY)
        assert dA.form == form
        dA.free()


def test_a_stencil_keeps_no_column_copies(ctx):
    """An upload holds the CSR arrays, a byte a row and a chunk of small blocks;
    the 16-bit columns and the pattern of a constant stencil (57 + 4 MB at
    160^3) come when they are asked for."""
    from test_gpu_serving import device_bytes_in_use

    def rounded(b):                              # the pool's size classes
        step = 1 << (b.bit_length() - 3)
        return (b + step - 1) // step * step

    A = ops.poisson3d(160)
    n, nnz = len(A[0]) - 1, len(A[1])
    c = bc.Context(0)
    c.sync()
    before = device_bytes_in_use()
    dA = bc.Csr(c, A)
    held = device_bytes_in_use() - before
    assert dA.form == bc.FORM_STENCIL
    assert held <= rounded(8 * nnz) + rounded(4 * nnz) + rounded(4 * (n + 1)) + (34 << 20)
    assert dA.column_bytes == 0
    assert device_bytes_in_use() - before <= held
    dA.set_columns(2)
    assert dA.column_bytes == 2 and device_bytes_in_use() - before >= held + 2 * nnz
    dA.free()
    c.close()


@pytest.mark.parametrize("kinds", [1, 63, 64, 65, 255, 256, 257])
def test_tables_of_any_length(ctx, kinds):
    """Row classes as many as the head of the analysis holds (64), as there may
    be (256) and one more: the kernels' bits are those of the columns. (A form
    fills a hundred rows at a time: a block of 256 rows may hold 128 at most.)"""
    n = 26011
    dA = bc.Csr(ctx, csr(sp.diags(1.0 + (np.arange(n) // 100 % kinds) / 1024.0)))
    assert dA.form == (bc.FORM_STENCIL if kinds == 1 else
                       bc.FORM_CLASSES if kinds <= 256 else bc.FORM_COLUMNS)
    rng = np.random.default_rng(8)
    x, f, d = rng.uniform(-1, 1, n), rng.uniform(-1, 1, n), rng.uniform(7, 8, n)
    got = row_ops(ctx, dA, n, x, f, d)
    dA.set_columns(4)
    for g, w in zip(got, row_ops(ctx, dA, n, x, f, d)):
        assert np.array_equal(bits(g), bits(w))
    dA.free()


@pytest.mark.parametrize("count", [1, 2, 8, 9, 16, 17])
def test_offsets_of_any_number(ctx, count):
    """The table of a large operator's distinct column offsets (16 slots): up to
    8 make a pattern, which is read with the bits of the columns."""
    n = 12_000_000 // count + 4099
    off = [0] + [37 * k * k + 11 * k for k in range(1, count)]
    vals = [1.0 + 0.25 * k for k in range(count)]
    S = sp.diags([np.full(n - o, v) for o, v in zip(off, vals)], off, format="csr")
    S.data *= 1.0 + (np.arange(S.nnz) % 1009) / 2048.0   # no classes
    dA = bc.Csr(ctx, (S.indptr.astype(np.int32), S.indices.astype(np.int32), S.data))
    assert dA.form == bc.FORM_COLUMNS and dA.column_bytes == (0 if count <= 8 else 4)
    x = bc.DeviceArray.from_numpy(ctx, ops.uniform_pm1(2, n))
    y = bc.DeviceArray(ctx, n)
    bc.spmv(ctx, dA, x, y)
    got = y.numpy()
    dA.set_columns(4)
    bc.spmv(ctx, dA, x, y)
    assert np.array_equal(bits(got), bits(y.numpy()))
    dA.free()


def eight_of_nine(N):
    """2D 9-point, every row without one corner, even and odd rows without
    another one: rows of 8 entries at 9 offsets."""
    T = sp.diags([np.ones(N - 1), np.ones(N), np.ones(N - 1)], [-1, 0, 1])
    S = sp.csr_matrix(10.0 * sp.eye(N * N) - sp.kron(T, T))
    S.sort_indices()
    r = np.repeat(np.arange(N * N), np.diff(S.indptr))
    drop = (S.indices - r) == np.where(r % 2 == 0, N + 1, -N - 1)
    S.data[drop] = 0.0
    S.eliminate_zeros()
    return csr(S)


@pytest.mark.parametrize("make,bytes_", [(lambda: ops.poisson3d(140), 0),
                                         (lambda: ops.poisson3d(100), 4),
                                         (lambda: eight_of_nine(1500), 2),
                                         (lambda: ops.lognormal3d(120, 4.0, seed=1), 0)])
def test_column_bytes_before_and_after_the_copies(ctx, make, bytes_):
    """bcmg_csr_column_bytes says what the copies will be before they are made,
    and what is not to come is refused."""
    dA = bc.Csr(ctx, make())
    assert dA.form != bc.FORM_COLUMNS and dA.column_bytes == bytes_
    for form in (0, 2):
        if form < bytes_:
            with pytest.raises(bc.BcmgError) as e:
                dA.set_columns(form)
            assert e.value.code == bc.EUNSUP
    if bytes_ < 4:
        dA.set_columns(bytes_)
        assert dA.form == bc.FORM_COLUMNS and dA.column_bytes == bytes_
        x = bc.DeviceArray.from_numpy(ctx, ops.uniform_pm1(2, dA.n))
        y = bc.DeviceArray(ctx, dA.n)
        bc.spmv(ctx, dA, x, y)
        got = y.numpy()
        dA.set_columns(bc.COLUMNS_ANY)
        assert dA.column_bytes == bytes_
        bc.spmv(ctx, dA, x, y)
        assert np.array_equal(bits(got), bits(y.numpy()))
    dA.free()
