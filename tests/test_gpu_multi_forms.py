"""Two steps of a five-point stencil a pass and several sweeps a launch, on
operators that take these forms: bcmg_level_multi says so, and solves of several
columns equal single solves bit for bit."""
import numpy as np
import pytest
import scipy.sparse as sp

import bootcmatchg_amd as bc
from bootcmatchg_amd import operators as ops

from common import SETTINGS, bits
from test_gpu_classes import csr

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = bc.Context(0)
    yield c
    c.close()


def five(N, n, across=False):
    """-1 at offsets -N, -1, 1, N and 4.125 on the diagonal, n rows that need
    not fill the last line of N; across: a line's end is coupled with the next
    line's begin."""
    i = np.arange(1, n)
    one = np.where((i % N == 0) & (not across), 0.0, -1.0)
    S = sp.diags([np.full(n - N, -1.0), one, np.full(n, 4.125), one, np.full(n - N, -1.0)],
                 [-N, -1, 0, 1, N], format="csr")
    S.eliminate_zeros()
    return csr(S)


def box(a, b, c):
    """7-point operator on a x b x c points, the longest side last: a narrow
    band."""
    def t(m):
        return sp.diags([np.full(m - 1, -1.0), np.full(m, 2.0), np.full(m - 1, -1.0)], [-1, 0, 1])
    ia, ib, ic = sp.eye(a), sp.eye(b), sp.eye(c)
    S = sp.csr_matrix(sp.kron(sp.kron(ic, ib), t(a)) + sp.kron(sp.kron(ic, t(b)), ia) +
                      sp.kron(sp.kron(t(c), ib), ia))
    S.eliminate_zeros()
    return csr(S)


# a block's vector of 32 MB or more for the pairs: rows x columns x bytes
PAIRS = [
    (lambda: ops.aniso2d(512, 0.01), 32, 16),        # 32 MB exactly, in FP32 and FP64
    (lambda: ops.poisson2d(603), 32, 18),            # several tiles and strips, ragged
    (lambda: five(700, 700 * 400 + 123), 32, 17),    # the last line not filled
    (lambda: five(129, 129 * 2200 + 128), 31, 16),   # just wide enough, one row short
    (lambda: five(700, 700 * 401 + 1, True), 32, 16),  # lines coupled, one row in the last
    (lambda: five(131072, 262144 + 9), 32, 16),      # three positions along the walk
]
SLABS = [
    (lambda: box(4, 4, 200), 32, 16),                # seven entries, 3200 rows
    (lambda: box(4, 4, 2003), 9, 6),                 # many workgroups, ragged
    (lambda: five(40, 40 * 130 + 3), 32, 16),        # more halo than rows
    (lambda: five(20, 20 * 205 + 7), 13, 5),         # a group of columns not filled
]


def check(ctx, A, k, prec, pre, post, form):
    n = len(A[0]) - 1
    dA = bc.Csr(ctx, A)
    assert dA.form == bc.FORM_STENCIL
    B = bc.Boot(ctx, dA, bc.make_params(**dict(SETTINGS["V_L1_2sweeps"], itnlim=4,
                                               prerelax_sweeps=pre, postrelax_sweeps=post)))
    B.set_precision(prec)
    assert B.level_multi(0, 0, k) & (bc.MULTI_PAIRS | bc.MULTI_SLAB) == form
    bs = [bc.DeviceArray.from_numpy(ctx, ops.uniform_pm1(j, n)) for j in range(k)]
    xs = [bc.DeviceArray(ctx, n) for _ in range(k)]
    its, res, _ = B.fcg_multi(bs, xs)
    dx = bc.DeviceArray(ctx, n)
    for j in range(0, k, max(1, k // 3)):
        it, r = B.fcg(bs[j], dx)
        assert its[j] == it and res[j] == r
        assert np.array_equal(bits(xs[j].numpy()), bits(dx.numpy())), j
    B.free()
    dA.free()


@pytest.mark.parametrize("pre,post", [(2, 1), (2, 2), (4, 4), (3, 5)])
@pytest.mark.parametrize("prec", [bc.PREC_FP32, bc.PREC_FP64])
@pytest.mark.parametrize("make,k32,k64", PAIRS)
def test_pairs(ctx, make, k32, k64, prec, pre, post):
    check(ctx, make(), k32 if prec == bc.PREC_FP32 else k64, prec, pre, post, bc.MULTI_PAIRS)


@pytest.mark.parametrize("pre,post", [(3, 3), (4, 4), (5, 2)])
@pytest.mark.parametrize("prec", [bc.PREC_FP32, bc.PREC_FP64])
@pytest.mark.parametrize("make,k32,k64", SLABS)
def test_slabs(ctx, make, k32, k64, prec, pre, post):
    check(ctx, make(), k32 if prec == bc.PREC_FP32 else k64, prec, pre, post, bc.MULTI_SLAB)


@pytest.mark.parametrize("prec", [bc.PREC_FP32, bc.PREC_FP64])
def test_neither_below_its_size(ctx, prec):
    """One column less than 32 MB a vector, and a single sweep."""
    A = ops.aniso2d(512, 0.01)
    k = 31 if prec == bc.PREC_FP32 else 15
    check(ctx, A, k, prec, 4, 4, 0)
    check(ctx, A, k + 1, prec, 1, 1, 0)
