"""Several sweeps in one launch (operators of narrow band): a single solve,
whose levels use the slab launches where they pay, has the bits of the same
right-hand side through the multi-column path, which launches every sweep.

The operators are strips and lines, so that workgroups own few rows, many
rows, or all; constant coefficients (a stencil per level) and varying ones
(rows in registers); the sweep counts split evenly, unevenly and not at all."""
import numpy as np
import pytest
import scipy.sparse as sp

import bootcmatchg_amd as bc
from bootcmatchg_amd import operators as ops
from oracle import oracle as orc

from common import SETTINGS, bits, check_fcg_vs_oracle

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


def strip(nx, ny, seed=None):
    """5-point Laplacian on nx x ny (band nx); with a seed the faces get
    coefficients in [1, 2)."""
    n = nx * ny
    i = np.arange(n)
    rng = np.random.default_rng(seed)
    ex = np.where(i % nx < nx - 1, 1.0 if seed is None else rng.uniform(1, 2, n), 0.0)[:-1]
    ey = np.full(n - nx, 1.0) if seed is None else rng.uniform(1, 2, n - nx)
    S = sp.diags([-ey, -ex, -ex, -ey], [-nx, -1, 1, nx], shape=(n, n))
    S = sp.csr_matrix(S)
    S.eliminate_zeros()
    d = 4.0 * np.ones(n) if seed is None else 0.05 - np.asarray(S.sum(axis=1)).ravel()
    return csr(S + sp.diags(d))


def line(n):
    return csr(sp.diags([np.full(n - 1, -1.0), np.full(n, 2.01), np.full(n - 1, -1.0)],
                        [-1, 0, 1]))


OPERATORS = {
    "line_1500": lambda: line(1500),
    "line_70001": lambda: line(70001),
    "strip_16x300": lambda: strip(16, 300),
    "strip_100x129": lambda: strip(100, 129),      # a few workgroups of many rows
    "strip_33x8001": lambda: strip(33, 8001),      # more workgroups than CUs can take at once
    "varying_16x300": lambda: strip(16, 300, 1),
    "varying_60x400": lambda: strip(60, 400, 2),
    "poisson3d_24": lambda: ops.poisson3d(24),
    "aniso2d_127": lambda: ops.aniso2d(127, 0.01),
}


@pytest.mark.parametrize("sweeps", [(1, 1, 1), (4, 4, 16), (3, 5, 7), (0, 2, 13)])
@pytest.mark.parametrize("name", list(OPERATORS))
def test_single_equals_multi(ctx, name, sweeps):
    A = OPERATORS[name]()
    n = len(A[0]) - 1
    b = ops.uniform_pm1(5, n)
    dA = bc.Csr(ctx, A)
    db = bc.DeviceArray.from_numpy(ctx, b)
    dx, dy = bc.DeviceArray(ctx, n), bc.DeviceArray(ctx, n)
    for setting, prec in (("V_L1_2sweeps", bc.PREC_FP64), ("W_L1_3sweeps", bc.PREC_FP32),
                          ("H_jacobi_1sweep", bc.PREC_BF16)):
        s = dict(SETTINGS[setting], prerelax_sweeps=sweeps[0], postrelax_sweeps=sweeps[1],
                 relaxnumber_coarse=sweeps[2], itnlim=40)
        B = bc.Boot(ctx, dA, bc.make_params(**s))
        B.set_precision(prec)
        it, res = B.fcg(db, dx)
        its, ress, st = B.fcg_multi([db], [dy])
        assert st[0] == bc.OK and its[0] == it and ress[0] == res, (setting, it, its[0])
        assert np.array_equal(bits(dx.numpy()), bits(dy.numpy())), setting
        B.free()
    for a in (dA, db, dx, dy):
        a.free()


@pytest.mark.parametrize("name", ["strip_16x300", "varying_16x300", "line_1500"])
def test_solution_against_the_oracle(ctx, name):
    A = OPERATORS[name]()
    n = len(A[0]) - 1
    b = ops.uniform_pm1(6, n)
    s = dict(SETTINGS["V_L1_2sweeps"])
    dA = bc.Csr(ctx, A)
    B = bc.Boot(ctx, dA, bc.make_params(**s))
    dx = bc.DeviceArray(ctx, n)
    it, _ = B.fcg(bc.DeviceArray.from_numpy(ctx, b), dx)
    O = orc.Boot(A, orc.params(**s))
    rc, xo, ro, _ = O.fcg(b)
    assert rc == 0
    check_fcg_vs_oracle(dx.numpy(), it, xo, ro.iterations, A, b, s["rtol"], name)
    B.free()
    dA.free()
