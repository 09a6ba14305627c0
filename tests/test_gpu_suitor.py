"""Suitor matching against the oracle where its chains are long or its rows
span several groups of lanes: displacement chains past the per-vertex limit
are listed and followed in a second launch by groups of 8 lanes."""
import numpy as np
import pytest
import scipy.sparse as sp

import bootcmatchg_amd as bc
from bootcmatchg_amd import operators as ops
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = bc.Context(0)
    yield c
    c.close()


def random_graph(n, per_row, seed):
    rng = np.random.default_rng(seed)
    r = np.repeat(np.arange(n), per_row)
    c = rng.integers(0, n, n * per_row)
    S = sp.csr_matrix((np.ones(len(r)), (r, c)), shape=(n, n))
    S = sp.csr_matrix(((S + S.T) > 0).astype(float) + sp.eye(n))
    S.sort_indices()
    return (S.indptr.astype(np.int32), S.indices.astype(np.int32), S.data.astype(np.float64))


def path(n):
    S = sp.csr_matrix(sp.diags([np.ones(n - 1), np.ones(n), np.ones(n - 1)], [-1, 0, 1]))
    S.sort_indices()
    return (S.indptr.astype(np.int32), S.indices.astype(np.int32), S.data.astype(np.float64))


def weights_of(A, kind, seed):
    """ties: every edge alike; few: three values; symmetric and asymmetric
    random; some edges without a positive weight; diagonal slots 0."""
    row, col, _ = A
    n = len(row) - 1
    i = np.repeat(np.arange(n), np.diff(row)).astype(np.int64)
    lo, hi = np.minimum(i, col), np.maximum(i, col)
    key = (lo * 1000003 + hi * 7919 + seed) % 1009
    if kind == "ties":
        W = np.ones(len(col))
    elif kind == "few":
        W = 1.0 + key % 3
    elif kind == "symmetric":
        W = (key - 100) / 1009.0
    else:
        W = np.random.default_rng(seed).uniform(-0.1, 1.0, len(col))
    W[i == col] = 0.0
    return W


GRAPHS = {
    "path_2": lambda: path(2),
    "path_4001": lambda: path(4001),            # one chain of 2000 displacements
    "path_300": lambda: path(300),
    "grid2d_61": lambda: ops.poisson2d(61),
    "grid3d_17": lambda: ops.poisson3d(17),
    "rows_of_4": lambda: random_graph(3000, 2, 1),
    "rows_of_9": lambda: random_graph(3000, 4, 2),    # just over a group of lanes
    "rows_of_40": lambda: random_graph(1500, 20, 3),
}


@pytest.mark.parametrize("kind", ["ties", "few", "symmetric", "asymmetric"])
@pytest.mark.parametrize("name", list(GRAPHS))
def test_matching_equals_the_oracle(ctx, name, kind):
    A = GRAPHS[name]()
    n = len(A[0]) - 1
    W = weights_of(A, kind, 11)
    Mr_o, Ms_o, nu_o = orc.matching(A, W)
    dA = bc.Csr(ctx, A)
    dW = bc.DeviceArray.from_numpy(ctx, W)
    Mr, Ms = bc.DeviceArray(ctx, n, np.int32), bc.DeviceArray(ctx, n, np.int32)
    nu = bc.matching(ctx, dA, dW, Mr, Ms)
    assert np.array_equal(Mr.numpy(), Mr_o)
    assert np.array_equal(Ms.numpy(), Ms_o)
    assert nu == nu_o
    for a in (dA, dW, Mr, Ms):
        a.free()
