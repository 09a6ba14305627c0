"""Two steps of a five-point stencil in one pass over an interleaved block, and
several sweeps of a small narrow-band one in one launch:
solves of several columns equal single solves bit for bit, at the edges of the
tiles, strips and column groups, for sweep counts that pair and that do not.
"""
import numpy as np
import pytest

import bootcmatchg_amd as bc
from bootcmatchg_amd import operators as ops

from common import SETTINGS, bits
from test_gpu_classes import neumann2d

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = bc.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("make,k", [
    (lambda: ops.aniso2d(128, 0.01), 4),      # one step a launch, or slabs
    (lambda: ops.poisson2d(257), 32),
    (lambda: ops.aniso2d(512, 0.01), 31),     # just in pairs in FP64 and FP32
    (lambda: ops.poisson2d(603), 32),         # several tiles and strips, ragged
    (lambda: ops.aniso2d(1025, 0.01), 9),     # a partly filled group of columns
    (lambda: neumann2d(725), 18),             # an L1 divisor that varies at the edges
    (lambda: ops.poisson2d(33), 32),          # level 0 in slabs
    (lambda: ops.aniso2d(64, 0.01), 9),
    (lambda: ops.poisson3d(12), 32),          # seven entries
])
@pytest.mark.parametrize("prec", [bc.PREC_FP64, bc.PREC_FP32])
@pytest.mark.parametrize("pre,post", [(1, 1), (2, 2), (4, 4), (3, 5)])
def test_columns_equal_single_solves(ctx, make, k, prec, pre, post):
    A = make()
    n = len(A[0]) - 1
    prm = dict(SETTINGS["V_L1_2sweeps"], itnlim=6, prerelax_sweeps=pre, postrelax_sweeps=post)
    dA = bc.Csr(ctx, A)
    B = bc.Boot(ctx, dA, bc.make_params(**prm))
    B.set_precision(prec)
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
