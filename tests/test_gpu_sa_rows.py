"""Smoothed hierarchies with long rows: the set-up kernels that take a row by a
wavefront (scaling, row sums, diagonal, product counts, transpose by ranks and
by bits) give the oracle's bits.
"""
import pytest

import bootcmatchg_amd as bc
from bootcmatchg_amd import operators as ops
from oracle import oracle as orc

from common import SETTINGS
from test_gpu_sa import SA, compare_sa_hierarchy

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,make", [
    ("poisson3d_21", lambda: ops.poisson3d(21)),
    ("poisson3d_33", lambda: ops.poisson3d(33)),        # transposed rows of 370 entries
    ("lognormal3d_26", lambda: ops.lognormal3d(26, 4.0, seed=3)),
])
def test_long_rows(name, make):
    A = make()
    prm = dict(SETTINGS["V_L1_2sweeps"], **SA)
    O = orc.Boot(A, orc.params(**prm))
    assert O.rc == 0
    ctx = bc.Context(0)
    B = bc.Boot(ctx, bc.Csr(ctx, A), bc.make_params(**prm))
    compare_sa_hierarchy(B, O, 0)
    B.free()
    ctx.close()
