"""The serving loop while the precision of a served composite changes: a lane
follows it, between requests and while requests run."""
import numpy as np
import pytest

import bootcmatchg_amd as bc
from bootcmatchg_amd import operators as ops

from common import SETTINGS, bits

pytestmark = pytest.mark.gpu

F64, F32, B16 = bc.PREC_FP64, bc.PREC_FP32, bc.PREC_BF16


@pytest.fixture(scope="module")
def ctx():
    c = bc.Context(0)
    yield c
    c.close()


def finish(S, rids):
    out = {}
    for _ in range(3000):
        S.step()
        for r in rids:
            if r not in out:
                got = S.result(r)
                if got is not None:
                    out[r] = got
        if len(out) == len(rids):
            return [out[r] for r in rids]
    raise AssertionError("requests still pending")


@pytest.mark.parametrize("make", [lambda: ops.aniso2d(80, 0.05), lambda: ops.lognormal3d(18, 4.0, seed=3)])
@pytest.mark.parametrize("precs", [(F64, F32, F64), (F32, F64), (B16, F64, F32, F64, B16)])
def test_between_requests(ctx, make, precs):
    """Each phase's requests have the bits of single solves in its precision."""
    A = make()
    n = len(A[0]) - 1
    B = bc.Boot(ctx, bc.Csr(ctx, A), bc.make_params(**SETTINGS["V_L1_2sweeps"]))
    B.set_precision(precs[0])
    S = bc.Server(ctx, 1 << 30, 8)
    op = S.add(B)
    dx = bc.DeviceArray(ctx, n)
    for phase, prec in enumerate(precs):
        B.set_precision(prec)
        bs = [bc.DeviceArray.from_numpy(ctx, ops.uniform_pm1(10 * phase + j, n)) for j in range(5)]
        xs = [bc.DeviceArray(ctx, n) for _ in bs]
        got = finish(S, [S.submit(op, b, x) for b, x in zip(bs, xs)])
        for b, x, r in zip(bs, xs, got):
            it, res = B.fcg(b, dx)
            assert (r["status"], r["iterations"], r["residual"]) == (bc.OK, it, res), (phase, prec)
            assert np.array_equal(bits(x.numpy()), bits(dx.numpy())), (phase, prec)
    S.close()
    B.free()


@pytest.mark.parametrize("first,second", [(F64, F32), (F32, F64), (F32, B16), (F64, B16)])
def test_while_requests_run(ctx, first, second):
    """The precision changes after three iterations: the requests end converged
    (the true residual within the tolerance), in a few iterations more at most
    than in the lower of the two precisions."""
    A = ops.aniso2d(80, 0.05)
    n = len(A[0]) - 1
    B = bc.Boot(ctx, bc.Csr(ctx, A), bc.make_params(**SETTINGS["V_L1_2sweeps"]))
    bh = [ops.uniform_pm1(j, n) for j in range(5)]
    bs = [bc.DeviceArray.from_numpy(ctx, b) for b in bh]
    dx = bc.DeviceArray(ctx, n)
    most = 0
    for prec in (first, second):
        B.set_precision(prec)
        most = max([most] + [B.fcg(b, dx)[0] for b in bs])
    B.set_precision(first)
    S = bc.Server(ctx, 1 << 30, 8)
    op = S.add(B)
    xs = [bc.DeviceArray(ctx, n) for _ in bs]
    rids = [S.submit(op, b, x) for b, x in zip(bs, xs)]
    for _ in range(4):
        assert S.step() == 0
    B.set_precision(second)
    M = ops.to_scipy(A)
    for r, b, x in zip(finish(S, rids), bh, xs):
        assert r["status"] == bc.OK and 3 <= r["iterations"] <= 2 * most
        # FP64's test is on the recursive residual: a margin for its drift
        assert np.linalg.norm(b - M @ x.numpy()) <= 1.01e-8 * np.linalg.norm(b)
    S.close()
    B.free()
