"""The context's device memory comes in chunks and goes back: a closed context
leaves nothing behind, and what a context holds stays near what its blocks
take.
"""
import time

import pytest

import bootcmatchg_amd as bc
from bootcmatchg_amd import operators as ops

from test_gpu_serving import device_bytes_in_use

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("make", [lambda: ops.poisson2d(9), lambda: ops.poisson3d(40),
                                  lambda: ops.lognormal3d(61, 4.0, seed=1)])
def test_closed_context_gives_its_memory_back(make):
    A = make()

    def run():
        ctx = bc.Context(0)
        B = bc.Boot(ctx, bc.Csr(ctx, A), bc.make_params())
        ctx.sync()
        held = device_bytes_in_use()
        B.free()
        ctx.close()
        return held

    run()                                   # the library's and runtime's own memory
    before = device_bytes_in_use()
    for _ in range(3):
        held = run()
        # the operator and its hierarchy (about 3 times its 12 bytes an entry),
        # set-up temporaries, chunks at most as large again: 8 MiB at least
        assert held - before <= (16 << 20) + 40 * 12 * len(A[1])
        # the runtime may hand freed memory back a few milliseconds later
        end = time.monotonic() + 1.0
        while device_bytes_in_use() - before > 4 << 20 and time.monotonic() < end:
            time.sleep(0.005)
        assert device_bytes_in_use() - before <= 4 << 20
