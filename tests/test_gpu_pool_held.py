"""What a context holds after a set-up: chunks of the device memory serve blocks
of any size, so the temporaries of all levels take the same bytes."""
import pytest

import bootcmatchg_amd as bc
from bootcmatchg_amd import operators as ops

from test_gpu_serving import device_bytes_in_use

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("make", [lambda: ops.poisson3d(40),
                                  lambda: ops.lognormal3d(61, 4.0, seed=1)])
def test_held_memory_follows_the_hierarchy(make):
    """Three times the hierarchy's 12 bytes an entry (R, the vectors of a cycle
    and the temporaries of the finest set-up step beside it) and two smallest
    chunks; every block here is cut from a chunk (at most 16 MiB)."""
    A = make()

    def run():
        ctx = bc.Context(0)
        before = device_bytes_in_use()
        dA = bc.Csr(ctx, A)
        B = bc.Boot(ctx, dA, bc.make_params())
        ctx.sync()
        held = device_bytes_in_use() - before
        entries = sum(B.level_size(0, l)[1] for l in range(B.levels(0)))
        B.free()
        dA.free()
        ctx.close()
        return held, entries

    run()                                   # the library's and runtime's own memory
    held, entries = run()
    print("held %.1f MiB, hierarchy %.1f MiB" % (held / 2**20, 12 * entries / 2**20))
    assert held <= 3 * 12 * entries + (16 << 20)
