"""Plans of the LDS-resident sweeps: what the first solve on a handle pays for its plan, and which plan
a handle runs on when it is stepped alone and in batches in turn."""
import time

import numpy as np
import pytest

import mobydiff_amd as M

pytestmark = pytest.mark.gpu


def _first_and_later(shape):
    """ms of the first projection of a new handle and of the fastest of the next three, of which a
    solve is one residual (the tolerance holds at once)."""
    ch = M.Channel(M.channel_config(*shape, 4.0, 2.0, 2.0, 2000.0, solver=M.SOLVER_SOR, omega=1.8, tol=1e30, check_every=20))
    ch.synchronize()
    ms = []
    for _ in range(4):
        t = time.perf_counter()
        ch.pressure_projection(1e-3)
        ch.synchronize()
        ms.append((time.perf_counter() - t) * 1e3)
    ch.close()
    return ms[0], min(ms[1:])


def test_first_solve_is_not_slowed_by_the_search():
    """The search over decompositions of a grid that has none (512 x 256 x 256) went through millions
    of cuts, 5.6 ms in the first solve; a search bounded by the workgroups a device can hold, and the
    device's attributes, take well under a millisecond.  Bound: 2 ms, the better of two handles."""
    _first_and_later((32, 24, 16))   # code and buffers of the process
    extra = min(a - b for a, b in (_first_and_later((512, 256, 256)) for _ in range(2)))
    print("first solve: +%.2f ms" % extra, flush=True)
    assert extra < 2.0
