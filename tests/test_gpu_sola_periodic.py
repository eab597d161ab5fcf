"""SOLA iterations in one launch each with a periodic y, at even sizes around the edges of a tile's rows
(13 or 29 own ones) and of several tiles, against the oracle's sweeps, bit for bit."""
import numpy as np
import pytest

import mobydiff_amd as M
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx", [28, 58])
@pytest.mark.parametrize("ny", [2, 4, 12, 14, 26, 28, 30, 40, 58, 60])
def test_periodic_y_at_the_edges_of_a_tile(nx, ny):
    nz = 10
    for niter, ibm in ((1, True), (2, False), (3, True)):
        print(nx, ny, niter, ibm, flush=True)
        rng = np.random.default_rng(ny + niter)
        g = O.Grid(nx, ny, nz, lx=1.3, ly=0.9, lz=1.1, re=100.0, periodic=(1, 1, 1))
        plane = [np.where(rng.random(g.gshape[1:]) < 0.2, 1e28, 30.0 * rng.random(g.gshape[1:])) for _ in range(3)]
        coef = tuple(np.ascontiguousarray(np.broadcast_to(a, g.gshape)) for a in plane) if ibm else None
        f = O.random_fields(g, rng, amp=0.05)
        cfg = M.channel_config(nx, ny, nz, g.lx, g.ly, g.lz, g.re, periodic=(1, 1, 1), solver=M.SOLVER_SOLA, niter=niter,
                               omega=1.6)
        for q in range(24):
            cfg.bc_type[q], cfg.bc_value[q] = int(g.bc_type[q]), float(g.bc_value[q])
        ch = M.Channel(cfg)
        if coef is not None:
            ch.set_ibm(*coef)
        ch.upload(**f)
        ch.pressure_projection(0.01)
        out = ch.download()
        ch.close()
        O.sola_redblack(g, f, coef, niter, 1.6, 0.01)
        for k in ("un", "vn", "wn", "pn", "us", "vs", "ws"):
            assert np.array_equal(out[k], f[k]), (k, niter)
