"""SOLA iterations in one launch each against the oracle's sweeps, bit for bit: walls and periodic y,
no coefficients and z-invariant ones, an odd number of wall-normal cells, sizes at the edges of a
tile (14 pairs by 13 or 29 rows) and of a march, the smallest grids, wall values and both kinds of
pressure condition, one to four iterations (each parity of the ping-pong); and a step, whose last
iteration writes the boundary conditions, against the same step with separate fills."""
import numpy as np
import pytest

import mobydiff_amd as M
from oracle import oracle as O

pytestmark = pytest.mark.gpu

SHAPES = [(2, 2, 2), (4, 3, 2), (28, 13, 8), (30, 14, 10), (58, 29, 12), (56, 31, 34), (100, 45, 70), (130, 64, 96)]


def _grid(shape, per_y, seed):
    rng = np.random.default_rng(seed)
    g = O.Grid(*shape, lx=1.3, ly=0.9, lz=1.1, re=100.0, forcing=(0.1, 0.0, 0.0), periodic=(1, per_y, 1))
    for s in range(2):
        g.bc_type[O.bci(2, s, 0)] = int(rng.integers(0, 2))
        for q in range(4):
            g.bc_value[O.bci(2, s, q)] = 0.1 * rng.standard_normal()
    plane = [np.where(rng.random(g.gshape[1:]) < 0.2, 1e28, 30.0 * rng.random(g.gshape[1:])) for _ in range(3)]
    coef = tuple(np.ascontiguousarray(np.broadcast_to(a, g.gshape)) for a in plane)
    return g, coef, O.random_fields(g, rng, amp=0.05)


def _channel(g, f, coef, niter, per_y):
    cfg = M.channel_config(g.nx, g.ny, g.nz, g.lx, g.ly, g.lz, g.re, forcing=g.forcing, periodic=(1, per_y, 1),
                           solver=M.SOLVER_SOLA, niter=niter, omega=1.6)
    for q in range(24):
        cfg.bc_type[q], cfg.bc_value[q] = int(g.bc_type[q]), float(g.bc_value[q])
    ch = M.Channel(cfg)
    if coef is not None:
        ch.set_ibm(*coef)
    ch.upload(**f)
    return ch


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("per_y", [0, 1])
def test_iterations_equal_oracle_sweeps(shape, per_y):
    for niter, ibm in ((1, False), (2, True), (3, True), (4, False)):
        print(shape, per_y, niter, ibm, flush=True)
        if per_y and shape[1] % 2:
            continue   # colours need an even periodic extent
        g, coef, f = _grid(shape, per_y, 7 + niter)
        coef = coef if ibm else None
        ch = _channel(g, f, coef, niter, per_y)
        ch.pressure_projection(0.01)
        out = ch.download()
        ch.close()
        O.sola_redblack(g, f, coef, niter, 1.6, 0.01)
        for k in ("un", "vn", "wn", "pn", "us", "vs", "ws"):
            assert np.array_equal(out[k], f[k]), (k, niter)


@pytest.mark.parametrize("shape", SHAPES[1:7])
def test_step_writes_the_boundary_conditions(shape, monkeypatch):
    g, coef, f = _grid(shape, 0, 3)
    outs = []
    for fused in ("1", "0"):
        monkeypatch.setenv("MOBYDIFF_FUSED_BC", fused)
        ch = _channel(g, f, coef, 3, 0)
        for _ in range(2):
            ch.step(1e-4)
        outs.append(ch.download())
        ch.close()
    for k in outs[0]:
        assert np.array_equal(outs[0][k], outs[1][k]), k
