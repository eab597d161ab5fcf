"""A step with the FFT projection against the same stages as separate calls: inside a step the
projection takes the predictor's ghosts as filled, adds the flow-rate shift and writes the new
fields' ghosts itself.  Grids of two cells a side, of fewer planes than a thread marches, of
tile remainders, lengths the LDS transforms take, with and without flow rate, body and stretching."""
import numpy as np
import pytest

import mobydiff_amd as M
from oracle import oracle as O

pytestmark = pytest.mark.gpu

A, B, G = ([x / 120.0 for x in s] for s in ((64.0, 50.0, 90.0), (0.0, -34.0, -50.0), (64.0, 16.0, 40.0)))
SHAPES = [(2, 2, 2), (16, 2, 16), (16, 5, 2), (2, 4, 16), (4, 6, 64), (64, 9, 4), (32, 66, 8), (128, 7, 32), (256, 65, 64)]
NAMES = ("un", "vn", "wn", "pn", "us", "vs", "ws", "oru", "orv", "orw")


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("flow,body,beta,prec", [(True, False, 1.5, "fp64"), (False, False, None, "fp64"),
                                                 (True, True, None, "fp64"), (True, False, None, "mixed")])
def test_step_equals_the_calls(shape, flow, body, beta, prec):
    _compare(shape, flow, body, beta, prec)


# the routes that the switches leave: separate fills, sums and shift, other marches, other solves
@pytest.mark.parametrize("env", ["FUSED_BC=0", "FUSED_FLOWRATE=0", "MOMENTUM_DIRECT=1", "MOM_KZ=4", "PART_TRIDIAG=0",
                                 "WAVE_TRIDIAG=0"])
@pytest.mark.parametrize("shape", [(2, 2, 2), (32, 66, 8), (64, 20, 32)])
@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_switches(env, shape, prec, monkeypatch):
    name, value = env.split("=")
    monkeypatch.setenv("MOBYDIFF_" + name, value)
    _compare(shape, True, False, 1.5, prec)


def _compare(shape, flow, body, beta, prec):
    print(shape, flow, body, beta, prec, flush=True)
    rng = np.random.default_rng(5)
    g = O.Grid(*shape, lx=2.0, ly=2.0, lz=1.0, periodic=(1, 0, 1), beta=beta)
    f = O.random_fields(g, rng)
    dt = 1e-3
    mixed = dict(precision=M.PREC_MIXED, tol=1e-9) if prec == "mixed" else {}
    chs = [M.Channel(M.channel_config(*shape, g.lx, g.ly, g.lz, g.re, solver=M.SOLVER_FFT, p_neumann_y=False,
                                      stretch_beta=beta or 0.0, flowrate=flow, flow_height=2.0, **mixed))
           for _ in range(2)]
    coef = [np.abs(rng.standard_normal(chs[0].gshape)) * 10.0 for _ in range(3)] if body else None
    for ch in chs:
        ch.upload(**f)
        if body:
            ch.set_ibm(*coef)
        ch.apply_bc()
    step, calls = chs
    step.step(dt)
    for a, b, c in zip(A, B, G):
        calls.momentum(dt * a, dt * b, dt * c)
        if flow:
            calls.flowrate_shift(dt * c)
        calls.apply_bc()
        calls.pressure_projection(dt * c)
        calls.apply_bc()
    got, want = step.download(NAMES), calls.download(NAMES)
    # three projections, each within 1e-12 of its fields (the FP32 passes end within the tolerance on
    # the divergence instead, 1e-9 over velocities of order 1)
    tol = 1e-8 if prec == "mixed" else 1e-11
    for k in NAMES:
        d = np.linalg.norm(got[k] - want[k]) / max(np.linalg.norm(want[k]), 1e-300)
        assert d < tol, (k, d)
    # the ghosts are the fill's own, bit for bit
    step.apply_bc()
    again = step.download(NAMES)
    for k in NAMES:
        assert np.array_equal(again[k], got[k]), k
    for ch in chs:
        ch.close()
