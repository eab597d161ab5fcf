"""FFT steps with the fills inside the projection's kernels and with separate ones (MOBYDIFF_FUSED_BC=0):
the same bits without a flow rate, and with one over a body, whose shift has its own launch either way.
(With a flow rate and no body the right-hand side is formed before the shift or after it, which rounds
differently.)"""
import numpy as np
import pytest

import mobydiff_amd as M
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(2, 3, 2), (32, 66, 8), (64, 20, 32), (128, 33, 16), (256, 65, 64)])
@pytest.mark.parametrize("flow,body,beta", [(False, False, 1.5), (False, True, None), (True, True, None)])
@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_fused_fills_keep_the_bits(shape, flow, body, beta, prec, monkeypatch):
    print(shape, flow, body, beta, prec, flush=True)
    outs = []
    for fused in ("1", "0"):
        monkeypatch.setenv("MOBYDIFF_FUSED_BC", fused)
        rng = np.random.default_rng(6)
        g = O.Grid(*shape, lx=2.0, ly=2.0, lz=1.0, periodic=(1, 0, 1), beta=beta)
        f = O.random_fields(g, rng)
        mixed = dict(precision=M.PREC_MIXED, tol=1e-9) if prec == "mixed" else {}
        ch = M.Channel(M.channel_config(*shape, g.lx, g.ly, g.lz, g.re, solver=M.SOLVER_FFT, p_neumann_y=False,
                                        stretch_beta=beta or 0.0, flowrate=flow, flow_height=2.0, **mixed))
        ch.upload(**f)
        if body:
            ch.set_ibm(*[np.abs(rng.standard_normal(ch.gshape)) * 10.0 for _ in range(3)])
        ch.apply_bc()
        for _ in range(2):
            ch.step(1e-3)
        outs.append(ch.download())
        ch.close()
    for k in outs[0]:
        assert np.array_equal(outs[0][k], outs[1][k]), k
