"""Momentum on grids of few tiles (marches of one, two and four planes, the per-cell kernel) and past the
last-level cache gives the bits of the oracle and of the long march, with and without body and stretching, remainders in every
direction."""
import numpy as np
import pytest

import mobydiff_amd as M
from oracle import oracle as O

pytestmark = pytest.mark.gpu

# per cell; one plane (tile remainders; exactly 256 workgroups); two; four; the default march, past the cache
SHAPES = [(2, 2, 2), (32, 24, 16), (66, 35, 31), (64, 64, 16), (100, 70, 54), (128, 97, 64), (130, 129, 70), (190, 130, 126)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("body,beta", [(False, None), (True, 1.5)])
def test_marches_match(shape, body, beta, monkeypatch):
    print(shape, body, beta, flush=True)
    shape = tuple(n + n % 2 if d != 1 else n for d, n in enumerate(shape))   # x and z even
    rng = np.random.default_rng(9)
    g = O.Grid(*shape, lx=2.0, ly=2.0, lz=1.0, re=300.0, forcing=(1.0, 0.2, -0.1), periodic=(1, 0, 1), beta=beta)
    f = O.random_fields(g, rng)
    got = []
    for env in ({}, {"MOBYDIFF_MOM_KZ": "16"}, {"MOBYDIFF_MOMENTUM_DIRECT": "1"}):
        for k in ("MOBYDIFF_MOM_KZ", "MOBYDIFF_MOMENTUM_DIRECT"):
            monkeypatch.delenv(k, raising=False)
        for k, v in env.items():
            monkeypatch.setenv(k, v)
        ch = M.Channel(M.channel_config(*shape, g.lx, g.ly, g.lz, g.re, solver=M.SOLVER_SOLA, niter=1, omega=1.5,
                                        forcing=g.forcing, stretch_beta=beta or 0.0))
        ch.upload(**f)
        if body:
            c = np.abs(np.random.default_rng(4).standard_normal(ch.gshape)) * 10.0
            ch.set_ibm(c, c + 1.0, c + 2.0)
        ch.momentum(1e-3, -4e-4, 6e-4)
        got.append(ch.download(("us", "vs", "ws", "oru", "orv", "orw")))
        ch.close()
    coef = None
    if body:
        coef = (c, c + 1.0, c + 2.0)
    for other in got[1:]:
        for k in got[0]:
            assert np.array_equal(got[0][k], other[k]), k
    O.momentum(g, f, coef, 1e-3, -4e-4, 6e-4)
    I = (slice(1, -1),) * 3
    for k in ("us", "vs", "ws"):
        assert np.array_equal(got[0][k][I], f[k][I]), k
