"""The FFT projection at every transform length: 16 to 1024 points in x and in z (the register
transforms: one pass, two passes with each first radix, three passes), 2 to 8 (the LDS kernels),
numbers of rows and of spectrum columns that leave workgroups partly empty, both workgroup sizes, ny at
the edges of the tridiagonal solves' segments and of the column solves,
against the oracle's FFT projection (bound as for the other FFT tests: 1e-12 of each field), and the FP32 transforms
inside the defect correction against the FP64 solve."""
import numpy as np
import pytest

import mobydiff_amd as M
from oracle import oracle as O

pytestmark = pytest.mark.gpu

SHAPES = [(n, 5, 16) for n in (16, 32, 64, 128, 256, 512, 1024)] + [(16, 3, n) for n in (32, 64, 128, 256, 512, 1024)] \
    + [(2, 4, 32), (32, 4, 2), (8, 7, 64), (64, 70, 4), (128, 33, 32), (32, 17, 128)] \
    + [(32, ny, 16) for ny in (2, 63, 64, 65, 128, 129, 192, 193, 256, 257)] \
    + [(32, ny, 64) for ny in (2, 32, 33, 64, 65, 96, 97, 104, 105)] + [(16, 32, 128), (16, 33, 128), (64, 128, 32), (64, 129, 32)]
# enough lines for workgroups of 256 threads (the ones above take 64)
LARGE = [(256, 65, 256), (64, 257, 256), (1024, 65, 64)]


def _rel(a, b):
    return np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300)


def _channel(g, f, **kw):
    cfg = M.channel_config(g.nx, g.ny, g.nz, g.lx, g.ly, g.lz, g.re, solver=M.SOLVER_FFT, p_neumann_y=False,
                           stretch_beta=g.beta or 0.0, **kw)
    ch = M.Channel(cfg)
    ch.upload(**f)
    return ch


@pytest.mark.parametrize("shape", SHAPES + LARGE)
@pytest.mark.parametrize("beta", [None, 1.5])
def test_projection_matches_oracle(shape, beta):
    print(shape, beta, flush=True)
    g = O.Grid(*shape, lx=2.0, ly=2.0, lz=1.0, periodic=(1, 0, 1), beta=beta)
    f = O.random_fields(g, np.random.default_rng(31))
    ch = _channel(g, f)
    ch.apply_bc()
    ch.pressure_projection(0.07)
    ch.apply_bc()
    out = ch.download()
    div = ch.div_norm()
    ch.close()
    O.apply_bc_fft(g, f)
    O.projection_fft(g, f, None, 0.07)
    O.apply_bc_fft(g, f)
    for k in ("un", "vn", "wn", "pn"):
        assert _rel(out[k], f[k]) < 1e-12, (k, _rel(out[k], f[k]))
    # the divergence is a difference of velocities over a spacing: their rounding, over the smallest one
    assert div < 1e-11 * max(1.0, max(shape[0], shape[2]) / 64.0)


@pytest.mark.parametrize("shape", [s for s in SHAPES if s[0] * s[2] <= 8192] + LARGE[:1])
def test_mixed_solve_matches_fp64(shape):
    print(shape, flush=True)
    g = O.Grid(*shape, lx=2.0, ly=2.0, lz=1.0, periodic=(1, 0, 1), beta=1.5)
    f = O.random_fields(g, np.random.default_rng(32))
    got = []
    for prec in (M.PREC_FP64, M.PREC_MIXED):
        ch = _channel(g, f, precision=prec, tol=1e-9)
        ch.apply_bc()
        st = ch.pressure_projection(0.07)
        assert st.converged == 1
        got.append(ch.download(("un", "vn", "wn", "pn")))
        ch.close()
    for k in got[0]:
        assert _rel(got[1][k], got[0][k]) < 1e-7, (k, _rel(got[1][k], got[0][k]))


@pytest.mark.parametrize("shape", [(16, 6, 16), (8, 7, 64), (96 + 32, 33, 32), (64, 257, 256)])
@pytest.mark.parametrize("tol,passes", [(1e-2, 1), (1e-9, 2)])
def test_mixed_passes(shape, tol, passes):
    """One pass, several, and none: a predictor that is divergence-free within the tolerance already
    (the projected field again, its ghosts filled) stays as it is."""
    print(shape, tol, flush=True)
    g = O.Grid(*shape, lx=2.0, ly=2.0, lz=1.0, periodic=(1, 0, 1), beta=1.5)
    f = O.random_fields(g, np.random.default_rng(33))
    ch = _channel(g, f, precision=M.PREC_MIXED, tol=tol)
    ch.apply_bc()
    st = ch.pressure_projection(0.07)
    assert st.converged == 1 and st.checks == st.iterations + 1 and st.div0_inf > 1.0 and st.div_inf < tol
    assert st.iterations == 1 if passes == 1 else st.iterations >= 1
    ch.apply_bc()
    out = ch.download()
    ch.upload(us=out["un"], vs=out["vn"], ws=out["wn"])
    again = ch.pressure_projection(0.07)
    assert again.converged == 1 and again.iterations == 0 and again.checks == 1
    assert again.div_inf == again.div0_inf
    ch.apply_bc()
    new = ch.download()
    for k in ("un", "vn", "wn", "pn"):
        assert np.array_equal(new[k], out[k]), k
    ch.close()
