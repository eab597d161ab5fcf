"""The LDS-resident red-black sweeps where the subdomains are not all alike: grids whose pairs no
cut divides, an odd number of wall-normal cells, one workgroup along an axis, periodic y, a
stretched wall-normal grid and the smallest grid the half-column form takes.  FP64 batches against
the oracle and FP32 batches against the streaming sweeps, bit for bit; a batch of channels on its
share of the CUs against single runs; and a solve that finds the device's LDS turn taken."""
import threading

import numpy as np
import pytest

import mobydiff_amd as M
from oracle import oracle as O

pytestmark = pytest.mark.gpu

SHAPES = [((100, 70, 54), 0, "wavy"), ((102, 35, 22), 0, "wavy"), ((36, 21, 20), 0, None), ((52, 18, 30), 1, None),
          ((100, 70, 54), 0, "stretch"), ((46, 33, 26), 0, "stretch"), ((8, 5, 8), 0, None)]


def _grid(shape, per_y, kind):
    g = O.Grid(*shape, lx=4.0, ly=2.2, lz=2.0, re=2000.0, periodic=(1, per_y, 1),
               beta=1.5 if kind == "stretch" else None)
    g.bc_type[O.bci(2, 0, 0)] = 1
    g.bc_type[O.bci(2, 1, 0)] = 1
    return g, (O.ibm_coefs(g, O.Geometry(kind=1, A=0.1, lam=1.0, half_height=1.0)) if kind == "wavy" else None)


def _channel(shape, per_y, kind, coef, f, **kw):
    cfg = M.channel_config(*shape, 4.0, 2.2, 2.0, 2000.0, periodic=(1, per_y, 1), solver=M.SOLVER_SOR, omega=1.8,
                           stretch_beta=1.5 if kind == "stretch" else 0.0, **kw)
    ch = M.Channel(cfg)
    if coef is not None:
        ch.set_ibm(*coef)
    ch.upload(**f)
    return ch


@pytest.mark.parametrize("shape,per_y,kind", SHAPES)
def test_fp64_batches_equal_oracle(shape, per_y, kind):
    g, coef = _grid(shape, per_y, kind)
    f = O.random_fields(g, np.random.default_rng(41), amp=0.05)
    n, every = 17, 7   # two whole batches and a shorter one
    ch = _channel(shape, per_y, kind, coef, f, tol=1e-300, max_iter=n, check_every=every)
    st = ch.pressure_projection(0.02)
    print(shape, kind, ch.info(), flush=True)
    assert st.lds_sweeps == 1 and st.iterations == n and st.checks == 4
    out = ch.download()
    ch.close()
    O.projection_sor(g, f, coef, 1.8, 0.0, n, every, 0.02)
    for k in ("un", "vn", "wn", "pn"):
        assert np.array_equal(out[k], f[k]), k


@pytest.mark.parametrize("precision", [M.PREC_FP64, M.PREC_MIXED])
@pytest.mark.parametrize("shape,per_y,kind", SHAPES[:5])
def test_solves_equal_streaming_sweeps(shape, per_y, kind, precision, monkeypatch):
    g, coef = _grid(shape, per_y, kind)
    f = O.random_fields(g, np.random.default_rng(42), amp=0.05)
    got = []
    for mode in ("2", "0"):
        monkeypatch.setenv("MOBYDIFF_LDS_SOR", mode)
        ch = _channel(shape, per_y, kind, coef, f, tol=1e-6, max_iter=600, check_every=20, precision=precision,
                      inner_iters=20)
        st = ch.pressure_projection(5e-4 * 64 / 120)
        got.append((st.iterations, st.checks, st.div0_inf, st.div_inf, ch.download(), st.lds_sweeps))
        ch.close()
    assert got[0][5] == 1 and got[1][5] == 0
    assert got[0][:4] == got[1][:4]
    for k in ("un", "vn", "wn", "pn"):
        assert np.array_equal(got[0][4][k], got[1][4][k]), k


@pytest.mark.parametrize("precision", [M.PREC_FP64, M.PREC_MIXED])
def test_batch_runs_on_its_share_of_the_cus(precision):
    shape, n, dt = (48, 33, 26), 5, 5e-4
    starts, chs = [], []
    for q in range(n):
        g, coef = _grid(shape, 0, "wavy")
        f = O.random_fields(g, np.random.default_rng(50 + q), amp=0.02)
        starts.append((coef, f))
        chs.append(_channel(shape, 0, "wavy", coef, f, tol=1e-7, check_every=20, precision=precision))
    stats = [M.step_batch(chs, dt) for _ in range(2)][-1]
    assert all(s.stage[q].lds_sweeps == 1 for s in stats for q in range(3)), chs[0].info()
    outs = [ch.download(("un", "vn", "wn", "pn")) for ch in chs]
    for ch in chs:
        ch.close()
    for (coef, f), out in zip(starts, outs):
        ch = _channel(shape, 0, "wavy", coef, f, tol=1e-7, check_every=20, precision=precision)
        for _ in range(2):
            ch.step(dt)
        one = ch.download(("un", "vn", "wn", "pn"))
        ch.close()
        for k in out:
            assert np.array_equal(out[k], one[k]), k


def test_two_threads_step_two_channels():
    """Two handles stepped by two threads at once: one solve at a time holds the device's LDS turn,
    the other runs on the streaming sweeps; both give what they give alone, without a restart."""
    shape, dt, steps = (64, 48, 32), 5e-4, 4
    g, coef = _grid(shape, 0, "wavy")
    fs = [O.random_fields(g, np.random.default_rng(60 + q), amp=0.02) for q in range(2)]

    def alone(f):
        ch = _channel(shape, 0, "wavy", coef, f, tol=1e-7, check_every=20)
        for _ in range(steps):
            ch.step(dt)
        out = ch.download(("un", "vn", "wn", "pn"))
        ch.close()
        return out

    ref = [alone(f) for f in fs]
    chs = [_channel(shape, 0, "wavy", coef, f, tol=1e-7, check_every=20) for f in fs]
    restarts = [0, 0]

    def work(q):
        for _ in range(steps):
            st = chs[q].step(dt)
            restarts[q] += sum(st.stage[s].lds_restarts for s in range(3))

    th = [threading.Thread(target=work, args=(q,)) for q in range(2)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    outs = [ch.download(("un", "vn", "wn", "pn")) for ch in chs]
    for ch in chs:
        ch.close()
    assert restarts == [0, 0]
    for q in range(2):
        for k in ref[q]:
            assert np.array_equal(outs[q][k], ref[q][k]), (q, k)
