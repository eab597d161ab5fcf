"""A learned solve that finds the device's places for the LDS-resident sweeps taken gives the bits it
gives with them, and so does a handle that always streams: here the solves whose network start is
rejected after the stage's previous solve took one, whose first batch is queued before the choice is
read."""
import os
import threading
import time

import numpy as np
import pytest

import mobydiff_amd as M

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
WEIGHTS = os.path.join(ROOT, "mobydiff_amd", "weights", "unet_guess_s4_wavy_192x128x96.npz")
NX, NY, NZ, DT = 192, 128, 96, 5e-4


def _cfg(**kw):
    return M.channel_config(NX, NY, NZ, 4.0, 2.2, 2.0, 2000.0, solver=M.SOLVER_SOR, omega=1.8, flowrate=True,
                            flow_height=2.0, **dict(dict(tol=1e-8, max_iter=400000, check_every=20, inner_iters=20,
                                                         precision=M.PREC_MIXED), **kw))


@pytest.mark.skipif(not os.path.exists(WEIGHTS), reason="trained U-Net parameters not present")
def test_rejected_learned_start_has_the_same_bits_on_any_sweeps(monkeypatch):
    from mobydiff_amd import train_guess
    monkeypatch.setenv("MOBYDIFF_NET_MARGIN", "1.0")
    monkeypatch.setenv("MOBYDIFF_NET_TIME_GATE", "0")
    # a solve of its own that keeps all places: FP64 sweeps that never reach their tolerance
    holder = M.Channel(_cfg(precision=M.PREC_FP64, tol=1e-300, max_iter=200000))
    holder.init_fields(seed=9, amp=0.05, dt=DT)
    runs = []
    for taken, mode in ((False, "2"), (True, "2"), (False, "0")):
        monkeypatch.setenv("MOBYDIFF_LDS_SOR", mode)
        net = M.Net(NX, NY, NZ, seed=0, stride=train_guess.stride_of(WEIGHTS))
        train_guess.load(WEIGHTS, net)
        ch = M.Channel(_cfg())
        geo = M.wavy_geometry(A=0.1)
        ch.compute_ibm(geo)
        ch.init_fields(seed=0, amp=0.05, geo=geo, dt=DT)
        for _ in range(6):
            ch.step(DT)
        ch.attach_net(net)
        ch.set_guess(M.GUESS_LEARNED)
        for _ in range(40):   # until every stage's solve starts from the network's guess
            st = ch.step(DT)
            if all(st.stage[q].fallback == 0 for q in range(3)):
                break
        assert all(st.stage[q].fallback == 0 for q in range(3))
        p, c0 = net.get_params()
        net.set_params(p, 1e3 * c0)   # now its starts are far off
        done = []
        if taken:
            th = threading.Thread(target=lambda: done.append(holder.pressure_projection(1e-3)))
            th.start()
            time.sleep(0.1)
        st = ch.step(DT)
        if taken:
            assert not done, "the holder ended early"
            th.join()
        runs.append(([(s.iterations, s.checks, s.fallback, s.lds_restarts) for s in st.stage], [s.lds_sweeps for s in st.stage],
                     ch.download(("un", "vn", "wn", "pn"))))
        print(runs[-1][:2], flush=True)
        ch.attach_net(None)
        ch.close()
        net.close()
    holder.close()
    assert [r[1] for r in runs] == [[1, 1, 1], [0, 0, 0], [0, 0, 0]]
    assert all(s[2] == 1 for s in runs[0][0])
    for r in runs[1:]:
        assert r[0] == runs[0][0]
        for k in r[2]:
            assert np.array_equal(r[2][k], runs[0][2][k]), k
