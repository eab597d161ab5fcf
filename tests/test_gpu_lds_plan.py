"""Plans of the LDS-resident sweeps: what the first solve on a handle pays for its plan, and which plan
a handle runs on when it is stepped alone and in batches in turn."""
import threading
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


def _channels(shape, n, **kw):
    kw = dict(dict(solver=M.SOLVER_SOR, omega=1.8, tol=1e-7, check_every=20, max_iter=40, inner_iters=20), **kw)
    chs = []
    for q in range(n):
        ch = M.Channel(M.channel_config(*shape, 4.0, 2.0, 2.0, 2000.0, **kw))
        ch.init_fields(seed=q, amp=0.05, dt=5e-4)
        chs.append(ch)
    return chs


def _lds(stats):
    return [stats.stage[q].lds_sweeps for q in range(3)]


def test_a_batch_leaves_the_plan_of_single_steps():
    """FP64 at 160 x 128 x 96: the sweeps fit the whole device's LDS, not half of it.  A batch of two
    runs on the streaming sweeps, and each channel stepped alone before and after it on the same
    whole-device plan; the same for a smaller grid, whose batch has plans of its own."""
    dt = 5e-4
    for shape, batched in (((160, 128, 96), 0), ((48, 32, 24), 1)):
        chs = _channels(shape, 2)
        assert _lds(chs[0].step(dt)) == [1, 1, 1], chs[0].info()
        alone = chs[0].info()
        for _ in range(2):
            stats = M.step_batch(chs, dt)
            assert [_lds(s) for s in stats] == [[batched] * 3] * 2, [ch.info() for ch in chs]
            assert chs[0].info() != alone
            assert _lds(chs[0].step(dt)) == [1, 1, 1], chs[0].info()
            assert chs[0].info() == alone
        for ch in chs:
            ch.close()


@pytest.mark.parametrize("precision", [M.PREC_FP64, M.PREC_MIXED])
def test_single_and_batched_steps_give_the_same_bits(precision):
    dt, shape = 5e-4, (48, 33, 26)
    outs = []
    for batched in ((0, 1, 0, 1, 1, 0), (0,) * 6):
        chs = _channels(shape, 3, precision=precision, max_iter=100000)
        for b in batched:
            if b:
                M.step_batch(chs, dt)
            else:
                for ch in chs:
                    ch.step(dt)
        outs.append([ch.download(("un", "vn", "wn", "pn")) for ch in chs])
        for ch in chs:
            ch.close()
    for a, b in zip(*outs):
        for k in a:
            assert np.array_equal(a[k], b[k]), k


def test_a_timed_out_handle_stays_off_in_a_batch(monkeypatch):
    """After three solves whose neighbour waits gave up (a spin limit of 0 polls, set from the host) a
    handle keeps to the streaming sweeps, in a batch too."""
    monkeypatch.setenv("MOBYDIFF_LDS_SPIN_LIMIT", "0")
    chs = _channels((96, 64, 48), 2)
    off = lambda ch: "gave up 3 times" in ch.info()
    for ch in chs:
        for _ in range(10):
            if not off(ch):
                ch.step(5e-4)
    if not all(off(ch) for ch in chs):
        pytest.skip("the neighbours had always published")
    for _ in range(2):
        for s in M.step_batch(chs, 5e-4):
            assert _lds(s) == [0, 0, 0] and all(s.stage[q].lds_restarts == 0 for q in range(3))
    assert all(off(ch) for ch in chs)
    for ch in chs:
        ch.close()


@pytest.mark.parametrize("n", [2, 3, 5, 7])
def test_shares_fit_every_xcd(n):
    """The plans of a batch of n on the eight XCDs of 32 CUs, to which a launch's workgroups are dealt
    in turn: all of them have a CU of their own at once.  For three of 20 x 18 x 28 cells the third of
    256 CUs would hold 84 workgroups, 11 on an XCD and 33 for all three.  Same bits as alone, no
    restart."""
    shape, dt = (20, 18, 28), 5e-4
    outs = []
    for batched in (True, False):
        chs = _channels(shape, n, max_iter=100000)
        for _ in range(2):
            stats = M.step_batch(chs, dt) if batched else [ch.step(dt) for ch in chs]
            assert all(_lds(s) == [1, 1, 1] for s in stats), chs[0].info()
            assert sum(s.stage[q].lds_restarts for s in stats for q in range(3)) == 0
        if batched:
            print(n, chs[0].info(), flush=True)
            for ch in chs:
                cuts = [int(np.prod([int(v) for v in part.split(" workgroups")[0].split()[-1].split("x")]))
                        for part in ch.info().split("; ")]
                assert len(cuts) == 2 and all(n * -(-c // 8) <= 32 for c in cuts), ch.info()
        outs.append([ch.download(("un", "vn", "wn", "pn")) for ch in chs])
        for ch in chs:
            ch.close()
    for a, b in zip(*outs):
        for k in a:
            assert np.array_equal(a[k], b[k]), k


@pytest.mark.parametrize("precision", [M.PREC_FP64, M.PREC_MIXED])
def test_threads_share_the_device_where_their_workgroups_fit(precision):
    """Three channels of 64 workgroups (16^3 cells) stepped by three threads: a CU for each of their 192
    workgroups, so every solve of each stays on the LDS-resident sweeps, with the bits it has alone."""
    dt, steps = 5e-4, 12

    def run(together):
        chs = _channels((16, 16, 16), 3, precision=precision, max_iter=100000)
        lds = [[] for _ in chs]

        def work(q):
            for _ in range(steps):
                st = chs[q].step(dt)
                lds[q] += _lds(st) + [1 - st.stage[s].lds_restarts for s in range(3)]

        th = [threading.Thread(target=work, args=(q,)) for q in range(3)]
        for t in th:
            t.start()
            if not together:
                t.join()
        for t in th:
            t.join()
        out = [ch.download(("un", "vn", "wn", "pn")) for ch in chs]
        print(precision, chs[0].info(), [sum(v) for v in lds], flush=True)
        for ch in chs:
            ch.close()
        return lds, out

    (lds, out), (_, alone) = run(True), run(False)
    assert all(v == [1] * (6 * steps) for v in lds)
    for a, b in zip(out, alone):
        for k in a:
            assert np.array_equal(a[k], b[k]), k
