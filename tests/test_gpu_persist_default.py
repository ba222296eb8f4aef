"""Built-in launch rules: one launch per warping with neighbour flags while no
other solve of the process runs persistent warpings on the device, host-paced
launches otherwise.  The kernels compute the oracle's expressions in the
oracle's order, so every path has to give its bits."""
import threading

import numpy as np
import pytest

import oracle as O
from amdflow import PERSIST_HOST_PACED, PERSIST_PLAIN, TV_L1, persist_launch_mode, \
    set_persist_launch_mode, synth
from amdflow import debug as D

pytestmark = pytest.mark.gpu


@pytest.fixture
def restore_mode():
    set_persist_launch_mode(PERSIST_PLAIN)
    yield
    D.persist_force_not_resident(False)
    set_persist_launch_mode(PERSIST_PLAIN)


def _pair(w, h, seed):
    I0, I1, _, _ = synth.make_pair(w, h, 4.0, seed, bumps=True)
    return synth.quantize(I0), synth.quantize(I1)


def _solve(tv, q0, q1):
    """(flow, iterations, the launch modes the solve's scales took)."""
    tv.profile(True)
    tv.runDualTVL1Multiscale(q0, q1)
    modes = {p["persistent"] for p in tv.profile_results() if p["launches"]}
    tv.profile(False)
    return tv.getU().copy(), tv.iterations(), modes


def _check(got, q0, q1, **prm):
    uo, ito = O.tvl1(q0, q1, O.default_params(**prm))
    assert np.array_equal(got[1], ito)
    assert np.array_equal(got[0], uo)


@pytest.mark.parametrize("w,h,ns", [(16, 9, 1), (320, 240, 5), (641, 479, 5), (1600, 999, 2),
                                    (1601, 1000, 2)])
def test_builtin_rules_match_oracle(w, h, ns, restore_mode):
    print("builtin", w, h, flush=True)
    q0, q1 = _pair(w, h, 61)
    prm = dict(nscales=ns, max_iterations=60)
    with TV_L1(w, h, **prm) as tv:
        got = _solve(tv, q0, q1)
    assert got[2] == {2}
    _check(got, q0, q1, **prm)


def test_iteration_limits_past_the_flags_run_host_paced(restore_mode):
    """A flag numbers up to 2^20 chunks: longer limits keep the host-paced
    launches, and stop where the flow does."""
    q0, q1 = _pair(64, 48, 62)
    prm = dict(nscales=2, max_iterations=(1 << 20) + 1)
    with TV_L1(64, 48, **prm) as tv:
        got = _solve(tv, q0, q1)
    assert got[2] == {0}
    _check(got, q0, q1, **prm)


def test_not_resident_keeps_the_process_and_paces_the_handle(restore_mode):
    q0, q1 = _pair(160, 120, 63)
    with TV_L1(160, 120, nscales=3) as tv:
        D.persist_force_not_resident(True)
        tv.runDualTVL1Multiscale(q0, q1)
        first = (tv.getU().copy(), tv.iterations())
        D.persist_force_not_resident(False)
        assert persist_launch_mode() == PERSIST_PLAIN
        again = [_solve(tv, q0, q1) for _ in range(17)]
    assert all(g[2] == {0} for g in again[:16]) and again[16][2] == {2}
    for got in [first] + again:
        _check(got, q0, q1, nscales=3)


def test_back_off_starts_again_after_a_persistent_solve(restore_mode):
    """Two misses with persistent solves between pace 16 solves each; misses one
    after the other pace 16, 32, .. up to 256."""
    q0, q1 = _pair(80, 60, 65)

    def paced_after_a_miss(tv, missed):
        D.persist_force_not_resident(True)
        tv.runDualTVL1Multiscale(q0, q1)
        D.persist_force_not_resident(False)
        for n in range(missed):   # these do not try
            assert _solve(tv, q0, q1)[2] == {0}

    with TV_L1(80, 60, nscales=2, max_iterations=8) as tv:
        for _ in range(3):
            paced_after_a_miss(tv, 16)
            assert _solve(tv, q0, q1)[2] == {2}
        for missed in (16, 32, 64, 128, 256, 256):
            paced_after_a_miss(tv, missed)
        assert _solve(tv, q0, q1)[2] == {2}


def test_host_paced_process_takes_host_paced_rules(restore_mode):
    q0, q1 = _pair(160, 120, 64)
    set_persist_launch_mode(PERSIST_HOST_PACED)
    with TV_L1(160, 120, nscales=3) as tv:
        got = _solve(tv, q0, q1)
    assert got[2] == {0}
    _check(got, q0, q1, nscales=3)


def test_a_solve_behind_other_work_does_not_hold_the_turn(restore_mode):
    """A solve whose stream still has a tenth of a second of other work to do
    runs nothing persistent yet: another handle's solve takes the turn
    meanwhile instead of waiting in vain and running host-paced."""
    import time

    import torch
    W, H = 640, 480
    q0, q1 = _pair(W, H, 66)
    prm = dict(nscales=3, max_iterations=60)
    d0, d1 = torch.from_numpy(q0).cuda(), torch.from_numpy(q1).cuda()
    dU = torch.empty(2 * W * H, dtype=torch.float32, device="cuda")
    st = torch.cuda.Stream()
    with TV_L1(W, H, **prm) as a, TV_L1(W, H, **prm) as b:
        _solve(b, q0, q1)
        a.run_device_u8(d0.data_ptr(), d1.data_ptr(), dU.data_ptr(), st.cuda_stream)
        torch.cuda.synchronize()
        with torch.cuda.stream(st):
            torch.cuda._sleep(300_000_000)
        t = threading.Thread(target=a.run_device_u8,
                             args=(d0.data_ptr(), d1.data_ptr(), dU.data_ptr(), st.cuda_stream))
        t.start()
        time.sleep(0.02)
        behind = not st.query()
        got = _solve(b, q0, q1)
        behind &= not st.query()
        t.join()
        torch.cuda.synchronize()
        first = (dU.cpu().numpy(), a.iterations())
    assert behind, "the other work ended too early to show anything"
    assert got[2] == {2}
    _check(got, q0, q1, **prm)
    _check(first, q0, q1, **prm)


def test_own_rules_do_not_run_beside_a_builtin_solve(restore_mode):
    """While a long solve on the built-in rules has the device, a handle with
    persistent rules of its own waits 20 ms for it and then runs host-paced:
    beside it, either grid may not be resident, and the process would become
    host-paced for good."""
    import time
    q0, q1 = _pair(320, 240, 67)
    L0, L1 = _pair(1280, 720, 68)
    prm = dict(nscales=3, max_iterations=60)
    with TV_L1(1280, 720, nscales=1, warps=60, epsilon=0.0) as a, TV_L1(320, 240, **prm) as b:
        b.set_launch_rule(0, 4, 0, 2)
        t = threading.Thread(target=a.runDualTVL1Multiscale, args=(L0, L1))
        t0 = time.monotonic()
        t.start()
        time.sleep(0.01)
        got = _solve(b, q0, q1)
        t.join()
        took = time.monotonic() - t0
    assert took > 0.06, "the long solve ended too early to show anything"
    assert persist_launch_mode() == PERSIST_PLAIN
    assert got[2] == {0}
    _check(got, q0, q1, **prm)


def test_solves_from_several_threads(restore_mode):
    """One solve at a time takes the persistent rules, the others run host-paced
    beside it."""
    pairs = [_pair(320, 240, 70 + k) for k in range(3)]
    want = [O.tvl1(q0, q1, O.default_params(nscales=4)) for q0, q1 in pairs]
    results, errors = [[] for _ in pairs], []

    def worker(k):
        try:
            with TV_L1(320, 240, nscales=4) as tv:
                for _ in range(5):
                    tv.runDualTVL1Multiscale(*pairs[k])
                    results[k].append((tv.getU().copy(), tv.iterations()))
        except Exception as e:   # reported by the main thread
            errors.append(e)

    th = [threading.Thread(target=worker, args=(k,)) for k in range(len(pairs))]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not errors, errors
    assert persist_launch_mode() == PERSIST_PLAIN
    for k, (uo, ito) in enumerate(want):
        assert len(results[k]) == 5
        for u, it in results[k]:
            assert np.array_equal(it, ito)
            assert np.array_equal(u, uo)


def test_threads_take_turns_at_persistent_solves(restore_mode):
    """From 200000 pixels on a solve waits for the device's turn: solves
    of two threads are persistent one after the other."""
    q0, q1 = _pair(640, 480, 69)
    prm = dict(nscales=3, max_iterations=40)
    got, errors = [], []

    def worker():
        try:
            with TV_L1(640, 480, **prm) as tv:
                for _ in range(4):
                    got.append(_solve(tv, q0, q1))
        except Exception as e:   # reported by the main thread
            errors.append(e)

    th = [threading.Thread(target=worker) for _ in range(2)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not errors, errors
    assert len(got) == 8 and sum(g[2] == {2} for g in got) >= 1
    for g in got:
        _check(g, q0, q1, **prm)
