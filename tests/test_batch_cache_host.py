"""Which kept schedule a batch call takes (ftamd_batch_entry), on the CPU: a
schedule that a graph was captured from, or that cannot take other matrices
(the pipelined engine's), stays while others are empty or older; on the GPU a
captured batch replays after the same plans ran on other matrices."""
import ctypes

import numpy as np
import pytest

RUN, REBASE, BUILD = 0, 1, 2


class State(ctypes.Structure):
    _fields_ = [("match", ctypes.c_int), ("held", ctypes.c_int), ("captured", ctypes.c_int), ("rebase", ctypes.c_int),
                ("used", ctypes.c_ulonglong)]


def _entry(ft, states):
    """Entries as (match, captured, rebase, used), None an empty one."""
    e = (State * len(states))(*[State(s[0], 1, s[1], s[2], s[3]) if s else State(0, 0, 0, 0, 0) for s in states])
    action = ctypes.c_int(-1)
    fn = ft._lib.ftamd_batch_entry
    fn.restype, fn.argtypes = ctypes.c_int, [ctypes.c_void_p, ctypes.c_int, ctypes.c_void_p]
    k = fn(ctypes.byref(e), len(states), ctypes.byref(action))
    return k, action.value


@pytest.mark.parametrize("states,want", [
    ([None] * 8, (0, BUILD)),
    # the list itself, captured or not
    ([(0, 0, 0, 5), (2, 1, 0, 1), None], (1, RUN)),
    # the same plans on other matrices: taken over, or left alone beside an empty entry
    ([(1, 0, 1, 3), None], (0, REBASE)),
    ([(1, 1, 0, 3), None, None], (1, BUILD)),
    ([(1, 0, 0, 3), None], (1, BUILD)),
    # two of them: the one whose launch ended first; the captured one never
    ([(1, 0, 1, 9), (1, 0, 1, 4), None], (1, REBASE)),
    ([(1, 1, 0, 1), (1, 0, 1, 4), None], (1, REBASE)),
    # no empty one: the least recently used, captured ones last
    ([(1, 0, 0, 3), (0, 0, 0, 2), (0, 0, 0, 7)], (1, BUILD)),
    ([(0, 1, 0, 1), (0, 0, 0, 8), (0, 0, 0, 6)], (2, BUILD)),
    ([(0, 1, 0, 5), (1, 1, 0, 4), (0, 1, 0, 9)], (1, BUILD)),
])
def test_entry(ft, states, want):
    assert _entry(ft, states) == want


@pytest.mark.gpu
@pytest.mark.parametrize("engine", [1, 2])
def test_captured_batch_keeps_its_schedule(ft, engine):
    """A batch captured in a graph, then the same plans on other matrices and
    six other lists; every replay is the oracle's, bit for bit."""
    import oracle as O
    import torch
    ft.set_engine(engine)
    try:
        ns = [40, 21, 67]
        plans, Qs = [ft.plan_rotsphere(n) for n in ns], [O.Plan("sph", n) for n in ns]
        As = [O.fill("sph", n, 2 * n - 1, n) for n in ns]
        X = [torch.from_numpy(np.ascontiguousarray(A.T)).cuda() for A in As]
        T, other = [x.clone() for x in X], [torch.zeros_like(x) for x in X]
        want = [O.execute(Q, 0, A.copy(order="F")) for Q, A in zip(Qs, As)]
        ft.gpu_execute_batch(plans, 0, T)
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            ft.gpu_execute_batch(plans, 0, T)
        more = []
        for k in range(7):
            if k == 0:
                ft.gpu_execute_batch(plans, 0, other)
            else:
                more.append(ft.plan_rotsphere(10 + k))
                ft.gpu_execute_batch([more[-1]], 0, [torch.zeros(19 + 2 * k, 10 + k, dtype=torch.float64, device="cuda")])
            torch.cuda.synchronize()
            for t, x in zip(T, X):
                t.copy_(x)
            g.replay()
            torch.cuda.synchronize()
            assert all(torch.equal(o, torch.zeros_like(o)) for o in other)
            for t, w in zip(T, want):
                assert np.array_equal(t.cpu().numpy().T, w), k
    finally:
        ft.set_engine(ft.ENGINE_AUTO)


@pytest.mark.gpu
def test_a_streams_error_stays_its_own(ft):
    """A batch whose waits expire on one stream (a limit of one poll), then the
    same plans on other matrices on another stream: each stream's check reports
    its own launch."""
    import oracle as O
    import torch
    n = 300
    plans = [ft.plan_rotsphere(n), ft.plan_rotsphere(n - 7)]
    As = [O.fill("sph", P.n, 2 * P.n - 1, P.n) for P in plans]
    A, B = ([torch.from_numpy(np.ascontiguousarray(a.T)).cuda() for a in As] for _ in range(2))
    s1, s2 = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    ft.set_engine(ft.ENGINE_SYSTOLIC)
    try:
        ft.set_spin_limit(1)
        ft.gpu_execute_batch(plans, 0, A, stream=s1)
        torch.cuda.synchronize()
        ft.set_spin_limit(0)
        ft.gpu_execute_batch(plans, 0, B, stream=s2)
        ft.synchronize(s2)
        with pytest.raises(ft.GPUError, match="wait expired"):
            ft.synchronize(s1)
        ft.synchronize(s1)  # reported once
        for P, a, b in zip(plans, As, B):
            assert np.array_equal(b.cpu().numpy().T, O.execute(O.Plan("sph", P.n), 0, a.copy(order="F")))
    finally:
        ft.set_spin_limit(0)
        ft.set_engine(ft.ENGINE_AUTO)
