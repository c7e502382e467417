"""Batches called again on other matrices of the same plans and sizes: the
schedule is kept and its chains take the new matrices.  Every call's results
are bit for bit the oracle's, on one stream, on alternating streams without a
wait between the calls, with more than 256 matrices, and the earlier matrices
keep their values."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def _set(ns, dt, seed):
    import torch
    As = [O.fill("sph", n, 2 * n - 1, seed + k).astype(dt) for k, n in enumerate(ns)]
    return As, [torch.from_numpy(np.ascontiguousarray(A.T)).cuda() for A in As]


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("count,nmax", [(5, 90), (300, 12)])
def test_new_matrices_each_call(ft, precision, count, nmax):
    import torch
    rng = np.random.default_rng(count + precision)
    ns = [int(n) for n in rng.integers(3, nmax, count)]
    dt = np.float64 if precision == 0 else np.float32
    plans, Qs = [ft.plan_rotsphere(n) for n in ns], [O.Plan("sph", n) for n in ns]
    ref = O.execute if precision == 0 else O.execute_f32
    ft.set_engine(ft.ENGINE_SYSTOLIC)
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    try:
        sets = [_set(ns, dt, 1000 * k) for k in range(4)]
        torch.cuda.synchronize()
        for k, (As, Ts) in enumerate(sets):
            print("batch matrices", count, "set", k, flush=True)
            s = streams[(k // 2) % 2]
            with torch.cuda.stream(s):
                ft.gpu_execute_batch(plans, 0, Ts, precision=precision, stream=s)
        torch.cuda.synchronize()
        ft.synchronize()
        for As, Ts in sets:
            for n, Q, A, T in zip(ns, Qs, As, Ts):
                assert np.array_equal(T.cpu().numpy().T, ref(Q, 0, A.copy(order="F"))), (n, precision)
    finally:
        ft.set_engine(ft.ENGINE_AUTO)


def test_more_batches_than_are_kept(ft):
    """Ten batches in turn, twice, then one of them after one of its plans is
    destroyed: each call bit for bit the oracle's."""
    import torch
    ft.set_engine(ft.ENGINE_SYSTOLIC)
    try:
        batches = []
        for k in range(10):
            ns = [20 + k, 33, 7 + k]
            batches.append((ns, [ft.plan_rotsphere(n) for n in ns]))
        for turn in range(2):
            for k, (ns, plans) in enumerate(batches):
                As, Ts = _set(ns, np.float64, 100 * turn + k)
                print("batch in turn", turn, k, flush=True)
                ft.gpu_execute_batch(plans, 1, Ts)
                torch.cuda.synchronize()
                for n, A, T in zip(ns, As, Ts):
                    assert np.array_equal(T.cpu().numpy().T, O.execute(O.Plan("sph", n), 1, A.copy(order="F")))
        ns, plans = batches[9]
        plans[1] = ft.plan_rotsphere(33)
        As, Ts = _set(ns, np.float64, 1)
        ft.gpu_execute_batch(plans, 1, Ts)
        torch.cuda.synchronize()
        for n, A, T in zip(ns, As, Ts):
            assert np.array_equal(T.cpu().numpy().T, O.execute(O.Plan("sph", n), 1, A.copy(order="F")))
    finally:
        ft.set_engine(ft.ENGINE_AUTO)
