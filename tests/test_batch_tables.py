"""Band tables of a batch's plans, made together from the pairs of the largest
plan: on the CPU the pairs of a smaller plan are the first of a larger one's,
bit for bit, for every constructor with a closed form; on the GPU the first
call of a new batch is the oracle's, bit for bit, with plans that have tables
already, plans named twice, plans too small for any, and the annulus's, whose
pairs are each plan's own."""
import numpy as np
import pytest

import oracle as O

MAKERS = {"sph": ("plan_rotsphere", ()), "tri": ("plan_rottriangle", (0.25, -0.5, 1.75)),
          "disk": ("plan_rotdisk", (0.5, -0.25)), "rectdisk": ("plan_rotrectdisk", (0.3,))}


def _columns(geometry, n, values):
    out, at = [], 0
    for m in range(2 * n - 1 if geometry == "disk" else n):
        rows = n - (m + 1) // 2 if geometry == "disk" else n - m
        out.append(values[at:at + rows])
        at += rows
    return out


@pytest.mark.parametrize("which", MAKERS)
def test_pairs_of_smaller_plans(ft, which):
    name, params = MAKERS[which]
    big = getattr(ft, name)(301, *params)
    for n in (1, 2, 3, 64, 177, 300):
        small = getattr(ft, name)(n, *params)
        for v in ("s", "c"):
            for a, b in zip(_columns(which, n, getattr(small, v)), _columns(which, 301, getattr(big, v))):
                assert np.array_equal(a, b[:len(a)]), (n, v)


def _run(ft, plans, Qs, kind, Ms, precision):
    import torch
    dt = np.float64 if precision == 0 else np.float32
    ref = O.execute if precision == 0 else O.execute_f32
    for d in (0, 1):
        As = [O.fill(kind, P.n, M, P.n + k).astype(dt) for k, (P, M) in enumerate(zip(plans, Ms))]
        Ts = [torch.from_numpy(np.ascontiguousarray(A.T)).cuda() for A in As]
        ft.gpu_execute_batch(plans, d, Ts, Ms=Ms, precision=precision)
        ft.synchronize()
        for k, (Q, A, T) in enumerate(zip(Qs, As, Ts)):
            assert np.array_equal(T.cpu().numpy().T, ref(Q, d, A.copy(order="F"))), (d, plans[k].n)


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("which", ["sph", "tri", "disk"])
def test_first_call(ft, which, precision):
    name, params = MAKERS[which]
    ns = [1, 2, 3, 4, 33, 34, 65, 130, 67, 33, 128]
    plans = [getattr(ft, name)(n, *params) for n in ns]
    plans.append(plans[7])
    Qs = [O.Plan(which, P.n, *params) for P in plans]
    Ms = [{"sph": 2 * P.n - 1, "tri": P.n, "disk": 4 * P.n - 3}[which] for P in plans]
    ft.set_engine(ft.ENGINE_SYSTOLIC)
    try:
        print("first call of a batch", which, precision, flush=True)
        _run(ft, plans[:5], Qs[:5], which, Ms[:5], precision)
        _run(ft, plans, Qs, which, Ms, precision)
    finally:
        ft.set_engine(ft.ENGINE_AUTO)


@pytest.mark.gpu
def test_first_call_annulus(ft):
    plans = [ft.plan_rotannulus(n, 0.25, -0.5, 0.0, 0.3) for n in (40, 7, 71)]
    Qs = [O.Plan("annulus", P.n, 0.25, -0.5, rho=0.3) for P in plans]
    ft.set_engine(ft.ENGINE_SYSTOLIC)
    try:
        _run(ft, plans, Qs, "disk", [4 * P.n - 3 for P in plans], 0)
    finally:
        ft.set_engine(ft.ENGINE_AUTO)
