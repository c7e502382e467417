"""Edges of the band-systolic engine's blocks of 8 steps, against the oracle
bit for bit: streams whose last block is 1..8 positions, bands with every
phase (0, 2, 4, 6 idle steps), row requests that end inside a DMA (4 rows in
FP64, 8 in FP32), chains with absent columns, split chains."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,params", [("sph", ()), ("tri", (0.0, 0.0, 0.0)), ("disk", (0.0, 0.0))])
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("maxpart", [0, 2])
def test_block_edges(ft, kind, params, precision, maxpart):
    import torch
    dt = np.float64 if precision == 0 else np.float32
    plan = {"sph": ft.plan_rotsphere, "tri": ft.plan_rottriangle, "disk": ft.plan_rotdisk}[kind]
    ft.set_engine(ft.ENGINE_SYSTOLIC)
    ft.set_systolic(maxpart)
    try:
        for n in (6, 34, 65, 66, 67, 68, 69, 131, 136, 141, 262, 327):
            P, Q = plan(n, *params), O.Plan(kind, n, *params)
            full = {"sph": 2 * n - 1, "tri": n, "disk": 4 * n - 3}[kind]
            for M in (full, (full * 2 // 3) | 1):
                A = O.fill(kind, n, full, n)[:, :M].astype(dt).copy(order="F")
                for d in (0, 1):
                    T = torch.from_numpy(np.ascontiguousarray(A.T)).cuda()
                    ft.gpu_execute(P, d, T, M=M, precision=precision)
                    ft.synchronize()
                    R = (O.execute if precision == 0 else O.execute_f32)(Q, d, A.copy(order="F"), M)
                    assert np.array_equal(T.cpu().numpy().T, R), (n, M, d)
    finally:
        ft.set_engine(ft.ENGINE_AUTO)
        ft.set_systolic(0)


@pytest.mark.parametrize("kind,params,n", [("sph", (), 128), ("sph", (), 256), ("tri", (0.0, 0.0, 0.0), 64),
                                           ("disk", (0.0, 0.0), 64), ("disk", (0.0, 0.0), 128)])
@pytest.mark.parametrize("d", [0, 1])
def test_tables_that_end_with_their_page(ft, kind, params, n, d):
    """FP32 tables whose last byte is the last of a 4 KB page: what the last
    steps read ahead is still inside them."""
    import torch
    plan = {"sph": ft.plan_rotsphere, "tri": ft.plan_rottriangle, "disk": ft.plan_rotdisk}[kind]
    M = {"sph": 2 * n - 1, "tri": n, "disk": 4 * n - 3}[kind]
    ft.set_engine(ft.ENGINE_SYSTOLIC)
    try:
        P, Q = plan(n, *params), O.Plan(kind, n, *params)
        A = O.fill(kind, n, M, n).astype(np.float32).copy(order="F")
        T = torch.from_numpy(np.ascontiguousarray(A.T)).cuda()
        print("page end", kind, n, d, flush=True)
        ft.gpu_execute(P, d, T, M=M, precision=1)
        ft.synchronize()
        assert np.array_equal(T.cpu().numpy().T, O.execute_f32(Q, d, A.copy(order="F"), M))
    finally:
        ft.set_engine(ft.ENGINE_AUTO)
