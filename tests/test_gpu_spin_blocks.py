"""The first stage of the spin-weighted sphere's rotations at the edges of its
blocks (16 elements of a column) and waves (four columns; one, two or four
sequences at a time, orders below |s| apart), bit for bit against the oracle.
"""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("s", [1, -2, 3, 4, -5, 7, 8])
@pytest.mark.parametrize("n", [9, 15, 16, 17, 18, 19, 31, 33, 35, 49, 52])
def test_edges_bitwise(ft, s, n):
    P, Q = ft.plan_rotspinsphere(n, s), O.SpinPlan(n, s)
    for M in sorted({3, 2 * abs(s) - 1, 2 * abs(s) + 5, 2 * n - 1} & set(range(1, 2 * n))):
        g = np.random.default_rng(100 * n + M)
        A = np.asfortranarray(g.uniform(-1, 1, (n, M)) + 1j * g.uniform(-1, 1, (n, M)))
        for d, run in ((0, ft.execute_spinsph_hi2lo), (1, ft.execute_spinsph_lo2hi)):
            print("spin blocks s=%d n=%d M=%d dir=%d" % (s, n, M, d), flush=True)
            got = run(P, A.copy(order="F"), M)
            ref = O.execute_spinsph(Q, d, A.copy(order="F"), M)
            assert np.array_equal(got, ref), (s, n, M, d, O.rel2(got, ref))
