"""The triangular products of the harmonic transforms at the edges of their
tiles (32 x 32) and stages (16 along k): degrees around multiples of 16 and
32, column counts that leave classes of a few columns, both sides, both
transposes, and the Chebyshev normalization that goes with the product beside
it (tri2cheb and cheb2tri with both products and with either alone).

Tolerance: the products are FP64 sums of at most n terms of matrices whose
condition grows slowly with n; the bar of the larger sizes, a relative 2-norm
of 1e-14 against the long double composite, covers n <= 96 with room.
"""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

EDGES = [15, 16, 17, 31, 32, 33, 48, 63, 65, 96]


def _compare(ft, transform, H, Q, P, Pinv, n, Ms, **kw):
    for M in Ms:
        for trans in "NT":
            A = np.asfortranarray(np.random.default_rng(n + M).uniform(-1, 1, (n, M)))
            print("tiles", transform, trans, n, M, flush=True)
            G = getattr(ft, "execute_" + transform)(trans, H, A.copy(order="F"))
            R = O.harmonic(transform, trans, Q, P, Pinv, A.copy(order="F"), **kw)
            assert O.rel2(G, R) <= 1e-14, (transform, trans, n, M, O.rel2(G, R))


@pytest.mark.parametrize("n", EDGES)
@pytest.mark.parametrize("transform", ["sph2fourier", "fourier2sph"])
def test_classes(ft, transform, n):
    P = (O.connection("leg2cheb", 1, 0, n), O.connection("ultra2ultra", 1, 0, n, 1.5, 1.0))
    Pinv = (O.connection("cheb2leg", 0, 1, n), O.connection("ultra2ultra", 0, 1, n, 1.0, 1.5))
    _compare(ft, transform, ft.plan_sph2fourier(n), O.Plan("sph", n), P, Pinv, n, (1, n - 1 + n % 2, 2 * n - 1))


@pytest.mark.parametrize("n", EDGES)
@pytest.mark.parametrize("params", [(0.0, 0.0, 0.0), (0.25, -0.5, -0.5), (-0.5, -0.75, -0.75)])
@pytest.mark.parametrize("transform", ["tri2cheb", "cheb2tri"])
def test_both_sides(ft, transform, params, n):
    H = ft.plan_tri2cheb(n, *params)
    P, Pinv = (H.P(0), H.P(1)), (H.Pinv(0), H.Pinv(1))
    _compare(ft, transform, H, O.Plan("tri", n, *params), P, Pinv, n, (1, n - 1, n), params=params)
