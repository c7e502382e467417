"""Edges of the line transforms behind the sphere's, the vector field's, the
annulus's and the disk's grids: lengths on both sides of every power of two
(where the convolution's length changes), powers of two, the longest lines
they take and the first that fall to hipFFT, odd N (a last row alone), an X
that is not 16-byte aligned.  Bar: the relative 2-norm 2e-14 of
test_gpu_grid.py, from log2(2 L) passes of a few eps each."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

SIZES = [(3, 1), (4, 7), (31, 33), (32, 65), (33, 63), (63, 31), (64, 129), (127, 5), (128, 255), (129, 257),
         (511, 9), (512, 7), (513, 511), (1023, 5), (1025, 3), (2048, 5), (2049, 3), (4095, 3), (4096, 3), (4097, 3),
         (8192, 3), (6, 4095), (7, 2049), (6, 4097), (7, 4099)]
CASES = [(w, t) for w in ("sph_synthesis", "sphv_analysis", "annulus_synthesis", "annulus_analysis", "disk_synthesis",
                          "disk_analysis") for t in ("N", "T")]


@pytest.mark.parametrize("which,trans", CASES)
def test_line_lengths(ft, which, trans):
    import torch
    geo = which.split("_")[0]
    syn = (which.endswith("synthesis")) == (trans == "N")
    make = getattr(ft, "plan_%s_%s" % (geo, "synthesis" if syn else "analysis"))
    rho = 0.4 if geo == "annulus" else None
    for N, M in SIZES:
        P = make(N, M, rho) if rho else make(N, M)
        X = np.asfortranarray(np.random.default_rng(N + 3 * M).standard_normal((N, M)))
        ref = O.grid(which, trans, syn, geo == "sphv", X, rho)
        for shift in (0, 1):
            buf = torch.empty(N * M + 2, dtype=torch.float64, device="cuda")
            T = buf[shift:shift + N * M].view(M, N)
            T.copy_(torch.from_numpy(np.ascontiguousarray(X.T)))
            ft.gpu_execute_sph_grid(which, trans, P, T)
            ft.synchronize()
            err = O.rel2(T.cpu().numpy().T, ref)
            assert err <= 2e-14, (N, M, shift, err)
