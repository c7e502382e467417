"""Which N x M grids the line transforms run (ftamd_grid_lines), on the CPU, at
sizes on both sides of the rule; on the GPU grids of lengths up to 4096 that
hipFFT runs, against the oracle at the 2-norm 2e-14 of test_gpu_grid.py."""
import numpy as np
import pytest

# N, M, disk, lines: us by the line transforms and by hipFFT (synthesis)
SIZES = [
    (1120, 1125, 0, 0),  # 57.5 / 44.5
    (600, 1215, 0, 0),   # 34.6 / 31.7
    (280, 525, 0, 0),    # 18.9 / 16.9
    (160, 315, 0, 0),    # 17.1 / 15.4
    (1080, 1875, 0, 0),  # 69.8 / 56.8
    (1200, 2401, 0, 0),  # 130.7 / 84.9
    (64, 2187, 0, 0),    # 32.0 / 24.0
    (2250, 63, 0, 0),    # 32.3 / 22.7
    (3072, 3645, 0, 0),  # 431 / 293
    (2187, 2187, 0, 0),  # 300 / 195
    (675, 2187, 0, 0),   # 88.2 / 74.2
    (1000, 1575, 0, 1),  # 44.0 / 52.7
    (1344, 2025, 0, 1),  # 67.5 / 78.9
    (512, 945, 0, 1),    # 23.1 / 27.7
    (64, 125, 0, 1),     # 12.1 / 15.1
    (126, 225, 0, 1),    # 14.6 / 15.0
    (675, 1215, 0, 1),   # 38.5 / 51.6
    (1875, 2401, 0, 1),  # 173 / 201
    (2048, 3125, 0, 1),  # 162 / 173
    (1024, 2047, 0, 1),  # 46.3 / 96.7
    (600, 1199, 0, 1),   # a prime M
    (2500, 1009, 0, 1),  # 92.7 / 93.3
    (1009, 2187, 0, 1),  # 90.6 / 131
    (8192, 255, 0, 1),   # 49.4 / 58.9
    (1200, 2401, 1, 0),  # 171 / 141
    (2250, 63, 1, 0),    # 53.6 / 42.1
    (1080, 1875, 1, 1),  # 98.2 / 97.7
    (1000, 1323, 1, 1),  # 65.6 / 78.8
    (4097, 63, 0, 0), (63, 4097, 0, 0),  # longer than the lines
]


@pytest.mark.parametrize("N,M,disk,lines", SIZES)
def test_rule(ft, N, M, disk, lines):
    assert ft._lib.ftamd_grid_lines(N, M, disk) == lines


@pytest.mark.gpu
@pytest.mark.parametrize("which", ["sph_synthesis", "sphv_analysis", "annulus_synthesis", "disk_synthesis",
                                   "disk_analysis"])
def test_hipfft_grids(ft, which):
    import oracle as O
    import torch
    geo = which.split("_")[0]
    rho = 0.4 if geo == "annulus" else None
    for N, M in ((160, 315), (2187, 63)):
        assert ft._lib.ftamd_grid_lines(N, M, geo == "disk") == (N == 160 and geo == "disk")
        X = np.asfortranarray(np.random.default_rng(N + M).standard_normal((N, M)))
        for trans in ("N", "T"):
            syn = which.endswith("synthesis") == (trans == "N")
            make = getattr(ft, "plan_%s_%s" % (geo, "synthesis" if syn else "analysis"))
            print("grid", which, trans, N, M, flush=True)
            P = make(N, M, rho) if rho else make(N, M)
            ref = O.grid(which, trans, syn, geo == "sphv", X, rho)
            for shift in (0, 1):
                buf = torch.empty(N * M + 2, dtype=torch.float64, device="cuda")
                T = buf[shift:shift + N * M].view(M, N)
                T.copy_(torch.from_numpy(np.ascontiguousarray(X.T)))
                ft.gpu_execute_sph_grid(which, trans, P, T)
                ft.synchronize()
                assert O.rel2(T.cpu().numpy().T, ref) <= 2e-14, (N, M, shift, trans)
