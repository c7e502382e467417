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
    (1875, 1875, 0, 0),  # 85.1 / 143, by the error
    (1875, 2401, 0, 1),  # 173 / 201
    (2048, 3125, 0, 1),  # 162 / 173
    (1024, 2047, 0, 1),  # 46.3 / 96.7
    (600, 1199, 0, 1),   # a prime M
    (2500, 1009, 0, 1),  # 92.7 / 93.3
    (1009, 2187, 0, 1),  # 90.6 / 131
    (8192, 255, 0, 1),   # 49.4 / 58.9
    (1200, 2401, 1, 0),  # 171 / 141
    (2250, 63, 1, 0),    # 53.6 / 42.1
    (1000, 1323, 1, 1),  # 65.6 / 78.8
    (4097, 63, 0, 0), (63, 4097, 0, 0),  # longer than the lines
    (1, 1, 0, 1), (1, 9, 0, 1), (9, 1, 0, 1),  # nothing to transform one way
]


# N, M, lines: relative errors of the analysis, 1e-16, by the lines and by hipFFT
ERRORS = [
    (25, 33, 0),    # 3.5 / 2.7
    (39, 51, 0),    # 4.3 / 3.0
    (64, 125, 0),   # 3.8 / 3.75
    (100, 105, 0),  # 4.7 / 3.9
    (85, 121, 0),   # 4.2 / 3.2
    (125, 231, 0),  # 4.0 / 4.3, synthesis 3.9 / 3.3
    (400, 625, 0),  # 4.6 / 4.3
    (500, 845, 0),  # 4.8 / 4.3
    (715, 825, 0),  # 4.8 / 4.5
    (867, 867, 0),  # 5.2 / 4.9
    (67, 133, 1),   # 3.7 / 7.8
    (24, 47, 1),    # 3.5 / 6.9
    (128, 231, 1),  # 3.6 / 4.8
    (256, 405, 1),  # 4.1 / 4.8
    (360, 539, 1),  # 4.1 / 5.6
    (512, 765, 1),  # 4.2 / 5.0
    (1000, 1215, 1),  # 4.6 / 5.2
]


@pytest.mark.parametrize("N,M,lines", ERRORS)
def test_rule_by_error(ft, N, M, lines):
    assert ft._lib.ftamd_grid_lines(N, M, 0) == lines


@pytest.mark.parametrize("N,M,disk,lines", SIZES)
def test_rule(ft, N, M, disk, lines):
    assert ft._lib.ftamd_grid_lines(N, M, disk) == lines


@pytest.mark.gpu
@pytest.mark.parametrize("which", ["sph_synthesis", "sphv_analysis", "annulus_synthesis", "disk_synthesis",
                                   "disk_analysis"])
def test_hipfft_and_shortest_grids(ft, which):
    import oracle as O
    import torch
    geo = which.split("_")[0]
    rho = 0.4 if geo == "annulus" else None
    for N, M in ((60, 119), (2187, 63), (2, 3), (1, 1), (1, 9), (2, 1)):
        assert ft._lib.ftamd_grid_lines(N, M, geo == "disk") == (N == 1 or M == 1)
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
