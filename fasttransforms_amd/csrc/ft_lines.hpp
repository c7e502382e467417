// ft_lines.hpp -- the interface of the line transforms (ft_dft.hpp) to the
// grid transforms (ft_grid.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "ft_hip_abi.h"

// Tables of a DFT of length len on the current device.  A length runs on
// these kernels where ftamd_dft_fits: up to FTAMD_DFT_MAX (the convolution's
// 2 FTAMD_DFT_MAX points are 139 KB of the 160 KB of LDS), powers of two from
// 64 up to twice that.
constexpr int FTAMD_DFT_MAX = 4096;
struct FtamdDft;
bool ftamd_dft_fits(int len);
int ftamd_dft_points(int len);  // of its power-of-two DFTs: len, or the convolution's
int ftamd_dft_create(int len, FtamdDft **out);
void ftamd_dft_destroy(FtamdDft *d);

// One launch over the theta lines (columns) or the phi lines (row pairs) of
// the N x M grid X (column-major), to or from the half spectra Y (N x
// (M/2+1) complex, column-major).
enum {
    FTAMD_LINES_THETA3 = 0,    // X to Y: fix-ups f0, f1, DCT-III / DST-III, weights, scalings a, b, data_r2c
    FTAMD_LINES_THETA2 = 1,    // Y to X: data_c2r, scalings, weights, DCT-II / DST-II, fix-ups
    FTAMD_LINES_PHI_BACK = 2,  // Y to X: c2r along the rows
    FTAMD_LINES_PHI_FWD = 3    // X to Y: r2c along the rows
};
struct FtamdLines {
    double *X;
    double2 *Y;
    const double2 *turn;       // e^{i pi k / 2N}, k < N (theta)
    const double *w;           // the annulus's weights, or NULL
    int kind, lines;           // FTAMD_LINES_*; M/2+1 orders (theta), (N+1)/2 row pairs (phi)
    int N, M;
    int plan_mode, exec_mode;  // column classes of the plan and of the executor
    int skip_sin;              // theta: leave the sine class alone
    int wmode;                 // weights: 0 none, 1 multiply, 2 divide
    int aligned;               // phi: N even and X 16-byte aligned
    double f0, f1, a, b;
    // set by ftamd_dft_lines
    int len;
    const double2 *tw, *filter, *chirp;
};
int ftamd_dft_lines(const FtamdDft *d, FtamdLines *a, void *stream);
// the launches of the convolution's instantiations (ft_dft_chirp.hip)
int ftamd_dft_launch_chirp(int logl, const FtamdLines &a, void *stream);
