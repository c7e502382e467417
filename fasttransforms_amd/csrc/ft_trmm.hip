// ft_trmm.hip -- the upper-triangular products of the harmonic transforms
// (drivers.c:833-1021: cblas_dtrmm from the left on the column classes
// j = c mod 4, or on every column, and from the right on every row) as one
// launch each on the FP64 matrix cores.
//
// Left: Y[:, j] = op(U_c) X[:, j] for every column j of every class c.
// Right: Y = X op(U) with U's leading M x M block.  Out of place.  A
// workgroup of 2 x 2 waves computes a tile of 32 rows x 32 columns of Y, a
// wave 16 x 16 of it by v_mfma_f64_16x16x4_f64 over k in stages of 16 through
// two LDS buffers, one barrier a stage.  Only the triangle's k range is
// visited.  Lane layout of the 16x16x4 FP64 MFMA: A operand lane i =
// A[i % 16][i / 16], B operand lane i = B[i / 16][i % 16], result register j
// of lane i = D[i / 16 + 4 j][i % 16].  The operand that runs along Y's
// columns is the A operand, so that 16 lanes hold 16 consecutive rows of one
// column of Y (a whole 128-byte line of the store).
//
// What bounds it: at n = 1024, M = 2047 the matrix pipes (30 us of 50 at the
// rate of a large product), below n = 600 the chain of stages of the longest
// tile, some 350 clocks each, of which the products take 256.  So a stage's
// loads are issued two stages ahead and without conditions: rows and columns
// past the edge are clamped (their results are not stored), addresses advance
// by one add, and the one stage that K cuts is left for the end.  One stage
// ahead and with bounds checked at each load it was 65 us, and at n = 511 19
// us for 11.6.  Held to 64 registers, so that eight waves share a SIMD (at 80
// it is 56 us).  Tiles of 64 x 32 and 64 x 64 make the chain longer (17 and 27
// us at n = 511) and are no faster at n = 1024 (49 .. 62 us).  Tiles are dealt
// longest first and back and forth over the 256 CUs, so that a CU's
// workgroups add up to equal work.  n = 1024, M = 2047: 74 us before (64 x 32
// tiles, loads one stage ahead), 50 now; n = 600, M = 1199: 34, 18.
// The products sum in another order than the reference's BLAS, so results
// agree to rounding, not bit for bit.
#include <hip/hip_runtime.h>

#include "ft_hip_abi.h"

namespace fttrmm {

typedef double v4d __attribute__((ext_vector_type(4)));

constexpr int TK = 16;             // k per stage
constexpr int TR = 32, TC = 32;    // rows and columns of a tile
constexpr int PAD = 2;             // LDS row padding (doubles): stores of 16 k x 4 columns spread over the banks
constexpr int NE = TR * TK / 256;  // elements of each operand that a thread stages

// Column tiles before each class, and all of them.
struct Tiles {
    int at[5];
};

// RIGHT, TRANS as above; SCALE: X's entries as the Chebyshev normalization
// (cheb_scale) leaves them.
template <bool RIGHT, bool TRANS, bool SCALE>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(8, 8))) trmm_kernel(FtamdTrmmLaunch a, int rtiles, Tiles ct) {
    __shared__ double sR[2][TK][TR + PAD];  // op(U) (left) or X (right): [k][row]
    __shared__ double sC[2][TK][TC + PAD];  // X (left) or op(U) (right): [k][column]
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int n = a.n, K = RIGHT ? a.M : n;
    // the tile: by decreasing length of its k range, every other run of 256 backwards
    int id = blockIdx.x;
    {
        const int total = gridDim.x, run = id & ~255, end = min(run + 256, total);
        if (id & 256) id = run + end - 1 - id;
    }
    const int ctiles = ct.at[4];
    int rt, cq;
    if (RIGHT) {
        const int rank = id / rtiles;
        rt = id - rank * rtiles;
        cq = TRANS ? rank : ctiles - 1 - rank;
    } else {
        const int rank = id / ctiles;
        cq = id - rank * ctiles;
        rt = TRANS ? rtiles - 1 - rank : rank;
    }
    int c = 0;
    while (c < 3 && cq >= ct.at[c + 1]) ++c;
    const double *U = a.U[c];
    if (U == nullptr) return;
    const int xcol = a.cstride;
    const int count = (a.M - c + xcol - 1) / xcol;  // columns of the class
    const int r0 = rt * TR, q0 = (cq - ct.at[c]) * TC;
    const int kbeg = RIGHT ? (TRANS ? q0 : 0) : (TRANS ? 0 : r0);
    const int kend = RIGHT ? (TRANS ? K : min(K, q0 + TC)) : (TRANS ? min(n, r0 + TR) : n);
    const int kfirst = kbeg / TK * TK;

    // element s of the thread: (row or column, k) in the stage and its address,
    // consecutive threads along the direction that is contiguous in memory
    constexpr bool RK = !RIGHT && TRANS;  // op(U) = U^T from the left: contiguous in k
    constexpr bool CK = !RIGHT || !TRANS; // X from the left, U from the right: contiguous in k
    const double *pr[NE], *pc[NE];
    int rr[NE], rk[NE], cc[NE], ck[NE];
#pragma unroll
    for (int s = 0; s < NE; ++s) {
        const int e = tid + 256 * s;
        rr[s] = RK ? e / TK : e % TR;
        rk[s] = RK ? e % TK : e / TR;
        cc[s] = CK ? e / TK : e % TC;
        ck[s] = CK ? e % TK : e / TC;
        const long long row = min(r0 + rr[s], n - 1), kr = kfirst + rk[s];
        const long long q = min(q0 + cc[s], count - 1), kc = kfirst + ck[s];
        pr[s] = RIGHT ? a.X + row + kr * n : TRANS ? U + kr + row * n : U + row + kr * n;
        pc[s] = RIGHT ? (TRANS ? U + q + kc * n : U + kc + q * n) : a.X + kc + (c + q * xcol) * n;
    }
    const long long stepr = RK ? TK : (long long)TK * n, stepc = CK ? TK : (long long)TK * n;
    // the normalization of X's entry (i, j)
    auto scaled = [&](double v, int i, int j) {
        if (!SCALE) return v;
        if (j == 0) v *= a.pre1;
        if (i == 0) v *= a.pre1;
        return v * a.pre2;
    };
    struct Stage {
        double r[NE], c[NE];
    };
    auto load = [&](Stage &v, bool advance) {  // and on to the next stage
#pragma unroll
        for (int s = 0; s < NE; ++s) v.r[s] = *pr[s];
#pragma unroll
        for (int s = 0; s < NE; ++s) v.c[s] = *pc[s];
        const long long ar = advance ? stepr : 0, ac = advance ? stepc : 0;
#pragma unroll
        for (int s = 0; s < NE; ++s) pr[s] += ar, pc[s] += ac;
    };
    auto store = [&](const Stage &v, int buf, int k0) {
#pragma unroll
        for (int s = 0; s < NE; ++s) sR[buf][rk[s]][rr[s]] = RIGHT ? scaled(v.r[s], r0 + rr[s], k0 + rk[s]) : v.r[s];
#pragma unroll
        for (int s = 0; s < NE; ++s)
            sC[buf][ck[s]][cc[s]] = RIGHT ? v.c[s] : scaled(v.c[s], k0 + ck[s], c + (q0 + cc[s]) * xcol);
    };

    const int wr = (w & 1) * 16 + (lane & 15), wc = (w >> 1) * 16 + (lane & 15), wk = lane >> 4;
    v4d acc = {0, 0, 0, 0};
    auto multiply = [&](int buf) {
#pragma unroll
        for (int ks = 0; ks < TK; ks += 4)
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64(sC[buf][ks + wk][wc], sR[buf][ks + wk][wr], acc, 0, 0, 0);
    };
    // Full stages kfirst + TK i, i < full, and a last one that K cuts.
    const int full = (min(kend, K / TK * TK) - kfirst + TK - 1) / TK, klast = kfirst + full * TK;
    Stage v0, v1;
    if (full > 0) {
        load(v0, full > 1);
        load(v1, full > 2);
        store(v0, 0, kfirst);
        __syncthreads();
        // stage i in buffer i % 2; the loads of stage i + 2 (past the end: of the
        // last one again) are issued before its products, those of stage i + 1,
        // issued a stage earlier, stored after them
        for (int i = 0; i < full; i += 2) {
            load(v0, i + 3 < full);
            multiply(0);
            store(v1, 1, kfirst + (i + 1) * TK);
            __syncthreads();
            if (i + 1 == full) break;
            load(v1, i + 4 < full);
            multiply(1);
            store(v0, 0, kfirst + (i + 2) * TK);
            __syncthreads();
        }
    }
    if (klast < kend) {  // zeros past K; the addresses stand at the last full stage
        const long long ar = full > 0 ? stepr : 0, ac = full > 0 ? stepc : 0;
#pragma unroll
        for (int s = 0; s < NE; ++s) {
            const bool in = klast + rk[s] < K;
            const double x = *(in ? pr[s] + ar : a.X);
            v0.r[s] = in ? x : 0.0;
        }
#pragma unroll
        for (int s = 0; s < NE; ++s) {
            const bool in = klast + ck[s] < K;
            const double x = *(in ? pc[s] + ac : a.X);
            v0.c[s] = in ? x : 0.0;
        }
        store(v0, 0, klast);
        __syncthreads();
        multiply(0);
    }
    const int r = r0 + wr;
    if (r >= n) return;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int q = q0 + (w >> 1) * 16 + wk + 4 * e;
        if (q >= count) continue;
        const int col = c + q * xcol;
        double v = acc[e];
        if (a.scale_out) {  // cheb_scale
            if (col == 0) v *= a.post1;
            if (r == 0) v *= a.post1;
            v *= a.post2;
        }
        a.Y[r + (long long)col * n] = v;
    }
}

__global__ void cheb_scale_kernel(double *A, int n, int M, double s1, double s2) {
    const long long total = (long long)n * M;
    for (long long e = blockIdx.x * (long long)blockDim.x + threadIdx.x; e < total;
         e += (long long)gridDim.x * blockDim.x) {
        const int i = (int)(e % n), j = (int)(e / n);
        double v = A[e];
        if (j == 0) v *= s1;
        if (i == 0) v *= s1;
        A[e] = v * s2;
    }
}

// The annulus's semi-classical <-> classical conversion on the columns j = 1,
// 2 mod 4 of the n x M matrix A (drivers.c:1073-1121 with banded_source.c:
// 381-422 for the bidiagonal factor): x <- R^{-1} x, R^{-T} x (solves) or
// R x, R^T x (products), R upper bidiagonal with diagonal d and
// superdiagonal u, products and differences rounded one at a time in the
// reference's order.  Columns q = 0 .. count-1 of the two classes are
// column 4 (q / 2) + 1 + q % 2.
__device__ inline double *bidiag_column(double *A, int n, int q) { return A + (4LL * (q >> 1) + 1 + (q & 1)) * n; }

// The solves are a recurrence: one thread per column walks it (R^{-T} from row
// 0 up, R^{-1} from row n-1 down).  The column streams through registers in
// chunks of CH rows (one 128-byte line) with the next chunk's loads in flight
// during this one's arithmetic, so the division chain is the critical path.
template <bool TRANS>
__global__ void __launch_bounds__(64) bidiag_solve_kernel(double *__restrict__ A, int n, int count,
                                                          const double *__restrict__ d, const double *__restrict__ u) {
#pragma clang fp contract(off)
    constexpr int CH = 16;
    constexpr bool ASC = TRANS;
    const int q = blockIdx.x * 64 + threadIdx.x;
    if (q >= count) return;
    double *x = bidiag_column(A, n, q);
    // row i's superdiagonal entry is u[i - 1] (R^T) or u[i] (R); the walk's first row has none.
    // u[-1] and u[n - 1] are in the caller's buffer (d[n - 1] and the padding entry).
    auto has_u = [&](int i) { return TRANS ? i > 0 : i + 1 < n; };
    // full chunks: rows b .. b + CH - 1 with b = c CH (ascending) or n - (c + 1) CH (descending)
    const int nfull = n / CH;
    auto base = [&](int c) { return ASC ? c * CH : n - (c + 1) * CH; };
    double cx[CH], cd[CH], cu[CH], nx[CH], nd[CH], nu[CH];
    auto load = [&](int b, double *vx, double *vd, double *vu) {
#pragma unroll
        for (int k = 0; k < CH; ++k) {
            vx[k] = x[b + k];
            vd[k] = d[b + k];
            vu[k] = u[TRANS ? b + k - 1 : b + k];
        }
    };
    if (nfull > 0) load(base(0), cx, cd, cu);
    double carry = 0.0;  // the last new entry
    for (int c = 0; c < nfull; ++c) {
        const int b = base(c);
        load(c + 1 < nfull ? base(c + 1) : b, nx, nd, nu);
#pragma unroll
        for (int kk = 0; kk < CH; ++kk) {
            const int k = ASC ? kk : CH - 1 - kk;
            const int i = b + k;
            carry = (cx[k] - (has_u(i) ? cu[k] * carry : 0.0)) / cd[k];
            x[i] = carry;
        }
#pragma unroll
        for (int k = 0; k < CH; ++k) {
            cx[k] = nx[k];
            cd[k] = nd[k];
            cu[k] = nu[k];
        }
    }
    // the remaining n mod CH rows (ascending: the last ones, descending: the first ones)
    const int rem = n - nfull * CH;
    if (rem == 0) return;
    const int b = ASC ? nfull * CH : 0;
#pragma unroll
    for (int k = 0; k < CH; ++k) {
        const bool in = k < rem;
        cx[k] = in ? x[b + k] : 0.0;
        cd[k] = in ? d[b + k] : 1.0;
        cu[k] = in && has_u(b + k) ? u[TRANS ? b + k - 1 : b + k] : 0.0;
    }
#pragma unroll
    for (int kk = 0; kk < CH; ++kk) {
        const int k = ASC ? kk : CH - 1 - kk;
        if (k >= rem) continue;
        const int i = b + k;
        carry = (cx[k] - (has_u(i) ? cu[k] * carry : 0.0)) / cd[k];
        x[i] = carry;
    }
}

// The products have no recurrence: one wave per column, lane l on row r0 + l
// of each 64-row segment (coalesced 512-byte accesses), its neighbour from
// the next lane (R: x_{i+1}) or the previous one (R^T: x_{i-1}), the segment
// edge's from memory.  Segments run in the order that reads every neighbour
// before its own segment overwrites it: upward for R, downward for R^T.
template <bool TRANS>
__global__ void __launch_bounds__(256) bidiag_mul_kernel(double *A, int n, int count, const double *d,
                                                        const double *u) {
#pragma clang fp contract(off)
    const int q = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (q >= count) return;  // whole waves
    double *x = bidiag_column(A, n, q);
    const int nseg = (n + 63) / 64;
    for (int s = 0; s < nseg; ++s) {
        const int r0 = (TRANS ? nseg - 1 - s : s) * 64, i = r0 + lane;
        const bool in = i < n;
        const double xi = in ? x[i] : 0.0;
        double y;
        if (!TRANS) {  // x_i = d_i x_i + u_i x_{i+1}
            const double edge = r0 + 64 < n ? x[r0 + 64] : 0.0;
            const double nb = __shfl_down(xi, 1, 64);
            const double xn = lane == 63 ? edge : nb;
            y = in ? (i + 1 < n ? d[i] * xi + u[i] * xn : d[i] * xi) : 0.0;
        } else {  // x_i = u_{i-1} x_{i-1} + d_i x_i
            const double edge = r0 > 0 ? x[r0 - 1] : 0.0;
            const double nb = __shfl_up(xi, 1, 64);
            const double xp = lane == 0 ? edge : nb;
            y = in ? (i > 0 ? u[i - 1] * xp + d[i] * xi : d[i] * xi) : 0.0;
        }
        if (in) x[i] = y;
    }
}

}  // namespace fttrmm

extern "C" int ftamd_hip_bidiag(double *A, int n, int M, const double *R, int solve, int trans, void *stream) {
    if (n < 1 || M < 0 || !A || !R) return FTAMD_EINVAL;
    const int count = M / 4 * 2 + (M % 4 >= 2 ? 1 : 0) + (M % 4 >= 3 ? 1 : 0);  // columns j < M, j = 1, 2 mod 4
    if (count == 0) return FTAMD_OK;
    hipStream_t st = (hipStream_t)stream;
    const double *d = R, *u = R + n;
    const dim3 sgrid((count + 63) / 64), sblock(64);  // a thread per column
    const dim3 mgrid((count + 3) / 4), mblock(256);   // a wave per column
    if (solve && trans) hipLaunchKernelGGL(fttrmm::bidiag_solve_kernel<true>, sgrid, sblock, 0, st, A, n, count, d, u);
    else if (solve) hipLaunchKernelGGL(fttrmm::bidiag_solve_kernel<false>, sgrid, sblock, 0, st, A, n, count, d, u);
    else if (trans) hipLaunchKernelGGL(fttrmm::bidiag_mul_kernel<true>, mgrid, mblock, 0, st, A, n, count, d, u);
    else hipLaunchKernelGGL(fttrmm::bidiag_mul_kernel<false>, mgrid, mblock, 0, st, A, n, count, d, u);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? FTAMD_OK : FTAMD_EDEVICE;
}

namespace {

template <bool RIGHT, bool TRANS, bool SCALE> void launch(const FtamdTrmmLaunch &a, hipStream_t st) {
    using namespace fttrmm;
    Tiles ct;
    ct.at[0] = 0;
    for (int c = 0; c < 4; ++c) {
        const int count = c < a.ncls && a.M > c ? (a.M - c + a.cstride - 1) / a.cstride : 0;
        ct.at[c + 1] = ct.at[c] + (count + TC - 1) / TC;
    }
    const int rtiles = (a.n + TR - 1) / TR;
    hipLaunchKernelGGL((trmm_kernel<RIGHT, TRANS, SCALE>), dim3(ct.at[4] * rtiles), dim3(256), 0, st, a, rtiles, ct);
}

template <bool RIGHT> void launch_side(const FtamdTrmmLaunch &a, hipStream_t st) {
    if (a.trans) a.scale_in ? launch<RIGHT, true, true>(a, st) : launch<RIGHT, true, false>(a, st);
    else a.scale_in ? launch<RIGHT, false, true>(a, st) : launch<RIGHT, false, false>(a, st);
}

}  // namespace

extern "C" int ftamd_hip_trmm_launch(const FtamdTrmmLaunch *a, void *stream) {
    if (a->n < 1 || a->M < 0 || a->cstride < 1 || a->ncls < 1 || a->ncls > 4 || !a->X || !a->Y) return FTAMD_EINVAL;
    if (a->right && (a->ncls != 1 || a->cstride != 1 || a->M > a->n)) return FTAMD_EINVAL;
    if (a->M == 0) return FTAMD_OK;
    if (a->right) launch_side<true>(*a, (hipStream_t)stream);
    else launch_side<false>(*a, (hipStream_t)stream);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? FTAMD_OK : (e == hipErrorOutOfMemory ? FTAMD_ENOMEM : FTAMD_EDEVICE);
}

extern "C" int ftamd_hip_cheb_scale(double *A, int n, int M, double s1, double s2, void *stream) {
    if (n < 1 || M < 0 || !A) return FTAMD_EINVAL;
    if (M == 0) return FTAMD_OK;
    const long long total = (long long)n * M;
    const long long want = (total + 255) / 256;
    const int blocks = (int)(want < 4096 ? want : 4096);
    hipLaunchKernelGGL(fttrmm::cheb_scale_kernel, dim3(blocks), dim3(256), 0, (hipStream_t)stream, A, n, M, s1, s2);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? FTAMD_OK : FTAMD_EDEVICE;
}
