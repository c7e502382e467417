// ft_k_spin.hip -- first stage of the spin-weighted sphere's rotations
// (rotations_default.c:87-117, the loops over s2, c2): for a complex column
// of order m and spin s (am = |m|, as = |s|, d = |am - as|), the sequences
// j = min(am, as)-1 .. 0 of rotations of adjacent rows (k, k+1),
// k = n-2-d-j .. 0, with s2(k, j, d), c2(k, j, d) -- the rotation where
// m*s >= 0 and its transpose otherwise (hi2lo); lo2hi runs the transposes in
// the opposite order.  The real and imaginary parts take the same real
// rotation.
//
// A wave owns four columns and takes up to four of their sequences at a time:
// a lane for each sequence and real or imaginary part, which sweeps down
// (hi2lo) or up (lo2hi) the column in blocks of 16 rows, a step rotating the
// fresh row against the carried one and emitting a finished row.  A
// sequence's lane is a block behind the one before it and takes the rows that
// this one emitted from LDS.  All 64 lanes move data: a block is one 16-byte
// load a lane of rows and one of (s, c) for each sequence, two blocks ahead,
// passed on through LDS, and one store.
//
// What bounds it: the instructions of a step (four FP64, two LDS reads),
// issued in order by the one wave of a SIMD.  Loads by the computing lanes
// themselves (32 columns a wave, each lane its own line, one block of 12 rows
// ahead, one sequence a sweep) took 146 clocks a step and sequence, waiting
// for memory; two sequences in one lane take 26 us.  n = 512, s = 2: 68 us
// before, 22 now.
//
// The transpose of the rotation (s, c) is the rotation (-s, c), bit for bit
// in the fused forms: fma(c, x, (-s)*y) = fma(c, x, -(s*y)) and
// fma(c, y, -((-s)*x)) = fma(c, y, s*x), since negation is exact.  So every
// rotation here is X' = fma(c, x, t*y), Y' = fma(c, y, -(t*x)) with t = +-s.
#include <hip/hip_runtime.h>

#include "ft_hip_abi.h"

namespace ftspin {

__device__ __forceinline__ double rot_x(double C, double S, double x, double y) { return __builtin_fma(C, x, S * y); }
__device__ __forceinline__ double rot_y(double C, double S, double x, double y) { return __builtin_fma(C, y, -(S * x)); }

constexpr int CW = 4;   // columns of a wave
constexpr int KB = 16;  // elements of a block
constexpr int PITCH = KB + 1;
constexpr int MAXS = 4;  // most sequences at a time

struct Column {
    int R;            // last row of sequence 0
    int nrot;         // its sequences; 0 past the last column
    long long base;   // its row 0 (complex entries from A)
    long long tab;    // sequence 0's (s, c)
    double sg;        // sign of s
};

struct Args {
    const double2 *tab;
    int n, s;
    double2 *A;
    int c0, count;
    long long col_stride;
    int row_stride, use_fixed, fixed_m, dir;
    int nlow, low_blocks;  // the first nlow columns have waves of their own, low_blocks of them
};

// The wave's column of a slot.  The first nlow columns are of orders |m| < |s|,
// with |m| sequences: wave k - 1 takes orders -k and k.
__device__ Column column(const Args &a, int slot) {
    int c;
    bool in;
    if ((int)blockIdx.x < a.low_blocks) {
        c = 2 * (int)blockIdx.x + 1 + slot;
        in = slot < 2 && c >= a.c0 && c < a.c0 + a.nlow;
    } else {
        c = a.c0 + a.nlow + ((int)blockIdx.x - a.low_blocks) * CW + slot;
        in = c < a.c0 + a.count;
    }
    if (!in) c = a.c0;
    const int m = a.use_fixed ? a.fixed_m : ((c & 1) ? -((c + 1) >> 1) : (c >> 1));
    const int as = a.s < 0 ? -a.s : a.s, am = m < 0 ? -m : m;
    const int d = am > as ? am - as : as - am;
    const int nseq = am < as ? am : as;
    Column q;
    q.R = a.n - 1 - d;
    q.nrot = in ? max(0, min(nseq, q.R)) : 0;
    q.base = a.col_stride * (c - a.c0);
    q.tab = (long long)d * as * a.n;
    q.sg = (a.dir == 0) == ((m >= 0) == (a.s >= 0)) ? 1.0 : -1.0;
    return q;
}

__device__ int wave_max(int v) {
    for (int k = 32; k; k >>= 1) v = max(v, __shfl_xor(v, k));
    return __builtin_amdgcn_readfirstlane(v);
}

struct Shared {
    double2 rows[MAXS + 1][CW * PITCH];  // [s]: the rows that stage s takes, [s + 1]: those it emitted
    double2 sc[MAXS][CW * PITCH];
};

// The sequences jl .. jl + S - 1 over the wave's columns: lq the column whose
// data this lane moves, cq the one it computes on.  Stage st is sequence jl +
// S - 1 - st (hi2lo) or jl + st (lo2hi).  Element t of a column is row RL - t
// (t), RL the last row of sequence jl: a stage takes element t and emits
// element t - 1, rotated by the sequence's pair RL - t (t - 1) if it has that,
// else as it is; so nothing but t tells the first and the last steps apart.
// In round g stage st takes elements 16 (g - st) - st and up.
template <int DIR, int S>
__device__ void sweep(const Args &a, const Column &lq, const Column &cq, int jl, Shared &sh) {
    const int lane = threadIdx.x, lcol = lane / KB, lk = lane % KB;
    const int h = lane & 1, ccol = (lane >> 1) & (CW - 1), st = lane / (2 * CW);
    const bool lvalid = jl < lq.nrot, cvalid = jl < cq.nrot;
    const int RL = lvalid ? lq.R - jl : 0, RC = cvalid ? cq.R - jl : 0;
    const int rounds = (wave_max(RC) + S) / KB + S;
    const int full = -wave_max(cvalid ? -RC : -(1 << 30));  // every column has elements up to here
    const int act0 = DIR == 0 ? S - st : 1, act1 = DIR == 0 ? RC : RC - st;
    const double2 *lt = a.tab + (lvalid ? lq.tab + (long long)jl * a.n : 0);
    double2 *lA = a.A + lq.base;
    struct Block {
        double2 x, sc[S];
    };
    auto load = [&](Block &v, int g) {
        const int t = max(0, min(g * KB + lk, RL));
        v.x = lA[(long long)(DIR == 0 ? RL - t : t) * a.row_stride];
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const int j = lvalid ? (DIR == 0 ? S - 1 - s : s) : 0, ts = (g - s) * KB - s + lk;
            const int pair = DIR == 0 ? RL - ts : ts - 1;
            v.sc[s] = lt[(long long)j * a.n + max(0, min(pair, RL - j - 1))];
        }
    };
    // in this order, so that a wait for one block's loads is none for the next one's
    Block v0, v1;
    __builtin_amdgcn_sched_barrier(0);
    load(v0, 0);
    __builtin_amdgcn_sched_barrier(0);
    load(v1, 1);
    __builtin_amdgcn_sched_barrier(0);

    double cy = 0.0;
    auto rotate = [&](double2 sc, double x) {
        double em;
        if (DIR == 0) {  // x row r, the carried row r + 1, emits row r + 1
            em = rot_y(sc.y, sc.x, x, cy);
            cy = rot_x(sc.y, sc.x, x, cy);
        } else {  // the carried row r, x row r + 1, emits row r
            em = rot_x(sc.y, sc.x, cy, x);
            cy = rot_y(sc.y, sc.x, cy, x);
        }
        return em;
    };
    auto round = [&](int g, Block &v) {
        sh.rows[0][lcol * PITCH + lk] = v.x;
#pragma unroll
        for (int s = 0; s < S; ++s) sh.sc[s][lcol * PITCH + lk] = make_double2(lq.sg * v.sc[s].x, v.sc[s].y);
        load(v, g + 2);
        __syncthreads();
        if (lane < 2 * CW * S) {
            const double2 *in = &sh.rows[st][ccol * PITCH], *csc = &sh.sc[st][ccol * PITCH];
            double *out = (double *)&sh.rows[st + 1][ccol * PITCH] + h;
            double x[KB];
            double2 sc[KB];
#pragma unroll
            for (int k = 0; k < KB; ++k) {
                x[k] = ((const double *)&in[k])[h];
                sc[k] = csc[k];
            }
            if (g >= S && g * KB + KB - 1 <= full) {
#pragma unroll
                for (int k = 0; k < KB; ++k) out[2 * k] = rotate(sc[k], x[k]);
            } else {
                const int t0 = (g - st) * KB - st;
#pragma unroll
                for (int k = 0; k < KB; ++k) {
                    const bool act = t0 + k >= act0 && t0 + k <= act1;
                    const double c0 = cy, em = rotate(sc[k], x[k]);
                    if (!act) cy = x[k];
                    out[2 * k] = act ? em : c0;
                }
            }
        }
        __syncthreads();
        const int t = (g - S + 1) * KB - S + lk;
        if (lvalid && t >= 0 && t <= RL)
            lA[(long long)(DIR == 0 ? RL - t : t) * a.row_stride] = sh.rows[S][lcol * PITCH + lk];
    };
    int g = 0;  // (the odd round out of the loop: a branch in it costs 2 % at n = 512)
    for (; g + 1 < rounds; g += 2) {
        round(g, v0);
        round(g + 1, v1);
    }
    if (g < rounds) round(g, v0);
    __threadfence_block();  // the next sweep's loads take rows that other lanes stored
    __syncthreads();
}

template <int DIR> __global__ void __launch_bounds__(64) stage1_kernel(Args a) {
    __shared__ Shared sh;
    const int lane = threadIdx.x;
    const Column lq = column(a, lane / KB), cq = column(a, (lane >> 1) & (CW - 1));
    const int most = wave_max(cq.nrot), least = -wave_max(cq.nrot > 0 ? -cq.nrot : -(1 << 30));
    // several sequences at a time where the columns have the same number of them
    const int fours = most == least ? most / 4 : 0, twos = most == least ? (most - 4 * fours) / 2 : 0;
    const int single = 4 * fours + 2 * twos;
    if (DIR == 0) {
        for (int j = most - 1; j >= single; --j) sweep<0, 1>(a, lq, cq, j, sh);
        if (twos) sweep<0, 2>(a, lq, cq, 4 * fours, sh);
        for (int j = fours - 1; j >= 0; --j) sweep<0, 4>(a, lq, cq, 4 * j, sh);
    } else {
        for (int j = 0; j < fours; ++j) sweep<1, 4>(a, lq, cq, 4 * j, sh);
        if (twos) sweep<1, 2>(a, lq, cq, 4 * fours, sh);
        for (int j = single; j < most; ++j) sweep<1, 1>(a, lq, cq, j, sh);
    }
}

}  // namespace ftspin

extern "C" int ftamd_hip_spin_stage1(const double *tab2, int n, int s, double *A, int c0, int count,
                                     long long col_stride, int row_stride, int use_fixed, int fixed_m, int dir,
                                     void *stream) {
    if (!A || n < 1 || c0 < 0 || count < 0 || row_stride < 1 || col_stride < 0 || (dir != 0 && dir != 1))
        return FTAMD_EINVAL;
    if (count == 0 || s == 0) return FTAMD_OK;
    if (!tab2) return FTAMD_EINVAL;
    if (count > (1 << 29)) return FTAMD_EINVAL;
    const int as = s < 0 ? -s : s;
    // columns of orders |m| < |s|, c < 2 |s| - 1, have |m| sequences, the others |s|
    const long long low = use_fixed ? 0 : 2LL * as - 1 - c0;
    ftspin::Args a;
    a.tab = (const double2 *)tab2;
    a.n = n;
    a.s = s;
    a.A = (double2 *)A;
    a.c0 = c0;
    a.count = count;
    a.col_stride = col_stride;
    a.row_stride = row_stride;
    a.use_fixed = use_fixed;
    a.fixed_m = fixed_m;
    a.dir = dir;
    a.nlow = low < 0 ? 0 : low < count ? (int)low : count;
    a.low_blocks = a.nlow > 0 ? (c0 + a.nlow) / 2 : 0;  // orders 1 .. that of the last of them
    const int blocks = a.low_blocks + (count - a.nlow + ftspin::CW - 1) / ftspin::CW;
    if (blocks == 0) return FTAMD_OK;  // order 0 alone
    const dim3 grid(blocks), block(64);
    if (dir == 0) hipLaunchKernelGGL(ftspin::stage1_kernel<0>, grid, block, 0, (hipStream_t)stream, a);
    else hipLaunchKernelGGL(ftspin::stage1_kernel<1>, grid, block, 0, (hipStream_t)stream, a);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? FTAMD_OK : FTAMD_EDEVICE;
}
