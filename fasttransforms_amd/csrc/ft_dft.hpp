// ft_dft.hpp -- the DFT of one line in LDS, and the grid transforms built on
// it (ft_dft.hip): the theta transforms of the sphere's, the vector field's
// and the annulus's grids and the phi transforms of those and of the disk's
// (fftw.c:62-270, 400-655), each one kernel that reads its lines from memory,
// transforms them in LDS and writes the result with the fix-ups, scalings and
// layouts of the executors folded in.
//
// A DFT of length len is computed directly where len is a power of two, else
// as a convolution (Bluestein's chirp transform: jk = (j^2 + k^2 - (j-k)^2)/2)
// through DFTs of a power of two L >= 2 len - 1.  A DFT of length L = 2^LOGL
// takes L/16 threads with 16 points each in registers: decimation in
// frequency by radices 16, 16, .. and what is left, exchanged through LDS
// between the passes, from natural order into digit-reversed order; the
// convolution multiplies by its filter there (stored in that order) and runs
// the passes backwards, so nothing is ever reordered.  Twiddles come from
// tables (rounded from long double once, [r-1][o] per pass, so that a wave
// reads consecutive entries).
#pragma once

#include <hip/hip_runtime.h>

#include "ft_lines.hpp"

namespace ftdft {

__device__ __forceinline__ double2 add(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ double2 sub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ double2 conj(double2 a) { return make_double2(a.x, -a.y); }
__device__ __forceinline__ double2 mul(double2 a, double2 b) {
    return make_double2(__builtin_fma(a.x, b.x, -(a.y * b.y)), __builtin_fma(a.x, b.y, a.y * b.x));
}
// a * conj(b)
__device__ __forceinline__ double2 mulc(double2 a, double2 b) {
    return make_double2(__builtin_fma(a.x, b.x, a.y * b.y), __builtin_fma(a.y, b.x, -(a.x * b.y)));
}
// a * (-i), a * i: the forward and the backward transform's quarter turn
template <bool INV> __device__ __forceinline__ double2 quarter(double2 a) {
    return INV ? make_double2(-a.y, a.x) : make_double2(a.y, -a.x);
}

// DFTs of the R entries x[0], x[ST], x[2 ST], .. in natural order (INV: the
// conjugate roots)
template <int R, bool INV, int ST> struct Small;
template <bool INV, int ST> struct Small<1, INV, ST> {
    __device__ static void run(double2 *) {}
};
template <bool INV, int ST> struct Small<2, INV, ST> {
    __device__ static void run(double2 *x) {
        const double2 a = x[0], b = x[ST];
        x[0] = add(a, b);
        x[ST] = sub(a, b);
    }
};
template <bool INV, int ST> struct Small<4, INV, ST> {
    __device__ static void run(double2 *x) {
        const double2 a = add(x[0], x[2 * ST]), b = sub(x[0], x[2 * ST]), c = add(x[ST], x[3 * ST]),
                      d = quarter<INV>(sub(x[ST], x[3 * ST]));
        x[0] = add(a, c);
        x[ST] = add(b, d);
        x[2 * ST] = sub(a, c);
        x[3 * ST] = sub(b, d);
    }
};
constexpr double kC8 = 0.70710678118654752440;   // cos(pi/4)
constexpr double kC16 = 0.92387953251128675613;  // cos(pi/8)
constexpr double kS16 = 0.38268343236508977173;  // sin(pi/8)
// x * e^{-2 pi i k / 16} (INV: the conjugate)
template <int K, bool INV> __device__ __forceinline__ double2 root16(double2 a) {
    static_assert(K == 1 || K == 2 || K == 3 || K == 4 || K == 6 || K == 9, "the roots 2 x 4 and 4 x 4 splits need");
    if constexpr (K == 4) {
        return quarter<INV>(a);
    } else if constexpr (K == 2 || K == 6) {
        const double2 q = quarter<INV>(a);
        return K == 2 ? make_double2(kC8 * (a.x + q.x), kC8 * (a.y + q.y)) : make_double2(kC8 * (q.x - a.x), kC8 * (q.y - a.y));
    } else {
        constexpr double c = K == 1 ? kC16 : K == 3 ? kS16 : -kC16, s = K == 1 ? kS16 : K == 3 ? kC16 : -kS16;
        return mul(a, make_double2(c, INV ? s : -s));
    }
}
template <bool INV, int ST> struct Small<8, INV, ST> {
    __device__ static void run(double2 *x) {
        // 2 x 4: even and odd entries
        Small<4, INV, 2 * ST>::run(x);
        Small<4, INV, 2 * ST>::run(x + ST);
        const double2 e0 = x[0], e1 = x[2 * ST], e2 = x[4 * ST], e3 = x[6 * ST];
        const double2 o0 = x[ST], o1 = root16<2, INV>(x[3 * ST]), o2 = root16<4, INV>(x[5 * ST]),
                      o3 = root16<6, INV>(x[7 * ST]);
        x[0] = add(e0, o0);
        x[4 * ST] = sub(e0, o0);
        x[ST] = add(e1, o1);
        x[5 * ST] = sub(e1, o1);
        x[2 * ST] = add(e2, o2);
        x[6 * ST] = sub(e2, o2);
        x[3 * ST] = add(e3, o3);
        x[7 * ST] = sub(e3, o3);
    }
};
template <bool INV, int ST> struct Small<16, INV, ST> {
    __device__ static void run(double2 *x) {
        // 4 x 4: DFTs over the entries of each residue mod 4, roots, DFTs across
#pragma unroll
        for (int a = 0; a < 4; ++a) Small<4, INV, 4 * ST>::run(x + a * ST);
        // x[(a + 4 k) ST]: residue a, frequency k
        x[5 * ST] = root16<1, INV>(x[5 * ST]);
        x[9 * ST] = root16<2, INV>(x[9 * ST]);
        x[13 * ST] = root16<3, INV>(x[13 * ST]);
        x[6 * ST] = root16<2, INV>(x[6 * ST]);
        x[10 * ST] = root16<4, INV>(x[10 * ST]);
        x[14 * ST] = root16<6, INV>(x[14 * ST]);
        x[7 * ST] = root16<3, INV>(x[7 * ST]);
        x[11 * ST] = root16<6, INV>(x[11 * ST]);
        x[15 * ST] = root16<9, INV>(x[15 * ST]);
#pragma unroll
        for (int k = 0; k < 4; ++k) Small<4, INV, ST>::run(x + 4 * k * ST);
        // frequency k + 4 l is at (4 k + l) ST: transpose
#pragma unroll
        for (int k = 0; k < 4; ++k)
#pragma unroll
            for (int l = 0; l < k; ++l) {
                const double2 t = x[(4 * k + l) * ST];
                x[(4 * k + l) * ST] = x[(4 * l + k) * ST];
                x[(4 * l + k) * ST] = t;
            }
    }
};

// The passes of a DFT of length 2^LOGL (4 <= LOGL <= 13).
template <int LOGL> struct Shape {
    // 16 points a thread (8, with a pass more and twice the waves: phi at L = 4096
    // 39 us against 28, theta the same)
    static constexpr int LOGE = 4, EP = 1 << LOGE;
    static constexpr int L = 1 << LOGL, NT = L / EP;            // points, threads
    static constexpr int NP = (LOGL + LOGE - 1) / LOGE;         // passes: radix EP, the last what is left
    static constexpr int radix(int p) { return p < LOGL / LOGE ? EP : 1 << (LOGL % LOGE); }
    static constexpr int block(int p) { return p == 0 ? L : block(p - 1) / radix(p - 1); }  // points of a pass's blocks
    static constexpr int sub(int p) { return block(p) / radix(p); }
    // where pass p's twiddles start in the table: (R - 1) * sub entries each
    static constexpr int tw_off(int p) { return p == 0 ? 0 : tw_off(p - 1) + (radix(p - 1) - 1) * sub(p - 1); }
    // transforms of a workgroup of at least one wave
    static constexpr int PER = NT >= 64 ? 1 : 64 / NT;
    static constexpr int THREADS = NT * PER;
    // LDS slot of point i: padded so that the last pass's strided accesses spread over the banks
    __host__ __device__ static constexpr int slot(int i) { return i + i / EP; }
    static constexpr int SLOTS = L + L / EP;
};

template <int LOGL> struct Dft {
    using S = Shape<LOGL>;

    // point of thread t's register e in pass P
    template <int P> __host__ __device__ static int point(int t, int e) {
        constexpr int R = S::radix(P), sub = S::sub(P);
        // the last pass's smaller butterflies: a thread's are consecutive
        const int u = R == S::EP ? t : t * (S::EP / R) + e / R, r = e % R;
        return u / sub * S::block(P) + u % sub + r * sub;
    }
    template <int P> __device__ static void put(double2 *lds, int t, const double2 (&x)[S::EP]) {
#pragma unroll
        for (int e = 0; e < S::EP; ++e) lds[S::slot(point<P>(t, e))] = x[e];
    }
    template <int P> __device__ static void get(const double2 *lds, int t, double2 (&x)[S::EP]) {
#pragma unroll
        for (int e = 0; e < S::EP; ++e) x[e] = lds[S::slot(point<P>(t, e))];
    }
    template <int P, bool INV> __device__ static void twiddle(const double2 *__restrict__ tw, int t, double2 (&x)[S::EP]) {
        constexpr int R = S::radix(P), sub = S::sub(P);
        if (sub == 1) return;
#pragma unroll
        for (int e = 0; e < S::EP; ++e) {
            const int r = e % R;
            if (r == 0) continue;
            const int o = t % sub;
            const double2 w = tw[S::tw_off(P) + (r - 1) * sub + o];
            x[e] = INV ? mulc(x[e], w) : mul(x[e], w);
        }
    }
    template <int P, bool INV> __device__ static void butterflies(double2 (&x)[S::EP]) {
        constexpr int R = S::radix(P);
#pragma unroll
        for (int v = 0; v < S::EP / R; ++v) Small<R, INV, 1>::run(x + v * R);
    }
    // Between the write and the read of an exchange of passes P and P + 1.  The
    // exchange stays within the threads of a block of pass P; within a wave
    // LDS runs in order.  (Nothing is awaited before a write: a thread writes
    // the points it read last, or the caller has waited.)
    template <int P> __device__ static void exchanged() {
        if constexpr (S::NT > 64 && S::block(P) / S::EP > 64) {
            __syncthreads();
        } else {
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        }
    }
    // passes P .. NP-1 forward: x holds pass P's points of the natural order;
    // afterwards the last pass's points, digit-reversed
    template <int P> __device__ static void forward(double2 *lds, const double2 *__restrict__ tw, int t, double2 (&x)[S::EP]) {
        butterflies<P, false>(x);
        if constexpr (P + 1 < S::NP) {
            twiddle<P, false>(tw, t, x);
            put<P>(lds, t, x);
            exchanged<P>();
            get<P + 1>(lds, t, x);
            forward<P + 1>(lds, tw, t, x);
        }
    }
    // passes P .. 0 backward (unnormalized), undoing forward
    template <int P> __device__ static void backward(double2 *lds, const double2 *__restrict__ tw, int t, double2 (&x)[S::EP]) {
        twiddle<P, true>(tw, t, x);
        butterflies<P, true>(x);
        if constexpr (P > 0) {
            put<P>(lds, t, x);
            exchanged<P - 1>();
            get<P - 1>(lds, t, x);
            backward<P - 1>(lds, tw, t, x);
        }
    }
    // frequency the last pass leaves at point i: the digits of i, each pass's
    // the next lower ones of the point and the next higher of the frequency
    __host__ __device__ static int frequency(int i) {
        int f = 0, unit = 1;
#pragma unroll
        for (int p = 0; p < S::NP; ++p) {
            f += i / S::sub(p) % S::radix(p) * unit;
            unit *= S::radix(p);
        }
        return f;
    }
};


// Columns of the cosine class (fftw.c:84-96): j mod 4 in {0, 3}, that is both
// columns 2q-1 and 2q of an even order q; the vector-field plans (mode 1) swap
// the classes, the annulus's (mode 3, fftw.c:560-575) have one.
__device__ __forceinline__ bool cos_order(int q, int mode) { return mode == 3 || ((q & 1) == 0) != (mode == 1); }

// One launch: a transform of every line (FtamdLines, ft_lines.hpp).
//
// The theta lines are orders q: columns 2q-1 and 2q of X (column 0 alone for
// q = 0) are one complex line x_{2q} + i x_{2q-1} (the transforms are linear,
// and both columns take the same one), which is the half spectrum of
// data_r2c (fftw.c:40-49) conjugated.  The phi lines are pairs of rows 2p, 2p+1
// (the last one alone for odd N), one complex line whose spectrum holds both
// rows' half spectra.
//
// What bounds it: at L = 4096 a line is 68 KB of LDS, two workgroups a CU, and
// the passes (1800 FP64 instructions a thread and four exchanges, an LDS write
// of 16 bytes a lane taking 13 clocks of the CU) take 10 of a phi launch's 28
// us at n = 1024 (1024 x 2047), the rows' 16-byte pieces and the launch the
// rest; theta (18 us) is its 34 MB and the launch.  At L = 8192
// one workgroup is on a CU, 0.09 us a phi line and 0.16 a theta line (which
// ftamd_grid_lines counts in).  Memory is read and written once.  Workgroups go to XCDs in contiguous runs of lines, so that the
// 128-byte lines of memory that 4 to 8 neighbouring rows share stay in one L2.
template <int LOGL, bool CHIRP>
__global__ void __launch_bounds__(Shape<LOGL>::THREADS) lines_kernel(FtamdLines a) {
    using S = Shape<LOGL>;
    using D = Dft<LOGL>;
    __shared__ double2 lds_all[S::SLOTS * S::PER];
    // (one line a workgroup: the line's base addresses are scalars)
    const int t = S::PER == 1 ? threadIdx.x : threadIdx.x % S::NT, own = S::PER == 1 ? 0 : threadIdx.x / S::NT;
    const int chunk = gridDim.x / 8;
    const int line = ((int)(blockIdx.x % 8) * chunk + (int)(blockIdx.x / 8)) * S::PER + own;
    double2 *lds = lds_all + own * S::SLOTS;
    const int N = a.N, M = a.M, len = a.len;
    const int q = line;
    const bool tcos = cos_order(q, a.plan_mode), fcos = cos_order(q, a.exec_mode);
    const bool theta = a.kind <= FTAMD_LINES_THETA2;
    const bool on = line < a.lines && !(theta && a.skip_sin && !tcos);
    // Entries a thread has: all 16, or of a convolution (len <= L/2) the first 8.
    // Reads past the line are clamped to its last entry and dropped, and reads
    // come before anything that depends on them, so that no branch keeps a
    // thread's loads from being in flight together.
    constexpr int E = CHIRP ? S::EP / 2 : S::EP;
    // a column pair's weights (the annulus's, fftw.c:588-592) on the rows row(e)
    auto weigh = [&](double2 (&v)[S::EP], auto row) {
        if (a.wmode == 0 || (q & 1) == 0) return;
        double w[E];
#pragma unroll
        for (int e = 0; e < E; ++e) w[e] = a.w[row(e)];
#pragma unroll
        for (int e = 0; e < E; ++e)
            v[e] = a.wmode == 1 ? make_double2(v[e].x * w[e], v[e].y * w[e]) : make_double2(v[e].x / w[e], v[e].y / w[e]);
    };
    double2 x[S::EP];
#pragma unroll
    for (int e = 0; e < S::EP; ++e) x[e] = make_double2(0.0, 0.0);
    auto entry = [&](int e) { return t + S::NT * e; };
    auto within = [&](int k) { return CHIRP ? min(k, len - 1) : k; };
    auto keep = [&](int k, double2 v) { return CHIRP && k >= len ? make_double2(0.0, 0.0) : v; };
    if (on && a.kind == FTAMD_LINES_THETA3) {
        // DCT-III of z: the backward DFT of e^{i pi k / 2N} (z_k - i z_{N-k})
        // gives z's output m at 2m or 2 (N-1-m) + 1; DST-III: of the reversed
        // input, odd outputs negated.  (A backward DFT is the conjugate of
        // the forward one of the conjugate.)
        const double *c0 = a.X + (long long)N * (2 * q), *c1 = q > 0 ? c0 - N : c0;
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const unsigned k = within(entry(e)), i = tcos ? k : N - 1 - k;
            x[e] = make_double2(c0[i], c1[i]);
        }
        // z by entry of the line, through LDS for the mirrored entries
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int k = within(entry(e)), i = tcos ? k : N - 1 - k;
            const double f = fcos ? (i == 0 ? a.f0 : 1.0) : (i == N - 1 ? a.f1 : 1.0);
            x[e] = make_double2(x[e].x * f, q > 0 ? x[e].y * f : 0.0);
            lds[S::slot(entry(e))] = x[e];
        }
    }
    if (a.kind == FTAMD_LINES_THETA3) __syncthreads();
    if (on && a.kind == FTAMD_LINES_THETA3) {
        double2 w[E];
#pragma unroll
        for (int e = 0; e < E; ++e) w[e] = a.turn[within(entry(e))];
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int k = entry(e), kc = within(k);
            double2 v = lds[S::slot(kc > 0 ? N - kc : 0)];
            if (kc == 0) v = make_double2(0.0, 0.0);
            x[e] = keep(k, conj(mul(make_double2(x[e].x + v.y, x[e].y - v.x), w[e])));
        }
    }
    if (a.kind == FTAMD_LINES_THETA3) {
        __syncthreads();
    } else if (on && a.kind == FTAMD_LINES_THETA2) {
        // DCT-II of z: the forward DFT of its outputs' order; DST-II: of the
        // sign-alternated input, output reversed
        const double2 *y = a.Y + (long long)N * q;
        auto row = [&](int m) { return 2 * m <= N - 1 ? 2 * m : 2 * (N - 1 - m) + 1; };
#pragma unroll
        for (int e = 0; e < E; ++e) x[e] = y[(unsigned)row(within(entry(e)))];
#pragma unroll
        for (int e = 0; e < E; ++e) {
            x[e] = make_double2(x[e].x * a.a, -x[e].y * a.a);
            if (q == 0) x[e] = make_double2(x[e].x * a.b, 0.0);
        }
        weigh(x, [&](int e) { return row(within(entry(e))); });
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int n = row(within(entry(e)));
            x[e] = keep(entry(e), !tcos && (n & 1) ? make_double2(-x[e].x, -x[e].y) : x[e]);
        }
    } else if (on && a.kind == FTAMD_LINES_PHI_BACK) {
        // the half spectra y0, y1 of both rows give y0 + i y1 at f and
        // conj(y0) + i conj(y1) at M - f (conjugated); through LDS, so that
        // each entry is read once
        const int r0 = 2 * line, r1 = r0 + 1 < N ? 1 : 0;
        constexpr int H = E / 2 > 0 ? E / 2 : 1;
        double2 y0[H], y1[H];
#pragma unroll
        for (int e = 0; e < H; ++e) {
            const double2 *y = a.Y + (long long)N * min(entry(e), M / 2) + r0;
            y0[e] = y[0];
            y1[e] = y[r1];
        }
#pragma unroll
        for (int e = 0; e < H; ++e) {
            const int f = entry(e);
            if (2 * f > M) continue;
            if (!r1) y1[e] = make_double2(0.0, 0.0);
            if (f == 0) y0[e].y = y1[e].y = 0.0;  // a mean is real
            lds[S::slot(f)] = make_double2(y0[e].x - y1[e].y, -(y0[e].y + y1[e].x));
            if (f > 0) lds[S::slot(M - f)] = make_double2(y0[e].x + y1[e].y, y0[e].y - y1[e].x);
        }
    }
    if (a.kind == FTAMD_LINES_PHI_BACK) {
        __syncthreads();
#pragma unroll
        for (int e = 0; e < E; ++e) x[e] = keep(entry(e), lds[S::slot(within(entry(e)))]);
    }
    if (on && a.kind == FTAMD_LINES_PHI_FWD) {
        const int r0 = 2 * line, r1 = r0 + 1 < N ? 1 : 0;
        if (a.aligned) {
#pragma unroll
            for (int e = 0; e < E; ++e) x[e] = *(const double2 *)(a.X + (long long)N * within(entry(e)) + r0);
        } else {
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const double *r = a.X + (long long)N * within(entry(e)) + r0;
                x[e] = make_double2(r[0], r[r1]);
            }
        }
#pragma unroll
        for (int e = 0; e < E; ++e) x[e] = keep(entry(e), r1 ? x[e] : make_double2(x[e].x, 0.0));
    }

    if (CHIRP) {
        double2 c[E];
#pragma unroll
        for (int e = 0; e < E; ++e) c[e] = a.chirp[within(entry(e))];
#pragma unroll
        for (int e = 0; e < E; ++e) x[e] = mulc(x[e], c[e]);
        D::template forward<0>(lds, a.tw, t, x);
#pragma unroll
        for (int e = 0; e < S::EP; ++e) x[e] = mul(x[e], a.filter[entry(e)]);
        D::template backward<S::NP - 1>(lds, a.tw, t, x);
#pragma unroll
        for (int e = 0; e < E; ++e) x[e] = mulc(x[e], a.chirp[within(entry(e))]);
    } else {
        D::template forward<0>(lds, a.tw, t, x);
    }

    if (a.kind == FTAMD_LINES_PHI_BACK && CHIRP) {
        if (!on) return;
        const int r0 = 2 * line;
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int k = entry(e);
            if (k >= len) continue;
            double *r = a.X + (long long)N * k + r0;
            if (a.aligned) {
                *(double2 *)r = make_double2(x[e].x, -x[e].y);
            } else {
                r[0] = x[e].x;
                if (r0 + 1 < N) r[1] = -x[e].y;
            }
        }
        return;
    }
    // the spectrum in natural order (a convolution's is at the points of pass 0, the thread's own)
    if (!CHIRP) __syncthreads();
#pragma unroll
    for (int e = 0; e < E; ++e)
        lds[S::slot(CHIRP ? entry(e) : D::frequency(D::template point<S::NP - 1>(t, e)))] = x[e];
    __syncthreads();
    if (!on) return;
    auto at = [&](int k) { return lds[S::slot(k)]; };
    if (a.kind == FTAMD_LINES_THETA3) {
        double2 *y = a.Y + (long long)N * q;
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int n = within(entry(e));
            x[e] = conj(at((n & 1) ? N - 1 - (n >> 1) : n >> 1));
            if (!tcos && (n & 1)) x[e] = make_double2(-x[e].x, -x[e].y);
        }
        weigh(x, [&](int e) { return within(entry(e)); });
#pragma unroll
        for (int e = 0; e < E; ++e) {
            double2 v = make_double2(x[e].x * a.a, x[e].y * a.a);
            if (q == 0) v = make_double2(v.x * a.b, 0.0);
            if (!CHIRP || entry(e) < N) y[(unsigned)entry(e)] = conj(v);
        }
    } else if (a.kind == FTAMD_LINES_THETA2) {
        double *c0 = a.X + (long long)N * (2 * q), *c1 = c0 - N;
        double2 w[E];
#pragma unroll
        for (int e = 0; e < E; ++e) w[e] = a.turn[tcos ? within(entry(e)) : N - 1 - within(entry(e))];
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int k = within(entry(e)), s = tcos ? k : N - 1 - k;
            const double2 u = at(s), v = at(s > 0 ? N - s : 0);
            const double f = fcos ? (k == 0 ? a.f0 : 1.0) : (k == N - 1 ? a.f1 : 1.0);
            const double2 y = add(mulc(u, w[e]), mul(v, w[e]));
            x[e] = make_double2(y.x * f, y.y * f);
        }
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int k = entry(e);
            if (CHIRP && k >= N) continue;
            c0[k] = x[e].x;
            if (q > 0) c1[k] = x[e].y;
        }
    } else {
        // (M is odd, so these lines are convolutions: M/2 < L/4)
        const int r0 = 2 * line;
        const bool two = r0 + 1 < N;
#pragma unroll
        for (int e = 0; e < E / 2; ++e) {
            const int f = min(entry(e), M / 2);
            x[e] = at(f);
            x[E / 2 + e] = at(f == 0 ? 0 : M - f);
        }
#pragma unroll
        for (int e = 0; e < E / 2; ++e) {
            const int f = entry(e);
            if (2 * f > M) continue;
            const double2 zk = x[e], zm = x[E / 2 + e];
            double2 *y = a.Y + (long long)N * f + r0;
            y[0] = make_double2(0.5 * (zk.x + zm.x), 0.5 * (zk.y - zm.y));
            if (two) y[1] = make_double2(0.5 * (zk.y + zm.y), 0.5 * (zm.x - zk.x));
        }
    }
}

template <int LOGL, bool CHIRP> int launch_lines(const FtamdLines &a, void *stream) {
    using S = Shape<LOGL>;
    const int groups = (a.lines + S::PER - 1) / S::PER;
    hipLaunchKernelGGL((lines_kernel<LOGL, CHIRP>), dim3((groups + 7) / 8 * 8), dim3(S::THREADS), 0, (hipStream_t)stream, a);
    return hipGetLastError() == hipSuccess ? FTAMD_OK : FTAMD_EDEVICE;
}

}  // namespace ftdft
