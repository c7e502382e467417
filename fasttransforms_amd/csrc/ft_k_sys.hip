// ft_k_sys.hip -- instantiates the band-systolic engine (ft_systolic.hpp) and
// its C-ABI launcher.
#include "ft_systolic.hpp"

// Two sequences a lane: four in FP64 do not fit the 128 VGPRs a 16-wave
// workgroup allows without spilling.
extern "C" int ftamd_hip_sys_supported(int S, int precision) { return S == 2 && (precision == 0 || precision == 1); }

extern "C" int ftamd_hip_sys_launch(const FtamdSysLaunch *a, int precision, int S, void *stream) {
    using Fn = void (*)(FtamdSysLaunch);
    Fn fn = nullptr;
    if (!ftamd_hip_sys_supported(S, precision)) return FTAMD_EINVAL;
    // sph and disk chains pair the cosine and sine columns of each order
    // (one mask per lane row); tri chains have one order per column
    const bool rm = a->rowmask != 0;
    if (precision == 0) fn = rm ? ftsys::sys_kernel<double, 2, true> : ftsys::sys_kernel<double, 2, false>;
    else fn = rm ? ftsys::sys_kernel<float, 2, true> : ftsys::sys_kernel<float, 2, false>;
    if (!fn) return FTAMD_EINVAL;
    if (a->nchains <= 0) return FTAMD_OK;
    // the kernel indexes xcd_slot[0 .. nxcd] and one ticket per XCD
    if (a->nxcd < 1 || a->nxcd > FTAMD_MAX_XCD || a->grid < 1 || a->nslots < 1 || !a->ctl || (a->nprog > 0 && !a->prog))
        return FTAMD_EINVAL;
    hipLaunchKernelGGL(fn, dim3(a->grid), dim3(ftsys::kWaves * 64), 0, (hipStream_t)stream, *a);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) return FTAMD_OK;
    return e == hipErrorOutOfMemory ? FTAMD_ENOMEM : FTAMD_EDEVICE;
}

namespace ftsys {

// A thread writes the entry of one step and sequence of a band (blockIdx.y).
// Bound by the bus that brings the sines and cosines (n = 2048, FP64: 33 MB,
// and 39 MB of tables; on the host, entry by entry, 45 ms).
template <typename T>
__global__ void __launch_bounds__(256) tables_kernel(Pair<T> *tab, int S, FtamdSysClasses c, const FtamdSysBand *bands,
                                                     const double *sn, const double *cs) {
    const int b = blockIdx.y, B = kLanes * S;
    const FtamdSysBand bd = bands[b];
    const long long x = blockIdx.x * 256LL + threadIdx.x;
    const int t = (int)(x / B), q = (int)(x % B);
    if (t >= bd.steps + FTAMD_SYS_PREFETCH) return;
    int k = 0;
    while (k + 1 < c.ncls && b >= c.cls[k + 1].band0) ++k;
    const auto cl = c.cls[k];
    Pair<T> v{T(0), T(1)};
    if (q < bd.nseq) {
        const int g = bd.gbase + q, j = cl.jtop - cl.jstep * (c.dir == 0 ? g : cl.K - 1 - g);
        const int d = (S + 1) * (q / S) + q % S;  // the step at which position 0 reaches the sequence
        const int e = c.dir == 0 ? bd.R + d - t : t - d - 1;
        // the sequence's last class row
        const int left = c.n - 3 - j - cl.rpar;
        const int top = c.kind == FTAMD_SPH   ? (left >= 0 ? left / 2 : -1)
                        : c.kind == FTAMD_TRI ? c.n - 2 - j
                                              : c.n - 2 - (j + 1) / 2;
        if (e >= 0 && e <= top) {
            const long long row = cl.rstep * e + cl.rpar, n = c.n;
            const long long ix = c.kind == FTAMD_DISK ? row + j * n - (long long)(j / 2) * ((j + 1) / 2)
                                                      : row + j * (2 * n + 1 - j) / 2;
            v = Pair<T>{(T)sn[ix], (T)cs[ix]};
        }
    }
    const int lane = q / S, s = q % S;
    tab[bd.tab + (long long)t * B + (FTAMD_SYS_SLOT_MAJOR(sizeof(T) == 4) ? s * kLanes + lane : q)] = v;
}

// The offsets of a batch's matrices (elements from the launch's A), passed by value.
struct Bases {
    long long off[256];
    int m0, count;
};

// Chains of the matrices m0 .. m0 + count - 1 take their matrix's offset.
__global__ void __launch_bounds__(256) rebase_kernel(FtamdSysChain *chains, const int *mat, int nchains, Bases b) {
    const int c = blockIdx.x * 256 + threadIdx.x;
    if (c >= nchains) return;
    const int m = mat[c] - b.m0;
    if (m >= 0 && m < b.count) chains[c].aoff = b.off[m];
}

}  // namespace ftsys

extern "C" int ftamd_hip_sys_tables(void *tab, int precision, int S, const FtamdSysClasses *c,
                                    const FtamdSysBand *bands, int nbands, int maxsteps, const double *sn,
                                    const double *cs, void *stream) {
    if (nbands <= 0) return FTAMD_OK;
    if (nbands > 65535 || S < 1 || maxsteps < 0 || c->ncls < 1 || c->ncls > 4) return FTAMD_EINVAL;
    const long long entries = (long long)(maxsteps + FTAMD_SYS_PREFETCH) * ftsys::kLanes * S;
    const dim3 grid((unsigned)((entries + 255) / 256), nbands), block(256);
    if (precision == 0)
        hipLaunchKernelGGL(ftsys::tables_kernel<double>, grid, block, 0, (hipStream_t)stream,
                           (ftsys::Pair<double> *)tab, S, *c, bands, sn, cs);
    else
        hipLaunchKernelGGL(ftsys::tables_kernel<float>, grid, block, 0, (hipStream_t)stream, (ftsys::Pair<float> *)tab,
                           S, *c, bands, sn, cs);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? FTAMD_OK : FTAMD_EDEVICE;
}

extern "C" int ftamd_hip_sys_rebase(FtamdSysChain *chains, const int *mat, int nchains, const long long *off,
                                    int count, void *stream) {
    if (nchains <= 0) return FTAMD_OK;
    for (int m0 = 0; m0 < count; m0 += 256) {
        ftsys::Bases b;
        b.m0 = m0;
        b.count = count - m0 < 256 ? count - m0 : 256;
        for (int k = 0; k < 256; ++k) b.off[k] = k < b.count ? off[m0 + k] : 0;
        hipLaunchKernelGGL(ftsys::rebase_kernel, dim3((nchains + 255) / 256), dim3(256), 0, (hipStream_t)stream,
                           chains, mat, nchains, b);
    }
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? FTAMD_OK : FTAMD_EDEVICE;
}
