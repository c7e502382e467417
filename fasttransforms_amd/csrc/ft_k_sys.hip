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
// The values come from the pairs that the plans' upload left on the device, and
// the plans of a batch are one launch: with an upload of the sines and cosines,
// two allocations and a wait for each plan, 48 spheres of degree 32 .. 1024
// took 11.3 ms on their first call, half of it here.  Bound by the 39 MB of
// tables at n = 2048 in FP64 (on the host, entry by entry, 45 ms).
template <typename T>
__global__ void __launch_bounds__(256) tables_kernel(const FtamdSysTableJob *jobs, const int *job,
                                                     const FtamdSysBand *bands, int b0, int S) {
    const int b = b0 + blockIdx.y, B = kLanes * S;
    const FtamdSysBand bd = bands[b];
    const FtamdSysTableJob &jb = jobs[job[b]];
    const long long x = blockIdx.x * 256LL + threadIdx.x;
    const int t = (int)(x / B), q = (int)(x % B);
    if (t >= bd.steps + FTAMD_SYS_PREFETCH) return;
    if (x == 0) jb.bands[b - jb.band0] = bd;
    const FtamdSysClasses &c = jb.c;
    int k = 0;
    while (k + 1 < c.ncls && b - jb.band0 >= c.cls[k + 1].band0) ++k;
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
            // the pair's place (ftamd_plan_upload: a sphere's column holds its even rows first)
            const long long n = jb.npairs;
            const int row = cl.rstep * e + cl.rpar;
            const int at = c.kind == FTAMD_SPH && (row & 1) ? (jb.npairs - j + 1) / 2 + row / 2
                           : c.kind == FTAMD_SPH            ? row / 2
                                                            : row;
            const long long col = c.kind == FTAMD_DISK ? j * n - (long long)(j / 2) * ((j + 1) / 2)
                                                       : j * (2 * n + 1 - j) / 2;
            v = ((const Pair<T> *)jb.pairs)[col + at];
        }
    }
    const int lane = q / S, s = q % S;
    ((Pair<T> *)jb.tab)[bd.tab + (long long)t * B + (FTAMD_SYS_SLOT_MAJOR(sizeof(T) == 4) ? s * kLanes + lane : q)] = v;
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

extern "C" int ftamd_hip_sys_tables(const FtamdSysTableJob *jobs, const int *job, const FtamdSysBand *bands,
                                    int nbands, int maxsteps, int precision, int S, void *stream) {
    if (S < 1 || maxsteps < 0 || nbands < 0) return FTAMD_EINVAL;
    const long long entries = (long long)(maxsteps + FTAMD_SYS_PREFETCH) * ftsys::kLanes * S;
    for (int b0 = 0; b0 < nbands; b0 += 65535) {
        const dim3 grid((unsigned)((entries + 255) / 256), nbands - b0 < 65535 ? nbands - b0 : 65535), block(256);
        if (precision == 0)
            hipLaunchKernelGGL(ftsys::tables_kernel<double>, grid, block, 0, (hipStream_t)stream, jobs, job, bands, b0, S);
        else
            hipLaunchKernelGGL(ftsys::tables_kernel<float>, grid, block, 0, (hipStream_t)stream, jobs, job, bands, b0, S);
    }
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
