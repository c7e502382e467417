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
