// ft_dft.hip -- tables of the line transforms (ft_dft.hpp), on the host in
// long double, and the launches of the power-of-two lengths.
#include "ft_dft.hpp"

#include <math.h>
#include <stdlib.h>

#include <complex>
#include <vector>

struct FtamdDft {
    int len, logl, chirp;
    double2 *tab;  // twiddles, then (chirp) filter and chirp
    const double2 *tw, *filter, *ch;
};

namespace {

typedef std::complex<long double> cld;
constexpr long double kPi = 3.141592653589793238462643383279502884L;

cld unit_root(long long num, long long den) {  // e^{i pi num / den}
    num %= 2 * den;
    return cld(cosl(kPi * num / den), sinl(kPi * num / den));
}

// in-place DFT of a power-of-two length (e^{-}), decimation in time
void dft(std::vector<cld> &v, const std::vector<cld> &root) {
    const size_t L = v.size();
    for (size_t i = 1, j = 0; i < L; ++i) {
        size_t bit = L >> 1;
        for (; j & bit; bit >>= 1) j ^= bit;
        j ^= bit;
        if (i < j) std::swap(v[i], v[j]);
    }
    for (size_t h = 1; h < L; h *= 2)
        for (size_t b = 0; b < L; b += 2 * h)
            for (size_t k = 0; k < h; ++k) {
                const cld t = v[b + k + h] * root[k * (L / (2 * h))];
                v[b + k + h] = v[b + k] - t;
                v[b + k] += t;
            }
}

double2 rounded(cld z) { return make_double2((double)z.real(), (double)z.imag()); }

// The device tables in the order the kernels of length 2^LOGL read them.
template <int LOGL> void tables(int len, bool chirp, std::vector<double2> &out, size_t &filter_at, size_t &chirp_at) {
    using S = ftdft::Shape<LOGL>;
    using D = ftdft::Dft<LOGL>;
    std::vector<cld> root(S::L);  // e^{-2 pi i k / L}
    for (int k = 0; k < S::L; ++k) root[k] = std::conj(unit_root(2LL * k, S::L));
    for (int p = 0; p < S::NP; ++p) {
        const int sub = S::sub(p), block = S::block(p);
        if (sub == 1) break;
        for (int r = 1; r < S::radix(p); ++r)
            for (int o = 0; o < sub; ++o) out.push_back(rounded(root[(size_t)o * r * (S::L / block) % S::L]));
    }
    if (!chirp) return;
    // the chirp's spectrum over L, in the last pass's order
    std::vector<cld> b(S::L);
    for (long long j = 0; j < len; ++j) {
        b[j] = unit_root(j * j, len);
        if (j > 0) b[S::L - j] = b[j];
    }
    const std::vector<cld> c(b.begin(), b.begin() + len);
    dft(b, root);
    filter_at = out.size();
    for (int e = 0; e < S::EP; ++e)
        for (int t = 0; t < S::NT; ++t)
            out.push_back(rounded(b[D::frequency(D::template point<S::NP - 1>(t, e))] / (long double)S::L));
    chirp_at = out.size();
    for (int k = 0; k < len; ++k) out.push_back(rounded(c[k]));
}

}  // namespace

bool ftamd_dft_fits(int len) {
    return len >= 1 && (len <= FTAMD_DFT_MAX || len == 2 * FTAMD_DFT_MAX);
}

static bool by_chirp(int len) { return len < 64 || (len & (len - 1)) != 0; }

int ftamd_dft_points(int len) {
    int points = 64;
    while (points < (by_chirp(len) ? 2 * len - 1 : len)) points *= 2;
    return points;
}

int ftamd_dft_create(int len, FtamdDft **out) {
    *out = NULL;
    if (!ftamd_dft_fits(len)) return FTAMD_EINVAL;
    const bool chirp = by_chirp(len);
    int logl = 6;
    while ((1 << logl) < ftamd_dft_points(len)) ++logl;
    FtamdDft *d = (FtamdDft *)calloc(1, sizeof(FtamdDft));
    if (!d) return FTAMD_ENOMEM;
    d->len = len;
    d->logl = logl;
    d->chirp = chirp;
    size_t fa = 0, ca = 0;
    int rc = FTAMD_OK;
    try {
        std::vector<double2> h;
        switch (logl) {
            case 6: tables<6>(len, chirp, h, fa, ca); break;
            case 7: tables<7>(len, chirp, h, fa, ca); break;
            case 8: tables<8>(len, chirp, h, fa, ca); break;
            case 9: tables<9>(len, chirp, h, fa, ca); break;
            case 10: tables<10>(len, chirp, h, fa, ca); break;
            case 11: tables<11>(len, chirp, h, fa, ca); break;
            case 12: tables<12>(len, chirp, h, fa, ca); break;
            default: tables<13>(len, chirp, h, fa, ca); break;
        }
        if (hipMalloc((void **)&d->tab, sizeof(double2) * (h.size() + 1)) != hipSuccess) rc = FTAMD_ENOMEM;
        else if (hipMemcpy(d->tab, h.data(), sizeof(double2) * h.size(), hipMemcpyHostToDevice) != hipSuccess)
            rc = FTAMD_EDEVICE;
    } catch (...) {  // out of host memory
        rc = FTAMD_ENOMEM;
    }
    if (rc != FTAMD_OK) {
        ftamd_dft_destroy(d);
        return rc;
    }
    d->tw = d->tab;
    d->filter = d->tab + fa;
    d->ch = d->tab + ca;
    *out = d;
    return FTAMD_OK;
}

void ftamd_dft_destroy(FtamdDft *d) {
    if (!d) return;
    hipFree(d->tab);
    free(d);
}

int ftamd_dft_lines(const FtamdDft *d, FtamdLines *a, void *stream) {
    if (!d || !a->X || !a->Y || a->lines < 1) return FTAMD_EINVAL;
    // the kernel indexes len entries of each line
    const bool theta = a->kind == FTAMD_LINES_THETA3 || a->kind == FTAMD_LINES_THETA2;
    if (d->len != (theta ? a->N : a->M) || a->lines != (theta ? a->M / 2 + 1 : (a->N + 1) / 2)) return FTAMD_EINVAL;
    if (theta && !a->turn) return FTAMD_EINVAL;
    a->len = d->len;
    a->tw = d->tw;
    a->filter = d->filter;
    a->chirp = d->ch;
    if (d->chirp) return ftamd_dft_launch_chirp(d->logl, *a, stream);
    switch (d->logl) {
        case 6: return ftdft::launch_lines<6, false>(*a, stream);
        case 7: return ftdft::launch_lines<7, false>(*a, stream);
        case 8: return ftdft::launch_lines<8, false>(*a, stream);
        case 9: return ftdft::launch_lines<9, false>(*a, stream);
        case 10: return ftdft::launch_lines<10, false>(*a, stream);
        case 11: return ftdft::launch_lines<11, false>(*a, stream);
        case 12: return ftdft::launch_lines<12, false>(*a, stream);
        case 13: return ftdft::launch_lines<13, false>(*a, stream);
    }
    return FTAMD_EINVAL;
}
