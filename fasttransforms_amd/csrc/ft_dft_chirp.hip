// ft_dft_chirp.hip -- the line transforms of lengths that are no power of two
// (ft_dft.hpp), by the length of the convolution.
#include "ft_dft.hpp"

int ftamd_dft_launch_chirp(int logl, const FtamdLines &a, void *stream) {
    switch (logl) {
        case 6: return ftdft::launch_lines<6, true>(a, stream);
        case 7: return ftdft::launch_lines<7, true>(a, stream);
        case 8: return ftdft::launch_lines<8, true>(a, stream);
        case 9: return ftdft::launch_lines<9, true>(a, stream);
        case 10: return ftdft::launch_lines<10, true>(a, stream);
        case 11: return ftdft::launch_lines<11, true>(a, stream);
        case 12: return ftdft::launch_lines<12, true>(a, stream);
        case 13: return ftdft::launch_lines<13, true>(a, stream);
    }
    return FTAMD_EINVAL;
}
