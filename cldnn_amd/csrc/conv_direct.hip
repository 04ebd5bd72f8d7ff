// Instances of the direct-activation tile kernel with a table entry per 16-byte chunk of K (feature slices that do not come
// in fours): 64, 128 or 256 pixels x 64 or 128 output features per workgroup.
#include "conv_mfma_kernel.h"

namespace chip {

void launch_direct(hipStream_t s, const MfmaArgs& a, int ofm, int nt, int grid, int lds, int epi)
{
    if (ofm == 64) {
        if (nt == 1) launch_bdir_instance<64, 1, 1, true>(s, a, grid, lds, epi);
        else if (nt == 2) launch_bdir_instance<64, 2, 1, true>(s, a, grid, lds, epi);
        else launch_bdir_instance<64, 4, 1, true>(s, a, grid, lds, epi);
    } else {
        if (nt == 1) launch_bdir_instance<128, 1, 1, true>(s, a, grid, lds, epi);
        else if (nt == 2) launch_bdir_instance<128, 2, 1, true>(s, a, grid, lds, epi);
        else launch_bdir_instance<128, 4, 1, true>(s, a, grid, lds, epi);
    }
}

}  // namespace chip
