// Instances of the split-K kernel whose lanes find their own taps (fewer than four feature slices, input without a border).
#include "conv_ksplit_kernel.h"

namespace chip {

void launch_ksplit_lanes(hipStream_t s, const KsplitArgs& a, int ft, int pt, int grid, int epi)
{
    launch_ksplit_tile<ADDR_LANES>(s, a, ft, pt, grid, epi);
}

}  // namespace chip
