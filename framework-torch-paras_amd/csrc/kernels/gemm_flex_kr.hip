// Instantiations of the kernel in gemm_flex_kernel.h for one pair of operand layouts.
#include "kernels/gemm_flex_kernel.h"

namespace paras {
namespace flex {
void launch_kr(bool bf16, int tile, const Params& p, unsigned grid, hipStream_t s) {
    if (bf16) launch_tile<bf16_t, false, true>(tile, p, grid, s);
    else      launch_tile<f16_t, false, true>(tile, p, grid, s);
}
}  // namespace flex
}  // namespace paras
