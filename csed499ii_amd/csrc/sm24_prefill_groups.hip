// Large-M 2:4 INT4 x FP16 GEMM: the two-group tiles of sm24_prefill_kernel (256 columns
// x 64 or 96 rows, two k-groups of 4 waves), in a translation unit of their own.
#include "sm24_prefill.h"

namespace sm24 {

hipError_t launch_prefill_groups(const GemmArgs& a, int rows, bool grouped, dim3 grid, hipStream_t stream) {
  constexpr int NW = kPreNarrowChunks;
  const dim3 block(128 * NW);
  if (rows == 64) {
    if (grouped) hipLaunchKernelGGL((sm24_prefill_kernel<true, 2, NW, 2>), grid, block, 0, stream, a);
    else hipLaunchKernelGGL((sm24_prefill_kernel<false, 2, NW, 2>), grid, block, 0, stream, a);
  } else {
    if (grouped) hipLaunchKernelGGL((sm24_prefill_kernel<true, 3, NW, 2>), grid, block, 0, stream, a);
    else hipLaunchKernelGGL((sm24_prefill_kernel<false, 3, NW, 2>), grid, block, 0, stream, a);
  }
  return hipGetLastError();
}

}  // namespace sm24
