// Instantiations and launcher of the dense decode- and mid-batch kernel
// (marlin_dense_mid.h).
#include "marlin_dense_mid.h"

namespace sm24 {

template <int NCH, int RB, int AI>
static void launch_dm(const DensePreArgs& a, bool grouped, hipStream_t stream) {
  const dim3 grid(a.N / (64 * NCH) * ((a.M + 16 * RB - 1) / (16 * RB)) * a.splits), block(64 * kDmWaves);
  if (grouped)
    hipLaunchKernelGGL((marlin_dense_mid_kernel<NCH, RB, AI, true>), grid, block, 0, stream, a.A, a.B, a.s, a.M, a.N,
                       a.K, a.splits, a.C, a.partial, a.counters);
  else
    hipLaunchKernelGGL((marlin_dense_mid_kernel<NCH, RB, AI, false>), grid, block, 0, stream, a.A, a.B, a.s, a.M, a.N,
                       a.K, a.splits, a.C, a.partial, a.counters);
}

hipError_t launch_dense_mid(const DensePreArgs& a, const DenseMidShape& d, bool grouped, hipStream_t stream) {
  // up to 8 rows one activation instruction per stage moves them all
  if (d.rb == 1 && a.M <= 8) {
    if (d.nch == 1) launch_dm<1, 1, 1>(a, grouped, stream);
    else launch_dm<2, 1, 1>(a, grouped, stream);
  } else if (d.nch == 1) {
    if (d.rb == 1) launch_dm<1, 1, 2>(a, grouped, stream);
    else if (d.rb == 2) launch_dm<1, 2, 4>(a, grouped, stream);
    else if (d.rb == 3) launch_dm<1, 3, 6>(a, grouped, stream);
    else if (d.rb == 4) launch_dm<1, 4, 8>(a, grouped, stream);
    else launch_dm<1, 5, 10>(a, grouped, stream);
  } else {
    if (d.rb == 1) launch_dm<2, 1, 2>(a, grouped, stream);
    else if (d.rb == 2) launch_dm<2, 2, 4>(a, grouped, stream);
    else if (d.rb == 3) launch_dm<2, 3, 6>(a, grouped, stream);
    else launch_dm<2, 4, 8>(a, grouped, stream);
  }
  return hipGetLastError();
}

}  // namespace sm24
