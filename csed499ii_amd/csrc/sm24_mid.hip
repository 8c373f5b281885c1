// Mid-batch kernel launchers: 4-bit values and metadata (one translation unit per operand format, so that the
// library compiles in parallel).
#include "sm24_mid.h"

namespace sm24 {

SM24_MID_INSTANTIATE(VAL4, META4)

hipError_t launch_mid(const GemmArgs& a, const MidShape& d, int vf, int mf, bool grouped, hipStream_t stream) {
  hipError_t e;
  if (vf == VAL3) e = launch_mid_t<VAL3, META4>(a, d, grouped, stream);
  else if (mf == META3) e = launch_mid_t<VAL4, META3>(a, d, grouped, stream);
  else e = launch_mid_t<VAL4, META4>(a, d, grouped, stream);
  if (e != hipSuccess || a.splits == 1 || a.counters != nullptr) return e;
  const dim3 grid((unsigned)(((size_t)a.M * a.N / 4 + 255) / 256));
  const int mb = 16 * d.rb;
  if (d.ncb == 4) {
    if (grouped) hipLaunchKernelGGL((sm24_mid_reduce_kernel<64, true>), grid, dim3(256), 0, stream, a, mb);
    else hipLaunchKernelGGL((sm24_mid_reduce_kernel<64, false>), grid, dim3(256), 0, stream, a, mb);
  } else {
    if (grouped) hipLaunchKernelGGL((sm24_mid_reduce_kernel<128, true>), grid, dim3(256), 0, stream, a, mb);
    else hipLaunchKernelGGL((sm24_mid_reduce_kernel<128, false>), grid, dim3(256), 0, stream, a, mb);
  }
  return hipGetLastError();
}

}  // namespace sm24
