// Mid-batch kernel launchers: 4-bit values and metadata (one translation unit per operand format, so that the
// library compiles in parallel).
#include "sm24_mid.h"

namespace sm24 {

SM24_MID_INSTANTIATE(VAL4, META4)

hipError_t launch_mid(const GemmArgs& a, const MidShape& d, int vf, int mf, bool grouped, hipStream_t stream) {
  if (vf == VAL3) return launch_mid_t<VAL3, META4>(a, d, grouped, stream);
  if (mf == META3) return launch_mid_t<VAL4, META3>(a, d, grouped, stream);
  return launch_mid_t<VAL4, META4>(a, d, grouped, stream);
}

}  // namespace sm24
