// Mid-batch kernel launchers: 3-bit metadata (one translation unit per operand format, so that the
// library compiles in parallel).
#include "sm24_mid.h"

namespace sm24 {

SM24_MID_INSTANTIATE(VAL4, META3)

}  // namespace sm24
