// Mid-batch kernel launchers: 3-bit values (one translation unit per operand format, so that the
// library compiles in parallel).
#include "sm24_mid.h"

namespace sm24 {

SM24_MID_INSTANTIATE(VAL3, META4)

}  // namespace sm24
