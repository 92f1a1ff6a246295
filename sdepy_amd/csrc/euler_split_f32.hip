// k_euler_split instances in FP32 (euler_split.hpp).
#include "euler_split.hpp"

namespace sdegpu {

SDEGPU_EULER_SPLIT_SET(float)

}  // namespace sdegpu
