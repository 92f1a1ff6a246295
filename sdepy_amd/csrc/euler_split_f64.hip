// k_euler_split instances in FP64 (euler_split.hpp).
#include "euler_split.hpp"

namespace sdegpu {

SDEGPU_EULER_SPLIT_SET(double)

}  // namespace sdegpu
