// FP32 register-stage passes.
#include <cmath>

#include "demag_reg_kernels.hpp"

namespace um {

UM_REG_INSTANTIATE(float)

}  // namespace um
