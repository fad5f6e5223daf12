// The GEMM family for fp32 operands.
#include "gemm_typed.h"

namespace ttmi {
TTMI_INSTANTIATE_GEMM(float)
}  // namespace ttmi
