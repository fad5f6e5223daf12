// The GEMM family for fp16 operands.
#include "gemm_typed.h"

namespace ttmi {
TTMI_INSTANTIATE_GEMM(f16)
}  // namespace ttmi
