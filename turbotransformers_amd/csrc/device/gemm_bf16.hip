// The GEMM family for bf16 operands.
#include "gemm_typed.h"

namespace ttmi {
TTMI_INSTANTIATE_GEMM(bf16)
}  // namespace ttmi
