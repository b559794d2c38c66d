// gemm_rowwide_kernel (gemm_rowwide.hip): short rows against all of W^T.
#pragma once

#include "gemm_kernel.hpp"

namespace clarus {
// the problem (row operands, batch 1, no gate) is one the kernel takes
bool gemm_rowwide_fits(const GemmP& p, int a_dt, int w_dt);
bool launch_gemm_rowwide(const GemmP& p, int a_dt, hipStream_t s);
}  // namespace clarus
