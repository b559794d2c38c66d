// gemm_smallm_kernel (gemm_smallm.hip): few rows, whole rows of K = 128 / 256 in registers.
#pragma once

#include "gemm_kernel.hpp"

namespace clarus {
// the problem (row operands, batch 1) is one the kernel takes; its prologue output is rounded once to bf16
bool gemm_smallm_fits(const GemmP& p, int a_dt, int w_dt);
void launch_gemm_smallm(const GemmP& p, int a_dt, bool gate, hipStream_t s);
}  // namespace clarus
