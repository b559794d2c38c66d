// gemm_f32_kernel (gemm_f32.hip): fp32 x fp32 GEMMs with long K.
#pragma once

#include "gemm_kernel.hpp"

namespace clarus {
// the problem (row operands, no gate) is one the kernel takes; LN / RMS need p.stats filled
bool gemm_f32_fits(const GemmP& p, int a_dt, int w_dt, int64_t batch);
void launch_gemm_f32(const GemmP& p, int64_t batch, hipStream_t s);
}  // namespace clarus
