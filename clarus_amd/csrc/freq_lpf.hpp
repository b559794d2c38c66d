// lpf_fft_kernel (freq_lpf.hip): linear_patch_filter on bf16 rows and weights with FFT patch transforms.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace clarus {

struct LpfFftP {
  const void* x;   // bf16 [batch, h, w, k]
  const void* wt;  // bf16 W^T [n][k]
  const float* bias;
  const float* gain;  // [n][80]
  const void* res;
  void* out;  // [batch, h, w, n]
  int64_t patches;
  int h, w, k, n;
  float eps;
  int rms, r_dt, o_dt;
};

// pro: LayerNorm / RMS rows. False (nothing launched) where the kernel does not take the problem: K over 96
// with a prologue, over 192 without one, patch rows past 32-bit buffer offsets.
bool launch_lpf_fft(const LpfFftP& p, bool pro, hipStream_t s);

}  // namespace clarus
