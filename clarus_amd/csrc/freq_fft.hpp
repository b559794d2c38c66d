// fft_patch_kernel (freq_fft.hip): patch_filter and patch_corr with FFT patch transforms.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace clarus {

struct FftPatchP {
  const void* x;
  const float* gain;  // [c][80]; NULL for the correlation
  const void* res;    // dense like out, or NULL
  void* out;          // dense [batch, h, w, c]
  int64_t sn, sh, sw;  // x strides (elements): batch, row, pixel
  int h, w, c, patches;
  int x_dt, r_dt, o_dt;
  int windows, span, groups, streams;  // set by the launch
};

// the x, residual and output bytes lie within one 2^31-byte buffer range each, the counts within 30 bits
bool fft_patch_fits(int64_t sn, int64_t sh, int64_t sw, int64_t batch, int64_t h, int64_t w, int64_t c, bool corr);
void launch_fft_patch(FftPatchP p, bool corr, hipStream_t s);

}  // namespace clarus
