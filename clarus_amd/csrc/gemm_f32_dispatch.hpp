// gemm_f32_kernel (gemm_f32.hip): fp32 x fp32 GEMMs with long K.
#pragma once

#include "gemm_kernel.hpp"

namespace clarus {
// the problem (row operands, no gate) is one the kernel takes; LN / RMS need p.stats filled
bool gemm_f32_fits(const GemmP& p, int a_dt, int w_dt, int64_t batch);
// It beats the general kernel's 64 x 64 tiles there. A tile of 64 x 128 takes about 4 / 3 of the time of one of
// those, so it wins where 4 / 3 of its rounds of tiles over the CUs are fewer than theirs (us, general / this one:
// 14400 rows 384 -> 2048 330 / 241, 3000 rows 384 -> 384 31.0 / 24.8; 40000 rows 1024 -> 48 89 / 111, 6000 rows 1024 ->
// 320 63 / 75). Two exceptions, both from half a round of tiles on. With one round for each, rows without a prologue
// wait for latency and this kernel's is shorter for long K and for channels that end within a 64-channel tile
// (8192 rows 256 -> 96 17.3 / 15.5; with LayerNorm 19.6 / 21.7, and -> 192, 5000 rows, 18.8 / 21.3). Up to 32 channels
// both tiles are mostly padding: up to two rounds of this one's (1024 -> 24: 8192 rows 95 / 46, 40000 rows 95 / 109).
inline bool gemm_f32_faster(int64_t m, int64_t n, int64_t k, int64_t batch, bool pro, int64_t cus) {
  const int64_t mt = cdiv(m, 64) * batch, tiles = mt * cdiv(n, 128), small = mt * cdiv(n, 64);
  if (n <= 32) return 2 * tiles >= cus && tiles <= 2 * cus;
  if (!pro && 2 * tiles >= cus && tiles <= cus && (n % 64 != 0 || k >= 1024)) return true;
  return 4 * cdiv(tiles, cus) < 3 * cdiv(small, cus);
}
void launch_gemm_f32(const GemmP& p, int64_t batch, hipStream_t s);
}  // namespace clarus
