// gemm_f32_kernel: fp32 rows x fp32 weights with long K (> 128), LayerNorm / RMS of the rows on the way.
//
//   out[q, :] = act(pro(a[q, :]) . W + bias) * scale * out_scale + res[q, :]      (per batch entry)
//
// Restormer's deep levels in fp32 (K = 192 .. 1024). Bound: the fp32 MFMA rate. The general tiled kernel reads
// A from global memory into each lane once per 64 channels and waits for it; here A and W^T pass through LDS.
//   * Tile: 64 pixels x 128 channels, 4 waves of 32 x 64 on 32x32x2 MFMAs with W^T as the A operand (rows
//     permuted so that a lane ends with 16 consecutive channels of a pixel).
//   * K in chunks of 32: rows of 128 bytes copied global -> LDS directly, two buffers, the next chunk in flight
//     during the current one's products. 16-byte units are XOR-swizzled with the row, so the 32 rows of a
//     fragment read fall on distinct banks. Which k a lane half supplies is free as long as both operands
//     agree: half h takes units 2 j + h, one 16-byte read feeding four MFMAs.
//   * Row statistics come from the separate pass; a fragment is normalised as it is read.
//   * Tiles dealt in contiguous runs per XCD, the channel tiles of a pixel tile next to each other.
// Measured (us, before -> now): 14400 rows, LayerNorm, 384 -> 1152 191 -> 146, 384 -> 2048 330 -> 241 (94 TFLOP/s of
// 150 that a large fp32 product reaches on this card); + residual, 1024 -> 384 158 -> 116, 384 -> 384 68 -> 52.
#include "capi.hpp"
#include "gemm_f32_dispatch.hpp"
#include "gemm_kernel.hpp"

namespace clarus {
namespace {

typedef __attribute__((ext_vector_type(16))) float f32x16;
constexpr int F3_KC = 32, F3_TN = 128, F3_TM = 64;
__device__ __attribute__((aligned(256))) unsigned char g_f32_zero[256];

template <bool STATS>
__global__ void __launch_bounds__(256, 2) gemm_f32_kernel(const GemmP p, const int ntiles, const int tiles) {
  constexpr int ROWS = F3_TN + F3_TM;                // W^T rows, then A rows
  constexpr int COPIES = ROWS * 8 / 256;             // 16-byte units per lane and chunk
  constexpr int BUF = ROWS * 128;
  __shared__ __attribute__((aligned(16))) unsigned char lds[2][BUF];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int lp = lane & 31, lh = lane >> 5;
  const int per = (tiles + 7) / 8, xcd = blockIdx.x & 7, idx = blockIdx.x >> 3;
  const int t = xcd * per + idx;
  if (idx >= per || t >= tiles) return;
  const int64_t q0 = (int64_t)(t / ntiles) * F3_TM;
  const int n0 = (t % ntiles) * F3_TN;
  const int N = (int)p.n, K = (int)p.k;
  const int64_t bz = blockIdx.z;
  const float* A = (const float*)p.a + bz * p.a_bs;
  const float* Wt = (const float*)p.wt + bz * p.w_bs;

  // copy j of a lane: unit (wave + 4 j) * 64 + lane: row u / 8, place u % 8 holding source unit (u % 8) ^ (row % 8)
  const float* src[COPIES];
  int uk[COPIES];
#pragma unroll
  for (int j = 0; j < COPIES; ++j) {
    const int u = (wave + 4 * j) * 64 + lane, row = u >> 3, unit = (u & 7) ^ (row & 7);
    uk[j] = unit * 4;
    if (row < F3_TN) {
      const int r = row & 31;  // MFMA row -> channel
      const int ch = n0 + (row & ~31) + 16 * ((r >> 2) & 1) + 4 * (r >> 3) + (r & 3);
      src[j] = Wt + (int64_t)min(ch, N - 1) * K + unit * 4;
    } else {
      src[j] = A + min(q0 + row - F3_TN, p.m - 1) * p.lda + unit * 4;
    }
  }
  auto issue = [&](int k0, unsigned char* dst) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < COPIES; ++j) {
      // past K W^T is zero and the operand must be finite: a normalised row repeats its last unit there, since
      // (0 - mean) * rstd can overflow (rows of one large value)
      const void* pad = STATS && j >= F3_TN / 32 ? (const void*)(src[j] - uk[j] + K - 4) : (const void*)g_f32_zero;
      const void* s = k0 + uk[j] < K ? (const void*)(src[j] + k0) : pad;
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)s,
                                       (__attribute__((address_space(3))) void*)(dst + (wave + 4 * j) * 1024), 16, 0, 0);
    }
  };
  const int wc = (wave & 1) * 64, wp = (wave >> 1) * (F3_TM / 2);  // the wave's channels and pixels in the tile
  const int64_t q = q0 + wp + lp;  // the lane's pixel
  float mean = 0.f, rstd = 1.f;
  if constexpr (STATS) {
    const f32x2 st = *reinterpret_cast<const f32x2*>(p.stats + 2 * min(q, p.m - 1));
    mean = st[0];
    rstd = st[1];
  }
  f32x16 acc[2];
#pragma unroll
  for (int c = 0; c < 2; ++c)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[c][i] = 0.f;

  const int nc = (K + F3_KC - 1) / F3_KC;
  wait_vmcnt<0>();  // the statistics: from here on only copies are counted
  issue(0, lds[0]);
  for (int c = 0; c < nc; ++c) {
    if (c + 1 < nc) {
      issue((c + 1) * F3_KC, lds[(c + 1) & 1]);
      wait_vmcnt<COPIES>();
    } else {
      wait_vmcnt<0>();
    }
    barrier_keep_vm();  // chunk c has landed for every wave
    const unsigned char* cur = lds[c & 1];
#pragma unroll
    for (int j = 0; j < F3_KC / 8; ++j) {
      const int place = ((2 * j + lh) ^ (lp & 7)) * 16;
      f32x4 w[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) w[i] = *reinterpret_cast<const f32x4*>(cur + (wc + 32 * i + lp) * 128 + place);
      f32x4 a = *reinterpret_cast<const f32x4*>(cur + (F3_TN + wp + lp) * 128 + place);
      if constexpr (STATS) {
#pragma unroll
        for (int e = 0; e < 4; ++e) a[e] = (a[e] - mean) * rstd;
      }
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < 2; ++i) acc[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(w[i][e], a[e], acc[i], 0, 0, 0);
    }
    barrier_keep_vm();  // every wave is done with this buffer before the copies two chunks on
  }
  // ---- epilogue: channels c0 .. c0 + 15 of the lane's pixel
  if (q >= p.m) return;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int c0 = n0 + wc + 32 * i + 16 * lh;
#pragma unroll
    for (int j = 0; j < 2; ++j) {  // two runs of 8 channels (N is a multiple of 8)
      const int c = c0 + 8 * j;
      if (c >= N) continue;
      float v[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = acc[i][8 * j + e];
      if (p.bias) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] += p.bias[c + e];
      }
      if (p.act == ACT_GELU) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = gelu_erf(v[e]);
      }
      if (p.scale) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] *= p.scale[c + e] * p.out_scale;
      } else if (p.out_scale != 1.0f) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] *= p.out_scale;
      }
      if (p.has_res) {
        const int64_t ro = bz * p.r_bs + q * p.ldr + c;
        const f32x8 r = p.r_dt == DT_BF16 ? load8<DT_BF16>((const unsigned short*)p.res + ro) : load8<DT_F32>((const float*)p.res + ro);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] += r.v[e];
      }
      const int64_t co = bz * p.c_bs + q * p.ldc + c;
      if (p.c_dt == DT_BF16) {
        *reinterpret_cast<u32x4*>((unsigned short*)p.c + co) =
            u32x4{pack2_bf16(v[0], v[1]), pack2_bf16(v[2], v[3]), pack2_bf16(v[4], v[5]), pack2_bf16(v[6], v[7])};
      } else {
        *reinterpret_cast<f32x4*>((float*)p.c + co) = f32x4{v[0], v[1], v[2], v[3]};
        *reinterpret_cast<f32x4*>((float*)p.c + co + 4) = f32x4{v[4], v[5], v[6], v[7]};
      }
    }
  }
}

}  // namespace

bool gemm_f32_fits(const GemmP& p, int a_dt, int w_dt, int64_t batch) {
  return a_dt == DT_F32 && w_dt == DT_F32 && p.k > 128 && p.n % 8 == 0 && p.c_mode == CM_ROWS && p.vec_out == 2 &&
         (!p.has_res || p.vec_res == 2) && (p.act == ACT_NONE || p.act == ACT_GELU) && batch < 65536 &&
         p.k < (1 << 28) && p.n < (1 << 24) && cdiv(p.m, F3_TM) * cdiv(p.n, F3_TN) < ((int64_t)1 << 30) &&
         (p.pro == PRO_NONE || ((p.pro == PRO_LN || p.pro == PRO_RMS) && p.stats && batch == 1));
}

void launch_gemm_f32(const GemmP& p, int64_t batch, hipStream_t s) {
  const int ntiles = (int)cdiv(p.n, F3_TN), tiles = (int)(cdiv(p.m, F3_TM) * ntiles);
  note_kernel("gemm_f32_kernel stats=%d", p.stats != nullptr);
  const dim3 g((unsigned)(cdiv(tiles, 8) * 8), 1, (unsigned)batch);
  if (p.stats) hipLaunchKernelGGL((gemm_f32_kernel<true>), g, dim3(256), 0, s, p, ntiles, tiles);
  else hipLaunchKernelGGL((gemm_f32_kernel<false>), g, dim3(256), 0, s, p, ntiles, tiles);
}

}  // namespace clarus
