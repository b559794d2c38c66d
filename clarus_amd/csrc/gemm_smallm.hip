// gemm_smallm_kernel: bf16-weight GEMMs of few rows with whole rows of K = 128 or 256 in registers.
//
//   out[q, :] = gate(pro(a[q, :]) . W + bias) * scale * out_scale + res[q, :],  pro(a) rounded once to bf16
//
// The deep levels of NAFNet on small images (251 x 333 through the width-32 network: 1344 rows of 256 channels
// at level 3, 28 blocks of four such GEMMs). Nothing there fills the chip: the persistent kernels keep 512
// W^T rows per workgroup in registers and run 42 row tiles on them, after a separate pass that normalises the
// fp32 rows or multiplies by the map. What counts is the latency of one short chain, so
//   * a workgroup takes 128 rows x 32 channels (with a gate 32 of each half): 4 waves of 32 rows, one channel
//     tile, hundreds of workgroups;
//   * a wave loads its whole rows into registers at once (A, and the map's rows), while the workgroup copies
//     its W^T tile into LDS in MFMA fragment order; LayerNorm / RMS (exact two-pass) or the map multiply run
//     in the registers of each workgroup again, which costs less than a launch;
//   * MFMA 32x32x16 with W^T as the A operand, rows as columns, two accumulators over the halves of K; a lane
//     ends with 16 consecutive channels of its row.
// Rows past M repeat the last one and are not stored.
// Bound: the latency of one load, LayerNorm, product and store chain. Measured (us, back to back in a graph, 1344
// rows of 256, before -> now): fp32 rows LayerNorm -> 512 10.5 -> 8.2, with the gate -> 256 10.0 -> 9.1; bf16 rows
// + fp32 residual 8.4 -> 6.5, with the map 9.5 -> 8.1. Past one workgroup per CU the persistent kernels win (3072
// rows, LayerNorm -> 512: 11.2 / 15.1).
#include <algorithm>

#include "capi.hpp"
#include "gemm_kernel.hpp"
#include "gemm_smallm_dispatch.hpp"

namespace clarus {
namespace {

typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef float f32x4_u __attribute__((ext_vector_type(4), aligned(4)));  // bias and scale need no alignment

template <int PRO, int TA, bool GATE, int KS>  // PRO_NONE (bf16 rows), PRO_LN (and RMS), PRO_MUL (bf16 rows, map)
__global__ void __launch_bounds__(256) gemm_smallm_kernel(const GemmP p) {
  constexpr int AES = TA == DT_BF16 ? 2 : 4;
  constexpr int G = GATE ? 2 : 1;
  constexpr int K = 16 * KS;
  __shared__ __attribute__((aligned(16))) unsigned char wl[G * KS * 1024];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int lp = lane & 31, lh = lane >> 5;
  const int N = (int)p.n;
  const int ctiles = (N + 31) / 32;
  const int ct = blockIdx.x % ctiles;  // the channel tiles of the same rows on neighbouring XCDs
  const int64_t t = (int64_t)(blockIdx.x / ctiles) * 4 + wave;
  const int64_t q0 = t * 32 + lp, q = min(q0, p.m - 1);
  RawFrag<TA> raw[KS];
  u32x4 mp[PRO == PRO_MUL ? KS : 1];
  {
    const unsigned char* ap = (const unsigned char*)p.a + (q * p.lda + 8 * lh) * AES;
#pragma unroll
    for (int s = 0; s < KS; ++s) raw[s] = raw_load<TA>(ap + 16 * s * AES);
    if constexpr (PRO == PRO_MUL) {
      const int hw = p.h * p.w;
      const int64_t im = q / hw;
      const int r = (int)(q - im * hw), y = r / p.w;
      const int sy = min(max(y - p.pt, 0), p.oh - 1), sx = min(max(r - y * p.w - p.pl, 0), p.ow - 1);
      const unsigned short* sp = (const unsigned short*)p.small + ((im * p.oh + sy) * p.ow + sx) * K + 8 * lh;
#pragma unroll
      for (int s = 0; s < KS; ++s) mp[s] = *reinterpret_cast<const u32x4*>(sp + 16 * s);
    }
  }
  u32x4 wst[G * KS / 4];
#pragma unroll
  for (int j = 0; j < G * KS / 4; ++j) {
    const int e = threadIdx.x + 256 * j, l = e & 63, gs = e >> 6, s = gs % KS, g = gs / KS;
    const int r = l & 31, ch = 32 * ct + 16 * ((r >> 2) & 1) + 4 * (r >> 3) + (r & 3);
    wst[j] = *reinterpret_cast<const u32x4*>((const unsigned short*)p.wt + ((int64_t)min(ch, N - 1) + g * N) * K + 16 * s +
                                             8 * (l >> 5));
  }
  const int c0 = 32 * ct + 16 * lh, left = N - c0;  // the lane's 16 channels, of which so many exist
  const bool live = q0 < p.m;
  u32x4 rr[4];
  if (p.has_res) {
    const int64_t ro = q * p.ldr + c0;
    if (p.r_dt == DT_BF16) {
#pragma unroll
      for (int j = 0; j < 2; ++j)
        rr[j] = left >= 8 * (j + 1) ? *reinterpret_cast<const u32x4*>((const unsigned short*)p.res + ro + 8 * j) : u32x4{0u, 0u, 0u, 0u};
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        rr[j] = left >= 4 * (j + 1) ? *reinterpret_cast<const u32x4*>((const float*)p.res + ro + 4 * j) : u32x4{0u, 0u, 0u, 0u};
    }
  }
  float b[G][16], sc[16];
  auto vec16 = [&](const float* src, float (&o)[16]) __attribute__((always_inline)) {
    if (left >= 16) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const f32x4_u v = *reinterpret_cast<const f32x4_u*>(src + c0 + 4 * j);
#pragma unroll
        for (int i = 0; i < 4; ++i) o[4 * j + i] = v[i];
      }
    } else {
#pragma unroll
      for (int i = 0; i < 16; ++i) o[i] = src[min(c0 + i, N - 1)];
    }
  };
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    sc[i] = 1.f;
#pragma unroll
    for (int g = 0; g < G; ++g) b[g][i] = 0.f;
  }
  if (p.bias) {
#pragma unroll
    for (int g = 0; g < G; ++g) vec16(p.bias + g * N, b[g]);
  }
  if (p.scale) vec16(p.scale, sc);
#pragma unroll
  for (int j = 0; j < G * KS / 4; ++j) *reinterpret_cast<u32x4*>(wl + (threadIdx.x + 256 * j) * 16) = wst[j];

  // ---- the rows as bf16 operands
  bf16x8 a[KS];
  if constexpr (PRO == PRO_NONE) {
    static_assert(PRO != PRO_NONE || TA == DT_BF16, "plain rows are bf16");
#pragma unroll
    for (int s = 0; s < KS; ++s) a[s] = __builtin_bit_cast(bf16x8, raw[s].q);
  } else if constexpr (PRO == PRO_MUL) {
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      f32x8 v = raw_f32<TA>(raw[s]);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        v.v[2 * i] *= __uint_as_float(mp[s][i] << 16);
        v.v[2 * i + 1] *= __uint_as_float(mp[s][i] & 0xffff0000u);
      }
      a[s] = pack_bf16(v);
    }
  } else {
    constexpr float invk = 1.0f / (float)K;
    float mean = 0.f;
    if (p.pro != PRO_RMS) {
      float sum[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const f32x8 v = raw_f32<TA>(raw[s]);
#pragma unroll
        for (int i = 0; i < 8; ++i) sum[i & 3] += v.v[i];
      }
      const float h = (sum[0] + sum[1]) + (sum[2] + sum[3]);
      mean = (h + __shfl_xor(h, 32, 64)) * invk;
    }
    float ss[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const f32x8 v = raw_f32<TA>(raw[s]);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float d = v.v[i] - mean;
        ss[i & 3] = fmaf(d, d, ss[i & 3]);
      }
    }
    const float h = (ss[0] + ss[1]) + (ss[2] + ss[3]);
    const float rstd = rsqrtf((h + __shfl_xor(h, 32, 64)) * invk + p.ln_eps);
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      f32x8 v = raw_f32<TA>(raw[s]);
#pragma unroll
      for (int i = 0; i < 8; ++i) v.v[i] = (v.v[i] - mean) * rstd;
      a[s] = pack_bf16(v);
    }
  }
  __syncthreads();
  f32x16 acc[G][2];
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int i = 0; i < 16; ++i) { acc[g][0][i] = b[g][i]; acc[g][1][i] = 0.f; }
  const unsigned char* wp = wl + lane * 16;
#pragma unroll
  for (int s = 0; s < KS / 2; ++s)
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int g = 0; g < G; ++g)
        acc[g][h] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
            *reinterpret_cast<const bf16x8*>(wp + (g * KS + s + h * (KS / 2)) * 1024), a[s + h * (KS / 2)], acc[g][h], 0, 0, 0);
  float v[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    v[i] = acc[0][0][i] + acc[0][1][i];
    if constexpr (GATE) v[i] *= acc[G - 1][0][i] + acc[G - 1][1][i];
  }
  if (p.act == ACT_GELU) {
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] = gelu_erf(v[i]);
  }
#pragma unroll
  for (int i = 0; i < 16; ++i) v[i] *= sc[i] * p.out_scale;
  if (p.has_res) {
    if (p.r_dt == DT_BF16) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const unsigned w = rr[i >> 2][i & 3];
        v[2 * i] += __uint_as_float(w << 16);
        v[2 * i + 1] += __uint_as_float(w & 0xffff0000u);
      }
    } else {
#pragma unroll
      for (int i = 0; i < 16; ++i) v[i] += __uint_as_float(rr[i >> 2][i & 3]);
    }
  }
  if (!live) return;
  if (p.c_dt == DT_BF16) {
    unsigned short* op = (unsigned short*)p.c + q * p.ldc + c0;
#pragma unroll
    for (int j = 0; j < 2; ++j)
      if (left >= 8 * (j + 1))
        *reinterpret_cast<u32x4*>(op + 8 * j) = u32x4{pack2_bf16(v[8 * j], v[8 * j + 1]), pack2_bf16(v[8 * j + 2], v[8 * j + 3]),
                                                      pack2_bf16(v[8 * j + 4], v[8 * j + 5]), pack2_bf16(v[8 * j + 6], v[8 * j + 7])};
  } else {
    float* op = (float*)p.c + q * p.ldc + c0;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (left >= 4 * (j + 1))
        *reinterpret_cast<f32x4*>(op + 4 * j) = f32x4{v[4 * j], v[4 * j + 1], v[4 * j + 2], v[4 * j + 3]};
  }
}

template <int PRO, int TA, bool GATE>
void launch_sm(const GemmP& p, hipStream_t s) {
  const unsigned blocks = (unsigned)(cdiv(p.m, 128) * cdiv(p.n, 32));
  note_kernel("gemm_smallm_kernel pro=%d a=%s gate=%d k=%d", p.pro, TA == DT_BF16 ? "bf16" : "f32", (int)GATE, (int)p.k);
  if (p.k == 128) hipLaunchKernelGGL((gemm_smallm_kernel<PRO, TA, GATE, 8>), dim3(blocks), dim3(256), 0, s, p);
  else hipLaunchKernelGGL((gemm_smallm_kernel<PRO, TA, GATE, 16>), dim3(blocks), dim3(256), 0, s, p);
}

template <int PRO, int TA>
void pick_sm(const GemmP& p, bool gate, hipStream_t s) {
  if (gate) launch_sm<PRO, TA, true>(p, s);
  else launch_sm<PRO, TA, false>(p, s);
}

}  // namespace

// K = 128 and 256 only: a lane holds half a row, which with fp32 rows of K = 512 is all 256 registers before the operands
bool gemm_smallm_fits(const GemmP& p, int a_dt, int w_dt) {
  if (w_dt != DT_BF16 || (p.k != 128 && p.k != 256) || p.n % 8 || p.vec_out != 2 || (p.has_res && p.vec_res != 2) ||
      (p.act != ACT_NONE && p.act != ACT_GELU) || p.c_mode != CM_ROWS || cdiv(p.m, 128) * cdiv(p.n, 32) >= ((int64_t)1 << 30))
    return false;
  if (p.pro == PRO_LN || p.pro == PRO_RMS) return true;
  return a_dt == DT_BF16 && (p.pro == PRO_NONE || (p.pro == PRO_MUL && p.s_dt == DT_BF16));
}

void launch_gemm_smallm(const GemmP& p, int a_dt, bool gate, hipStream_t s) {
  if (p.pro == PRO_NONE) pick_sm<PRO_NONE, DT_BF16>(p, gate, s);
  else if (p.pro == PRO_MUL) pick_sm<PRO_MUL, DT_BF16>(p, gate, s);
  else if (a_dt == DT_BF16) pick_sm<PRO_LN, DT_BF16>(p, gate, s);
  else pick_sm<PRO_LN, DT_F32>(p, gate, s);
}

}  // namespace clarus
