// fft_lpf_kernel: linear_patch_filter for bf16 rows and weights with the patch transforms as FFTs.
//
//   out = patch_filter(prologue(x) . W + bias) (+ residual), the GEMM output never leaving the registers
//
// The dense form (lpf_kernel) multiplies every patch by the 80 x 64 and 64 x 80 DFT matrices, three bf16 MFMAs
// per product, and was bound by that and the splitting into hi + lo around it. Bound now: fp32 VALU work and
// the 2-byte stores (64 bytes per pixel and channel tile). Here:
//   * GEMM on 32x32x16 MFMAs with the patch's pixels as rows (two tiles of 32) and 32 channels as columns. The
//     row order is free, so it is chosen that lane half h accumulates the patch rows 4 h .. 4 h + 3 of its
//     channel: 32 values per lane, two lanes per (patch, channel).
//   * Row transforms in the lane (4 x 20 operations), then 16 permlane32 swaps give half 0 columns 0 + 4 (both
//     real, as one complex column) and 2, half 1 columns 1 and 3, over all 8 rows: two complex 8-point
//     transforms per lane, gains, the inverse ones, the swaps back, the inverse row transforms. About 480 fp32
//     operations per lane; fp32 throughout (the dense products carried 3.5e-6 of split error, this 1e-7).
//   * Real columns packed as z = y0 + i y4: their gains act on z and its mirror, W(u) = P z(u) + Q conj z(-u)
//     per component; irfft2 keeps the Hermitian part of columns 0 and 4, so their gains enter symmetrised.
//   * A workgroup (8 waves) takes PB patches at a time: their rows normalised once and kept in LDS as MFMA
//     operands (hi + lo pairs with a prologue), the next PB patches' rows on the way meanwhile. The (channel
//     tile, patch) items go to the waves tile by tile, so a wave holds a tile's weights and 48 gain factors in
//     registers over several patches.
// Measured (us, bf16, LayerNorm, before -> now): 720 x 1280, 48 -> 288 551 -> 281 (2.2 TB/s); 360 x 640, 96 -> 576 334 -> 170; 180 x 320,
// 192 -> 1152 (rows normalised before) 381 -> 94; 24 x 40, 96 -> 576 119 -> 22.
#include <algorithm>

#include "capi.hpp"
#include "common.hpp"
#include "fft8.hpp"
#include "freq_lpf.hpp"

namespace clarus {
namespace {

typedef __attribute__((ext_vector_type(16))) float f32x16;
constexpr int LF_WAVES = 8;

template <int KS, bool PRO, int PB>
__global__ void __launch_bounds__(64 * LF_WAVES, 2) fft_lpf_kernel(const LpfFftP p) {
  constexpr int HL = PRO ? 2 : 1;                 // operand parts: hi (, lo)
  constexpr int TILEB = KS * HL * 1024;           // LDS bytes of one 32-pixel tile
  constexpr int UW = (2 * PB + LF_WAVES - 1) / LF_WAVES;  // (patch, tile) units a wave normalises
  __shared__ __attribute__((aligned(16))) unsigned char rows[2 * PB * TILEB];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lp = lane & 31, lh = lane >> 5;
  const int H = p.h, W = p.w, K = p.k, N = p.n;
  const int ph = (H + 7) / 8, pw = (W + 7) / 8;
  const int ctall = (N + 31) / 32;  // the workgroup's channel tiles [ct0, ct0 + ctiles): all of them but for few patches
  const int ct0 = ctall * blockIdx.y / gridDim.y, ctiles = ctall * (blockIdx.y + 1) / gridDim.y - ct0;
  const float invk = 1.0f / (float)K;

  auto patch_of = [&](int64_t pt, int64_t& n, int& py, int& px) __attribute__((always_inline)) {
    n = pt / ((int64_t)ph * pw);
    const int rem = (int)(pt - n * ph * pw);
    py = rem / pw;
    px = rem - py * pw;
  };
  // MFMA row of this lane in tile t: patch row dy, column dx (see the accumulator order above)
  const int rr = 4 * (lp >> 3) + (lp & 3);
  const int dy0 = 4 * ((lp >> 2) & 1) + (rr >> 3), dx0 = rr & 7;
  u32x4 raw[UW][KS];
  auto load_rows = [&](int64_t b) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < UW; ++i) {
      const int unit = wave * UW + i, t = unit & 1;
      if (2 * PB % LF_WAVES != 0 && unit >= 2 * PB) continue;
      const int64_t pt = min(b + (unit >> 1), p.patches - 1);
      int64_t n;
      int py, px;
      patch_of(pt, n, py, px);
      int yy = py * 8 + dy0 + 2 * t, xx = px * 8 + dx0;
      yy = yy >= H ? 2 * (H - 1) - yy : yy;
      xx = xx >= W ? 2 * (W - 1) - xx : xx;
      const unsigned short* src = (const unsigned short*)p.x + ((n * H + yy) * W + xx) * K;
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const int k = 16 * s + 8 * lh;
        raw[i][s] = k < K ? *reinterpret_cast<const u32x4*>(src + k) : u32x4{0u, 0u, 0u, 0u};
      }
    }
  };
  auto stage_rows = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < UW; ++i) {
      if (2 * PB % LF_WAVES != 0 && wave * UW + i >= 2 * PB) continue;
      unsigned char* dst = rows + (wave * UW + i) * TILEB + lane * 16;
      if constexpr (!PRO) {
#pragma unroll
        for (int s = 0; s < KS; ++s) *reinterpret_cast<u32x4*>(dst + s * 1024) = raw[i][s];
      } else {
        auto val = [&](int s, int e) __attribute__((always_inline)) {
          const unsigned w = raw[i][s][e >> 1];
          return __uint_as_float((e & 1) ? (w & 0xffff0000u) : (w << 16));
        };
        float mean = 0.f;
        if (!p.rms) {
          float sum = 0.f;
#pragma unroll
          for (int s = 0; s < KS; ++s)
#pragma unroll
            for (int e = 0; e < 8; ++e) sum += val(s, e);
          mean = (sum + __shfl_xor(sum, 32, 64)) * invk;
        }
        float ss = 0.f;
#pragma unroll
        for (int s = 0; s < KS; ++s) {
          float part = 0.f;
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float d = val(s, e) - mean;
            part = fmaf(d, d, part);
          }
          ss += 16 * s + 8 * lh < K ? part : 0.f;
        }
        const float rstd = rsqrtf((ss + __shfl_xor(ss, 32, 64)) * invk + p.eps);
#pragma unroll
        for (int s = 0; s < KS; ++s) {
          f32x8 a;
#pragma unroll
          for (int e = 0; e < 8; ++e) a.v[e] = 16 * s + 8 * lh < K ? (val(s, e) - mean) * rstd : 0.f;
          bf16x8 hi, lo;
          split_bf16(a, hi, lo);
          *reinterpret_cast<bf16x8*>(dst + s * 1024) = hi;
          *reinterpret_cast<bf16x8*>(dst + (KS + s) * 1024) = lo;
        }
      }
    }
  };

  // this workgroup's patches [b, bend), PB at a time
  int64_t b = p.patches * blockIdx.x / gridDim.x;
  const int64_t bend = p.patches * (blockIdx.x + 1) / gridDim.x;
  if (b < bend) load_rows(b);
  for (; b < bend; b += PB) {
    stage_rows();
    __syncthreads();
    if (b + PB < bend) load_rows(b + PB);
    const int items = ctiles * PB;
    int i0 = items * wave / LF_WAVES;
    const int i1 = items * (wave + 1) / LF_WAVES;
    while (i0 < i1) {
      // ---- one channel tile: weights, bias and gain factors of the lane's channel
      const int ct = i0 / PB, iend = min(i1, (ct + 1) * PB);
      const int ch = (ct0 + ct) * 32 + lp, chl = min(ch, N - 1);
      bf16x8 wv[KS];
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const int k = 16 * s + 8 * lh;
        wv[s] = k < K ? *reinterpret_cast<const bf16x8*>((const unsigned short*)p.wt + (int64_t)chl * K + k) : bf16x8{};
      }
      const float bias = p.bias ? p.bias[chl] : 0.f;
      float pr[8], pi[8], qr[8], qi[8], cr[8], ci[8];
      patch_gains(reinterpret_cast<const f32x2*>(p.gain) + (int64_t)chl * 40, lh, pr, pi, qr, qi, cr, ci);
      for (; i0 < iend; ++i0) {
        const int slot = i0 - ct * PB;
        const int64_t pt = b + slot;
        if (pt >= bend) continue;
        // ---- GEMM: z[4 rows][8] of the lane's channel
        float z[4][8];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          f32x16 acc;
#pragma unroll
          for (int i = 0; i < 16; ++i) acc[i] = bias;
          const unsigned char* ar = rows + (2 * slot + t) * TILEB + lane * 16;
#pragma unroll
          for (int s = 0; s < KS; ++s) {
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*reinterpret_cast<const bf16x8*>(ar + s * 1024), wv[s], acc, 0, 0, 0);
            if constexpr (PRO)
              acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*reinterpret_cast<const bf16x8*>(ar + (KS + s) * 1024), wv[s], acc,
                                                            0, 0, 0);
          }
#pragma unroll
          for (int i = 0; i < 16; ++i) z[2 * t + (i >> 3)][i & 7] = acc[i];
        }
        // ---- transforms
#pragma unroll
        for (int j = 0; j < 4; ++j) rfft8(z[j]);
        float ar[8], ai[8], br[8], bi[8];  // half 0: columns 0 + 4 and 2; half 1: columns 1 and 3
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          ar[j] = z[j][0]; ar[j + 4] = z[j][1];
          ai[j] = z[j][4]; ai[j + 4] = z[j][5];
          br[j] = z[j][2]; br[j + 4] = z[j][3];
          bi[j] = z[j][6]; bi[j + 4] = z[j][7];
          half_swap(ar[j], ar[j + 4]);
          half_swap(ai[j], ai[j + 4]);
          half_swap(br[j], br[j + 4]);
          half_swap(bi[j], bi[j + 4]);
        }
        fft8<false>(ar, ai);
        fft8<false>(br, bi);
        float wr[8], wi[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const int m = (8 - u) & 7;
          wr[u] = fmaf(pr[u], ar[u], qr[u] * ar[m]);
          wi[u] = fmaf(pi[u], ai[u], qi[u] * ai[m]);
          br[u] *= cr[u];
          bi[u] *= ci[u];
        }
        fft8<true>(wr, wi);
        fft8<true>(br, bi);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          half_swap(wr[j], wr[j + 4]);
          half_swap(wi[j], wi[j + 4]);
          half_swap(br[j], br[j + 4]);
          half_swap(bi[j], bi[j + 4]);
          z[j][0] = wr[j]; z[j][1] = wr[j + 4];
          z[j][4] = wi[j]; z[j][5] = wi[j + 4];
          z[j][2] = br[j]; z[j][3] = br[j + 4];
          z[j][6] = bi[j]; z[j][7] = bi[j + 4];
          irfft8(z[j]);
        }
        // ---- residual, store: pixel (4 lh + j, s) of channel ch; offsets past the range drop the access
        int64_t n;
        int py, px;
        patch_of(pt, n, py, px);
        const int64_t o0 = ((n * H + py * 8) * W + px * 8) * N;
        unsigned off[4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
          off[j] = ch < N && py * 8 + 4 * lh + j < H ? (unsigned)((4 * lh + j) * W * N + ch) : 0x1fffffffu;
        const int sn = min(8, W - px * 8);  // pixels of the patch inside the image
        if (p.res) {
          const int res = p.r_dt == DT_BF16 ? 2 : 4;
          const __amdgpu_buffer_rsrc_t rs = buf_rsrc_n((const unsigned char*)p.res + o0 * res, (1u << 30) - 64);
#pragma unroll
          for (int s = 0; s < 8; ++s) {
            if (s >= sn) continue;
#pragma unroll
            for (int j = 0; j < 4; ++j)
              z[j][s] += p.r_dt == DT_BF16
                             ? bf16_to_f32((unsigned short)__builtin_amdgcn_raw_buffer_load_b16(rs, off[j] * 2, s * N * 2, 0))
                             : __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, off[j] * 4, s * N * 4, 0));
          }
        }
        if (p.o_dt == DT_BF16) {
          const __amdgpu_buffer_rsrc_t rs = buf_rsrc_n((unsigned char*)p.out + o0 * 2, (1u << 30) - 64);
#pragma unroll
          for (int s = 0; s < 8; ++s) {
            if (s >= sn) continue;
#pragma unroll
            for (int j = 0; j < 4; ++j)
              __builtin_amdgcn_raw_buffer_store_b16(f32_to_bf16_bits(z[j][s]), rs, off[j] * 2, s * N * 2, 0);
          }
        } else {
          const __amdgpu_buffer_rsrc_t rs = buf_rsrc_n((unsigned char*)p.out + o0 * 4, (1u << 30) - 64);
#pragma unroll
          for (int s = 0; s < 8; ++s) {
            if (s >= sn) continue;
#pragma unroll
            for (int j = 0; j < 4; ++j)
              __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(z[j][s]), rs, off[j] * 4, s * N * 4, 0);
          }
        }
      }
    }
    __syncthreads();
  }
}

template <int KS, bool PRO, int PB>
void launch_pb(const LpfFftP& p, dim3 grid, hipStream_t s) {
  note_kernel("fft_lpf_kernel pro=%d ks=%d pb=%d grid=%ux%u", (int)PRO, KS, PB, grid.x, grid.y);
  hipLaunchKernelGGL((fft_lpf_kernel<KS, PRO, PB>), grid, dim3(64 * LF_WAVES), 0, s, p);
}

template <int KS, bool PRO>
void launch_t(const LpfFftP& p, hipStream_t s) {
  // one workgroup per CU (its registers fill it) with an even share of the patches, PB of them in LDS at a time
  // (96 KiB). Up to as many patches as CUs: one per workgroup (45 x 61, 48 -> 288: 34 -> 13 us), and its channel tiles on
  // several workgroups, up to one tile per wave, while CUs are left (16 x 16, 96 -> 576 without a prologue 16.7 -> 8.0 us).
  // Between one and two patches per CU, batches of two, not two rounds of workgroups: 176 x 184, 192 -> 48 21.1 -> 10.8.
  // Six waves with 72 KiB and two workgroups per CU: 342 us against 304 at 720 x 1280, 48 -> 288.
  constexpr int PB = KS * (PRO ? 2 : 1) <= 6 ? 8 : KS * (PRO ? 2 : 1) <= 8 ? 6 : 4;
  const int64_t cus = device_cus();
  if (p.patches >= 2 * cus) return launch_pb<KS, PRO, PB>(p, dim3((unsigned)cus), s);
  if (p.patches > cus) return launch_pb<KS, PRO, 2>(p, dim3((unsigned)cus), s);
  const dim3 grid((unsigned)p.patches, (unsigned)std::min(cdiv(cdiv(p.n, 32), LF_WAVES), cus / p.patches));
  launch_pb<KS, PRO, 1>(p, grid, s);
}

}  // namespace

bool launch_lpf_fft(const LpfFftP& p, bool pro, hipStream_t s) {
  if (p.k % 8 || (int64_t)8 * p.w * p.n * 4 >= ((int64_t)1 << 29)) return false;
  const int ks = (p.k + 15) / 16;
  if (pro) {
    if (ks <= 2) launch_t<2, true>(p, s);
    else if (ks == 3) launch_t<3, true>(p, s);
    else if (ks == 4) launch_t<4, true>(p, s);
    else if (ks <= 6) launch_t<6, true>(p, s);
    else return false;
  } else {
    if (ks <= 3) launch_t<3, false>(p, s);
    else if (ks <= 6) launch_t<6, false>(p, s);
    else if (ks <= 8) launch_t<8, false>(p, s);
    else if (ks <= 12) launch_t<12, false>(p, s);
    else return false;
  }
  return true;
}

}  // namespace clarus
