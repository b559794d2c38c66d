// fft_patch_kernel: patch_filter and patch_corr with the 8 x 8 transforms as FFTs in registers.
//
//   patch_filter : y = irfft2(g_c * rfft2(x)) (+ residual)        patch_corr : y = irfft2(rfft2(q) * rfft2(k))
//
// Bound: HBM (x in, y out). The dense form (patch_kernel) multiplies by the 80 x 64 and 64 x 80 matrices in three
// bf16 MFMAs per product, with hi + lo splits of every value, and reads 16 channels (32 bytes of bf16) at a time.
//   * Two lanes per (patch, channel): half h of the wave holds patch rows 4 h .. 4 h + 3, 32 values per operand;
//     row transforms in the lane, permlane32 swaps, two complex column transforms per lane and back, as in
//     fft_lpf_kernel: fp32 throughout (1e-7; the split products carried 3.5e-6).
//   * The 32 lane pairs of a wave take 32 consecutive entries of the (patch, channel) sequence, so no lane idles
//     whatever the channel count, and a load reads 128 bytes of fp32. 32 / gcd(C, 32) patches make C / gcd(C, 32)
//     whole windows; a wave keeps one window of the group and steps over groups: a lane's channel, its 48 gain
//     factors and its patch within the group are fixed.
//   * Correlation: columns 0 and 4 are real and travel as z = y0 + i y4. With a = Zq(u), a' = conj Zq(-u) and b, b'
//     alike, Q0 K0 + i Q4 K4 = ((a + a')(b + b') - i (a - a')(b - b')) / 4; the other half's plain product a b is
//     the same form with a' = a, b' = b.
//   * No LDS, no barriers; 32 or 64 loads per lane in flight before the first butterfly, occupancy does the rest.
// Measured (us in a graph, warm, patch_kernel -> this one): filter fp32 720 x 1280 x 48 117 -> 88 (4.0 TB/s), 360 x 640 x 96
// 38.6 -> 34.1, 181 x 323 x 96 (reflected edges) 17.0 -> 12.9, 24 x 40 x 48 6.7 -> 6.0; bf16 720 x 1280 x 48 64 -> 46;
// correlation bf16 -> fp32 720 x 1280 x 96 228 -> 171 (4.1 TB/s), fp32 281 -> 218, 24 x 40 x 96 7.2 -> 6.1.
#include <algorithm>
#include <numeric>

#include "capi.hpp"
#include "common.hpp"
#include "fft8.hpp"
#include "freq_fft.hpp"

namespace clarus {
namespace {

constexpr unsigned FP_DROP = 0x7ffffff0u;  // past every range: the access is dropped
constexpr unsigned FP_RANGE = 0x7fffff00u;

// rows 4 h .. 4 h + 3 of a patch -> column spectra: half 0 columns 0 + 4 (a) and 2 (b), half 1 columns 1 and 3
__device__ __forceinline__ void fp_forward(float (&z)[4][8], float (&ar)[8], float (&ai)[8], float (&br)[8], float (&bi)[8]) {
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    rfft8(z[j]);
    ar[j] = z[j][0]; ar[j + 4] = z[j][1];
    ai[j] = z[j][4]; ai[j + 4] = z[j][5];
    br[j] = z[j][2]; br[j + 4] = z[j][3];
    bi[j] = z[j][6]; bi[j + 4] = z[j][7];
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    half_swap(ar[j], ar[j + 4]);
    half_swap(ai[j], ai[j + 4]);
    half_swap(br[j], br[j + 4]);
    half_swap(bi[j], bi[j + 4]);
  }
  fft8<false>(ar, ai);
  fft8<false>(br, bi);
}

// and back
__device__ __forceinline__ void fp_inverse(float (&z)[4][8], float (&ar)[8], float (&ai)[8], float (&br)[8], float (&bi)[8]) {
  fft8<true>(ar, ai);
  fft8<true>(br, bi);
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    half_swap(ar[j], ar[j + 4]);
    half_swap(ai[j], ai[j + 4]);
    half_swap(br[j], br[j + 4]);
    half_swap(bi[j], bi[j + 4]);
    z[j][0] = ar[j]; z[j][1] = ar[j + 4];
    z[j][4] = ai[j]; z[j][5] = ai[j + 4];
    z[j][2] = br[j]; z[j][3] = br[j + 4];
    z[j][6] = bi[j]; z[j][7] = bi[j + 4];
    irfft8(z[j]);
  }
}

template <int DT>
__device__ __forceinline__ float fp_load(const __amdgpu_buffer_rsrc_t r, unsigned elem, int soff) {
  if constexpr (DT == DT_BF16)
    return bf16_to_f32((unsigned short)__builtin_amdgcn_raw_buffer_load_b16(r, (int)(elem * 2u), soff * 2, 0));
  else
    return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, (int)(elem * 4u), soff * 4, 0));
}

// EDGE: h or w is no multiple of 8 (reflected rows and columns in, none of them out)
template <int XDT, bool CORR, bool EDGE>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(4))) fft_patch_kernel(const FftPatchP p) {
  constexpr unsigned XES = XDT == DT_BF16 ? 2 : 4;
  const int lane = threadIdx.x & 63, lp = lane & 31, lh = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int W = p.w, C = p.c;
  const int H = p.h, ph = (H + 7) >> 3, pw = (W + 7) >> 3;
  const int wid = (int)blockIdx.x * ((int)blockDim.x >> 6) + wave;
  const int win = wid % p.windows;
  int g = wid / p.windows;  // the group: p.span patches
  if (g >= p.streams) return;
  const int flat = 32 * win + lp, pd = flat / C, ch = flat - pd * C;
  // the lane's patch and its step of p.streams groups
  int pt = g * p.span + pd, px, py, n;
  {
    const int rows = pt / pw;
    px = pt - rows * pw;
    n = rows / ph;
    py = rows - n * ph;
  }
  const int d_pt = p.streams * p.span, d_rows = d_pt / pw, d_px = d_pt - d_rows * pw, d_n = d_rows / ph,
            d_py = d_rows - d_n * ph;
  float pr[CORR ? 1 : 8], pi[CORR ? 1 : 8], qr[CORR ? 1 : 8], qi[CORR ? 1 : 8], cr[CORR ? 1 : 8], ci[CORR ? 1 : 8];
  if constexpr (!CORR) patch_gains(reinterpret_cast<const f32x2*>(p.gain) + (int64_t)ch * 40, lh, pr, pi, qr, qi, cr, ci);
  const __amdgpu_buffer_rsrc_t xr = buf_rsrc_n(p.x, FP_RANGE), orr = buf_rsrc_n(p.out, FP_RANGE);
  const __amdgpu_buffer_rsrc_t rr = buf_rsrc_n(p.res ? p.res : p.out, FP_RANGE);
  unsigned sh = (unsigned)p.sh, sw = (unsigned)p.sw;

  for (; g < p.groups; g += p.streams) {
    asm volatile("" : "+s"(sh), "+s"(sw), "+s"(C), "+s"(W));  // scalar offsets are formed again, not held in registers
    const bool live = pt < p.patches;
    // ---- element offsets of the lane's first pixel (row 4 lh of the patch), in x and in the dense output
    unsigned xo = 0;
    unsigned xrow[EDGE ? 4 : 1], xcol[EDGE ? 8 : 1];
    if constexpr (EDGE) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        int yy = py * 8 + 4 * lh + j;
        yy = yy >= H ? 2 * (H - 1) - yy : yy;
        xrow[j] = live ? (unsigned)n * (unsigned)p.sn + (unsigned)yy * sh + ch : FP_DROP / XES;
      }
#pragma unroll
      for (int s = 0; s < 8; ++s) {
        int xx = px * 8 + s;
        xx = xx >= W ? 2 * (W - 1) - xx : xx;
        xcol[s] = live ? (unsigned)xx * sw : 0u;
      }
    } else {
      xo = live ? (unsigned)n * (unsigned)p.sn + (unsigned)(py * 8 + 4 * lh) * sh + (unsigned)px * 8 * sw + ch : FP_DROP / XES;
    }
    const unsigned oo = (((unsigned)n * H + py * 8 + 4 * lh) * W + px * 8) * C + ch;
    float z[4][8], k[CORR ? 4 : 1][8];
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int s = 0; s < 8; ++s) {
        const unsigned e = EDGE ? xrow[EDGE ? j : 0] + xcol[EDGE ? s : 0] : xo;
        const int so = EDGE ? 0 : (int)(j * sh + s * sw);
        z[j][s] = fp_load<XDT>(xr, e, so);
        if constexpr (CORR) k[j][s] = fp_load<XDT>(xr, e, so + C);
      }
    float ar[8], ai[8], br[8], bi[8];
    fp_forward(z, ar, ai, br, bi);
    if constexpr (CORR) {
      float er[8], ei[8], fr[8], fi[8];
      fp_forward(k, er, ei, fr, fi);
      const float qs = lh ? 0.25f * 0.03125f : 0.25f / 64.f;
      float wr[8], wi[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int m = (8 - u) & 7;
        const float a1r = lh ? ar[u] : ar[m], a1i = lh ? ai[u] : -ai[m];
        const float e1r = lh ? er[u] : er[m], e1i = lh ? ei[u] : -ei[m];
        const float sr = ar[u] + a1r, si = ai[u] + a1i, tr = er[u] + e1r, ti = ei[u] + e1i;  // a + a', b + b'
        const float dr = ar[u] - a1r, di = ai[u] - a1i, vr = er[u] - e1r, vi = ei[u] - e1i;  // a - a', b - b'
        // s t - i d v
        wr[u] = (fmaf(sr, tr, -si * ti) + fmaf(dr, vi, di * vr)) * qs;
        wi[u] = (fmaf(sr, ti, si * tr) - fmaf(dr, vr, -di * vi)) * qs;
      }
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const float xr_ = br[u], xi_ = bi[u];
        br[u] = fmaf(xr_, fr[u], -xi_ * fi[u]) * 0.03125f;
        bi[u] = fmaf(xr_, fi[u], xi_ * fr[u]) * 0.03125f;
      }
      fp_inverse(z, wr, wi, br, bi);
    } else {
      float wr[8], wi[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int m = (8 - u) & 7;
        wr[u] = fmaf(pr[u], ar[u], qr[u] * ar[m]);
        wi[u] = fmaf(pi[u], ai[u], qi[u] * ai[m]);
        br[u] *= cr[u];
        bi[u] *= ci[u];
      }
      fp_inverse(z, wr, wi, br, bi);
    }
    // ---- residual, store: row j of the lane's four, column s
    auto each = [&](auto&& f) __attribute__((always_inline)) {
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int s = 0; s < 8; ++s) {
          const bool in = live && (!EDGE || (py * 8 + 4 * lh + j < H && px * 8 + s < W));
          f(j, s, in, (j * W + s) * C);
        }
    };
    if constexpr (!CORR) {
      if (p.res) {
        if (p.r_dt == DT_BF16)
          each([&](int j, int s, bool in, int so) __attribute__((always_inline)) {
            z[j][s] += fp_load<DT_BF16>(rr, in ? oo : FP_DROP / 2, so);
          });
        else
          each([&](int j, int s, bool in, int so) __attribute__((always_inline)) {
            z[j][s] += fp_load<DT_F32>(rr, in ? oo : FP_DROP / 4, so);
          });
      }
    }
    if (!CORR && p.o_dt == DT_BF16)
      each([&](int j, int s, bool in, int so) __attribute__((always_inline)) {
        __builtin_amdgcn_raw_buffer_store_b16(f32_to_bf16_bits(z[j][s]), orr, in ? (int)(oo * 2u) : (int)FP_DROP, so * 2, 0);
      });
    else
      each([&](int j, int s, bool in, int so) __attribute__((always_inline)) {
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(z[j][s]), orr, in ? (int)(oo * 4u) : (int)FP_DROP, so * 4, 0);
      });
    pt += d_pt;
    px += d_px;
    int carry = px >= pw;
    px -= carry ? pw : 0;
    py += d_py + carry;
    carry = py >= ph;
    py -= carry ? ph : 0;
    n += d_n + carry;
  }
}

template <int XDT, bool CORR, bool EDGE>
void launch_fp(FftPatchP& p, hipStream_t s) {
  const int gcd = std::gcd(p.c, 32);
  p.windows = p.c / gcd;
  p.span = 32 / gcd;
  p.groups = (p.patches + p.span - 1) / p.span;
  // a workgroup: whole groups of up to 8 waves, so the 128-byte lines that windows share stay in one CU
  const int waves = p.windows <= 8 ? 8 / p.windows * p.windows : 8;
  auto fn = &fft_patch_kernel<XDT, CORR, EDGE>;
  static OccupancyMemo occ;
  const int per_cu = occ.get(reinterpret_cast<const void*>(fn), 64 * waves, 0);
  // as many streams of groups as whole workgroups hold, up to the waves that run at once
  const int64_t cap = std::max<int64_t>(1, (int64_t)device_cus() * per_cu * waves / p.windows);
  p.streams = (int)std::min<int64_t>(p.groups, cap);
  const int64_t total = (int64_t)p.streams * p.windows;
  p.streams = (int)(cdiv(total, waves) * waves / p.windows);
  const int64_t blocks = cdiv((int64_t)p.streams * p.windows, waves);
  hipLaunchKernelGGL(fn, dim3((unsigned)blocks), dim3(64 * waves), 0, s, p);
}

template <int XDT>
void pick_fp(FftPatchP& p, hipStream_t s) {
  if (p.h % 8 || p.w % 8) launch_fp<XDT, false, true>(p, s);
  else launch_fp<XDT, false, false>(p, s);
}

}  // namespace

bool fft_patch_fits(int64_t sn, int64_t sh, int64_t sw, int64_t batch, int64_t h, int64_t w, int64_t c, bool corr) {
  constexpr int64_t most = FP_RANGE / 4, count = (int64_t)1 << 30;
  if (batch >= count || h >= count || w >= count || c >= (1 << 24) || sn < 0 || sh < 0 || sw < 0 || sn >= count || sh >= count ||
      sw >= count)
    return false;
  const double span = (double)(batch - 1) * (double)sn + (double)(h - 1) * (double)sh + (double)(w - 1) * (double)sw;
  return span + (corr ? 2 : 1) * c < (double)most && (double)batch * h * w * c < (double)most;
}

void launch_fft_patch(FftPatchP p, bool corr, hipStream_t s) {
  note_kernel("fft_patch_kernel corr=%d", (int)corr);
  if (corr) {
    if (p.x_dt == DT_BF16) launch_fp<DT_BF16, true, false>(p, s);
    else launch_fp<DT_F32, true, false>(p, s);
  } else {
    if (p.x_dt == DT_BF16) pick_fp<DT_BF16>(p, s);
    else pick_fp<DT_F32>(p, s);
  }
}

}  // namespace clarus
