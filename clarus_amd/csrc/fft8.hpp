// 8-point transforms in registers (the 8 x 8 patch DFT of FFTformer as row and column FFTs), fp32.
//
// rfft2 of a real 8 x 8 patch: a real transform of every row (bins v = 0 .. 4), then a transform of every
// column v over the rows. Columns 0 and 4 of the row transforms are real, so they take real transforms too
// (bins u = 0 .. 4; the others are their conjugates). Radix-2 butterflies, the only constant sqrt(1/2):
// 20 operations for a real transform of 8, 56 for a complex one, against 2 x 64 x 80 multiply-adds per patch
// for the dense matrices.
#pragma once

#include "common.hpp"

namespace clarus {

constexpr float FFT_R = 0.70710678118654752f;

// real x[0 .. 7] -> bins in place: x[0] = X0, x[4] = X4 (real), (x[1], x[5]) = X1, (x[2], x[6]) = X2,
// (x[3], x[7]) = X3 as (re, im); X_v = sum x_n exp(-2 pi i v n / 8)
__device__ __forceinline__ void rfft8(float (&x)[8]) {
  const float a0 = x[0] + x[4], a1 = x[1] + x[5], a2 = x[2] + x[6], a3 = x[3] + x[7];
  const float b0 = x[0] - x[4], b1 = x[1] - x[5], b2 = x[2] - x[6], b3 = x[3] - x[7];
  const float s = a0 + a2, t = a1 + a3, d = b1 - b3, e = b1 + b3;
  x[0] = s + t;
  x[4] = s - t;
  x[2] = a0 - a2;
  x[6] = a3 - a1;
  x[1] = fmaf(FFT_R, d, b0);
  x[5] = -fmaf(FFT_R, e, b2);
  x[3] = fmaf(-FFT_R, d, b0);
  x[7] = fmaf(-FFT_R, e, b2);
}

// the layout of rfft8 back to 8 reals: y_n = X0 + (-1)^n X4 + sum_{v = 1 .. 3} Re(X_v exp(2 pi i v n / 8))
// (the caller's bins 1 .. 3 carry the factor 2 of their conjugates)
__device__ __forceinline__ void irfft8(float (&x)[8]) {
  const float e = x[0] + x[4], o = x[0] - x[4];
  const float s0 = e + x[2], s2 = e - x[2], s1 = o - x[6], s3 = o + x[6];
  const float t0 = x[1] + x[3], t2 = x[7] - x[5], p = x[1] - x[3], q = x[5] + x[7];
  const float t1 = p - q, t3 = p + q;
  x[0] = s0 + t0;
  x[4] = s0 - t0;
  x[2] = s2 + t2;
  x[6] = s2 - t2;
  x[1] = fmaf(FFT_R, t1, s1);
  x[5] = fmaf(-FFT_R, t1, s1);
  x[3] = fmaf(-FFT_R, t3, s3);
  x[7] = fmaf(FFT_R, t3, s3);
}

// 4 complex points in place, natural order: z_u = sum z_k exp(-+ 2 pi i u k / 4) (INV: +)
template <bool INV>
__device__ __forceinline__ void fft4(float& r0, float& i0, float& r1, float& i1, float& r2, float& i2, float& r3,
                                     float& i3) {
  const float ar = r0 + r2, ai = i0 + i2, br = r0 - r2, bi = i0 - i2;
  const float cr = r1 + r3, ci = i1 + i3, dr = r1 - r3, di = i1 - i3;
  r0 = ar + cr; i0 = ai + ci;
  r2 = ar - cr; i2 = ai - ci;
  if constexpr (!INV) {  // -+ i d
    r1 = br + di; i1 = bi - dr;
    r3 = br - di; i3 = bi + dr;
  } else {
    r1 = br - di; i1 = bi + dr;
    r3 = br + di; i3 = bi - dr;
  }
}

// complex 8 points in place, natural order in and out: Z_u = sum z_k exp(-2 pi i u k / 8) (INV: +)
template <bool INV>
__device__ __forceinline__ void fft8(float (&r)[8], float (&i)[8]) {
  float ar[4], ai[4], br[4], bi[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    ar[k] = r[k] + r[k + 4]; ai[k] = i[k] + i[k + 4];
    br[k] = r[k] - r[k + 4]; bi[k] = i[k] - i[k + 4];
  }
  // b_k times w^k, w = exp(-+ 2 pi i / 8) = sqrt(1/2) (1 -+ i)
  float tr, ti;
  if constexpr (!INV) {
    tr = FFT_R * (br[1] + bi[1]); ti = FFT_R * (bi[1] - br[1]);
    br[1] = tr; bi[1] = ti;
    tr = bi[2]; ti = -br[2];
    br[2] = tr; bi[2] = ti;
    tr = FFT_R * (bi[3] - br[3]); ti = -FFT_R * (br[3] + bi[3]);
    br[3] = tr; bi[3] = ti;
  } else {
    tr = FFT_R * (br[1] - bi[1]); ti = FFT_R * (bi[1] + br[1]);
    br[1] = tr; bi[1] = ti;
    tr = -bi[2]; ti = br[2];
    br[2] = tr; bi[2] = ti;
    tr = -FFT_R * (bi[3] + br[3]); ti = FFT_R * (br[3] - bi[3]);
    br[3] = tr; bi[3] = ti;
  }
  fft4<INV>(ar[0], ai[0], ar[1], ai[1], ar[2], ai[2], ar[3], ai[3]);
  fft4<INV>(br[0], bi[0], br[1], bi[1], br[2], bi[2], br[3], bi[3]);
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    r[2 * k] = ar[k]; i[2 * k] = ai[k];
    r[2 * k + 1] = br[k]; i[2 * k + 1] = bi[k];
  }
}

// ---- a patch on two lanes: half h of the wave holds patch rows 4 h .. 4 h + 3; after the row transforms half 0 takes
// columns 0 + 4 (both real, as one complex column) and 2, half 1 columns 1 and 3

// v0.upper <-> v1.lower (lanes 32 .. 63 of v0 with lanes 0 .. 31 of v1); its own inverse
__device__ __forceinline__ void half_swap(float& a, float& b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  a = __uint_as_float(r[0]);
  b = __uint_as_float(r[1]);
}

// gain factors of a channel (gp: its 40 complex gains) for half lh: columns 0 + 4 or 1 as W(u) = P z(u) + Q conj z(-u) per
// component, column 2 or 3 as c. Gains over 64; columns 1 .. 3 doubled; irfft2 keeps the Hermitian part of columns 0
// and 4, so their gains are symmetrised over u and -u (the two halvings make 1 / 4)
__device__ __forceinline__ void patch_gains(const f32x2* gp, int lh, float (&pr)[8], float (&pi)[8], float (&qr)[8],
                                            float (&qi)[8], float (&cr)[8], float (&ci)[8]) {
  f32x2 a[8], d[8];
#pragma unroll
  for (int u = 0; u < 8; ++u) {
    a[u] = gp[5 * u + lh];
    d[u] = gp[5 * u + 4];
    const f32x2 c = gp[5 * u + 2 + lh];
    cr[u] = c[0] * 0.03125f;  // 2 / 64
    ci[u] = c[1] * 0.03125f;
  }
#pragma unroll
  for (int u = 0; u < 8; ++u) {
    const int m = (8 - u) & 7;
    const float r0 = a[u][0] + a[m][0], s0 = a[u][1] + a[m][1], r4 = d[u][0] + d[m][0], s4 = d[u][1] + d[m][1];
    constexpr float q = 0.25f / 64.f;
    pr[u] = lh ? a[u][0] * 0.03125f : (r0 + s4) * q;
    pi[u] = lh ? a[u][1] * 0.03125f : (s0 + r4) * q;
    qr[u] = lh ? 0.f : (r0 - s4) * q;
    qi[u] = lh ? 0.f : (r4 - s0) * q;
  }
}

}  // namespace clarus
