// Depthwise 3x3 convolution with fused gates on gfx950 (NHWC, HBM-bound streaming kernel).
//
//   y[p, c] = b[c] + sum_{ky, kx} w[c, ky, kx] * x[p + dil * (ky - 1, kx - 1), c]   ('same' zero padding)
//   gate 0: out = act(y)                          (C channels)
//   gate 1: out = y[:, :C/2] * y[:, C/2:]         (SimpleGate)
//   gate 2: out = gelu(y[:, :C/2]) * y[:, C/2:]   (GELU gate, Restormer / FFTformer GDFN)
//   act 1 (gate 0 only): out = gelu(y)
// Semantics of the reference backend's dwconv (python/clarus/ops/torch_ref.py:143-155): fp32
// math, one cast to the output dtype at the end.
//
// A workgroup owns a slice of 64 output channels (the taps and bias of its input channels,
// < 5 KiB, staged in LDS once) and walks pixels 32 at a time, so occupancy does not depend
// on C (a tap table of all C channels per workgroup left one workgroup per CU at C = 2048).
// A thread computes 8 consecutive output channels of one pixel: per tap one 16-byte load of
// each input half (bf16) or two (fp32), fp32 FMAs with the tap weights, then the gate and a
// 16-byte store. The 8 lanes of a pixel read 128 contiguous bytes per input half; the 3x3
// neighbourhood is re-read from L1 / L2.
#include <algorithm>

#include "capi.hpp"
#include "gemm_kernel.hpp"

namespace clarus {

struct DwP {
  const void* x;
  const float* w;   // [9][C_in] fp32 taps, tap = 3 ky + kx
  const float* b;   // [C_in] fp32 or null
  void* out;
  int64_t n, h, w_, cin, cout;  // cout = cin / 2 with a gate
  int dil, gate, act, x_dt, o_dt;
};

constexpr int DW_SLICE = 64;  // output channels per workgroup slice (8 lanes of 8 channels)

template <int XDT, int GATE>
__global__ void __launch_bounds__(256) dwconv3x3_kernel(const DwP p) {
  // taps of the slice's input channels: [9][2][DW_SLICE] fp32 (second half with a gate), bias [2][DW_SLICE]
  __shared__ __attribute__((aligned(16))) float wsh[10][2][DW_SLICE];
  const int cin = (int)p.cin, cout = (int)p.cout;
  const int half = GATE ? cout : 0;  // channel offset of the second input half
  const int nslices = (cout + DW_SLICE - 1) / DW_SLICE;
  const int slice = blockIdx.x % nslices;
  const int cs = slice * DW_SLICE;
  for (int i = threadIdx.x; i < 10 * 2 * DW_SLICE; i += 256) {
    const int tap = i / (2 * DW_SLICE), hh = (i / DW_SLICE) & 1, cc = cs + (i % DW_SLICE);
    const int ci = cc + hh * half;
    float v = 0.f;
    if (cc < cout && (GATE || hh == 0)) v = tap < 9 ? p.w[(int64_t)tap * cin + ci] : (p.b ? p.b[ci] : 0.f);
    wsh[tap][hh][i % DW_SLICE] = v;
  }
  __syncthreads();

  constexpr int XES = (XDT == DT_BF16) ? 2 : 4;
  const int o = threadIdx.x & 7;                    // channel lane of the slice
  const int c0 = cs + o * 8;
  const int H = (int)p.h, W = (int)p.w_, hw = H * W;
  const int npix = (int)p.n * hw;                   // the host checks that this fits 31 bits
  const int pstride = (gridDim.x / nslices) * 32;   // pixels per sweep of the grid
  const unsigned char* X = (const unsigned char*)p.x;
  const float* wb = &wsh[0][0][0] + o * 8;          // tap t, half h at wb + (2 t + h) DW_SLICE
  if (c0 >= cout) return;  // no barrier below
  for (int pix = (blockIdx.x / nslices) * 32 + (threadIdx.x >> 3); pix < npix; pix += pstride) {
    const int img = pix / hw;
    const int r = pix - img * hw;
    const int y = r / W, x = r - (r / W) * W;
    float a1[8], a2[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      a1[i] = wb[18 * DW_SLICE + i];
      a2[i] = GATE ? wb[19 * DW_SLICE + i] : 0.f;
    }
#pragma unroll
    for (int ky = 0; ky < 3; ++ky) {
      const int yy = y + (ky - 1) * p.dil;
      asm volatile("" ::: "memory");  // one tap row of loads in flight at a time: 8 waves per SIMD
      if (yy < 0 || yy >= H) continue;
#pragma unroll
      for (int kx = 0; kx < 3; ++kx) {
        const int xx = x + (kx - 1) * p.dil;
        if (xx < 0 || xx >= W) continue;
        const int tap = ky * 3 + kx;
        const unsigned char* src = X + ((int64_t)((img * H + yy) * W + xx) * cin + c0) * XES;
        const f32x8 v1 = load8<XDT>(src);
        f32x8 v2;
        if constexpr (GATE != 0) v2 = load8<XDT>(src + (int64_t)half * XES);
        const float* wt = wb + 2 * tap * DW_SLICE;
        const f32x4 w1a = *reinterpret_cast<const f32x4*>(wt), w1b = *reinterpret_cast<const f32x4*>(wt + 4);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          a1[i] = fmaf(w1a[i], v1.v[i], a1[i]);
          a1[4 + i] = fmaf(w1b[i], v1.v[4 + i], a1[4 + i]);
        }
        if constexpr (GATE != 0) {
          const f32x4 w2a = *reinterpret_cast<const f32x4*>(wt + DW_SLICE);
          const f32x4 w2b = *reinterpret_cast<const f32x4*>(wt + DW_SLICE + 4);
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            a2[i] = fmaf(w2a[i], v2.v[i], a2[i]);
            a2[4 + i] = fmaf(w2b[i], v2.v[4 + i], a2[4 + i]);
          }
        }
      }
    }
    float out[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      if constexpr (GATE == 1) out[i] = a1[i] * a2[i];
      else if constexpr (GATE == 2) out[i] = gelu_erf(a1[i]) * a2[i];
      else out[i] = p.act == ACT_GELU ? gelu_erf(a1[i]) : a1[i];
    }
    const int64_t oo = (int64_t)pix * cout + c0;
    if (p.o_dt == DT_BF16) {
      u32x4 q;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        q[i] = (unsigned)f32_to_bf16_bits(out[2 * i]) | ((unsigned)f32_to_bf16_bits(out[2 * i + 1]) << 16);
      *reinterpret_cast<u32x4*>((unsigned short*)p.out + oo) = q;
    } else {
      float* op = (float*)p.out + oo;
      *reinterpret_cast<f32x4*>(op) = f32x4{out[0], out[1], out[2], out[3]};
      *reinterpret_cast<f32x4*>(op + 4) = f32x4{out[4], out[5], out[6], out[7]};
    }
  }
}

// ------------------------------------------------------------------- TLC local mean
// out[i, j, c] = (1 / (k1 k2)) sum_{y = i}^{i + k1 - 1} sum_{x = j}^{j + k2 - 1} X[y, x, c],
// i < OH = h - k1 + 1, j < OW = w - k2 + 1 (the valid windows; python/clarus/ops/
// torch_ref.py:133-141 computes the same map from a 2-D prefix sum). Separable: a vertical
// pass sums k1 rows into V [n, OH, w, c] fp32, a horizontal pass sums k2 columns of V. Both
// are one 1-D sliding-window pass over "lines" (an (x, c) column of a plane, or a c of a V row):
//
//   W(i) = sum_{j = i}^{i + k - 1} X[j],  W(i + 1) = W(i) + X[i + k] - X[i]   (fp64, exact to the
//   final rounding for ordinary data).
//
// Outputs are cut into blocks of k positions (van Herk / Gil-Werman): the windows starting in
// block b cover only blocks b and b + 1. A workgroup owns one block of one plane for a range
// of lines; its T threads per line each own R = k / T consecutive positions. A thread loads
// its R rows of block b and of block b + 1 (16-byte loads: 8 bf16 or 4 fp32 channels), sums
// them (A_s, B_s), exchanges the sums through LDS, and starts its recurrence at
//   W(b k + s R) = sum_{s' >= s} A_s' + sum_{s' < s} B_s'
// so no thread walks a k - 1 element warm-up and every row is read twice.
struct BoxPass {
  const void* x;
  void* y;
  int64_t L, k, lo;   // axis length, window, outputs (L - k + 1)
  int64_t inner;      // elements per axis step (contiguous), a multiple of the lane width
  int64_t outer;      // planes (each L x inner)
  int64_t y_plane;    // output elements per plane (lo x inner)
  int T, R, QW;       // threads per line block, positions per thread, lane groups per workgroup
  int nblk, nqg;      // output blocks per plane, lane-group ranges per plane
  double scale;       // 1 / (k1 k2) on the final pass, 1 otherwise
};


// channel c of a raw 16-byte load: 8 bf16 or 4 fp32
template <int DT>
__device__ __forceinline__ float raw_elem(const u32x4& q, int c) {
  if constexpr (DT == DT_BF16) {
    const unsigned w = q[c >> 1];
    return __uint_as_float((c & 1) ? (w & 0xffff0000u) : (w << 16));
  } else {
    return __uint_as_float(q[c]);
  }
}

// NB: rows loaded per batch and stream (loads in flight per thread); with NB >= R a thread's
// rows are loaded once and stay in registers through the recurrence
template <int XDT, int YDT, int NB>
__global__ void __launch_bounds__(256) box_pass_kernel(const BoxPass p) {
  constexpr int BOX_BATCH = NB;
  constexpr int E = XDT == DT_BF16 ? 8 : 4;  // channels per 16-byte load
  constexpr int XES = XDT == DT_BF16 ? 2 : 4;
  constexpr int YES = YDT == DT_BF16 ? 2 : 4;
  __shared__ double part[2][256][E];         // A_s, B_s of every thread
  const int tid = threadIdx.x;
  const int qi = tid % p.QW, s = tid / p.QW;
  int64_t wg = blockIdx.x;
  const int qg = (int)(wg % p.nqg);
  wg /= p.nqg;
  const int b = (int)(wg % p.nblk);
  const int64_t plane = wg / p.nblk;
  const int64_t e0 = ((int64_t)qg * p.QW + qi) * E;  // first channel of this lane group
  const bool live = e0 < p.inner;
  const unsigned char* xp = (const unsigned char*)p.x + (plane * p.L * p.inner + e0) * XES;
  const int64_t pitch = p.inner * XES;
  const int64_t r0 = (int64_t)b * p.k + (int64_t)s * p.R;  // first position of the thread
  const int64_t pend = (int64_t)s * p.R + p.R < p.k ? (int64_t)s * p.R + p.R : p.k;
  const int nj = pend > (int64_t)s * p.R ? (int)(pend - (int64_t)s * p.R) : 0;  // positions in the block
  // rows r0 + j of block b and r0 + k + j of block b + 1 (zero past the axis)
  auto load_rows = [&](int j0, u32x4 (&va)[BOX_BATCH], u32x4 (&vb)[BOX_BATCH]) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < BOX_BATCH; ++j) {
      const int64_t ra = r0 + j0 + j, rb = ra + p.k;
      va[j] = vb[j] = u32x4{0u, 0u, 0u, 0u};
      if (live && j0 + j < nj && ra < p.L) va[j] = *reinterpret_cast<const u32x4*>(xp + ra * pitch);
      if (live && j0 + j < nj && rb < p.L) vb[j] = *reinterpret_cast<const u32x4*>(xp + rb * pitch);
    }
  };
  double sa[E], sb[E];
#pragma unroll
  for (int c = 0; c < E; ++c) sa[c] = sb[c] = 0.0;
  // rows of the last batch stay in registers; when the thread's positions fit one batch
  // (k <= BOX_BATCH T) the recurrence below reuses them instead of reloading
  u32x4 va[BOX_BATCH], vb[BOX_BATCH];
  for (int j0 = 0; j0 < nj; j0 += BOX_BATCH) {
    load_rows(j0, va, vb);
#pragma unroll
    for (int j = 0; j < BOX_BATCH; ++j)
#pragma unroll
      for (int c = 0; c < E; ++c) {
        sa[c] += (double)raw_elem<XDT>(va[j], c);
        sb[c] += (double)raw_elem<XDT>(vb[j], c);
      }
  }
#pragma unroll
  for (int c = 0; c < E; ++c) {
    part[0][tid][c] = sa[c];
    part[1][tid][c] = sb[c];
  }
  __syncthreads();
  double w[E];
#pragma unroll
  for (int c = 0; c < E; ++c) w[c] = 0.0;
  for (int t = 0; t < p.T; ++t) {
    const double* src = part[t >= s ? 0 : 1][t * p.QW + qi];  // A from sub-range s on, B before it
#pragma unroll
    for (int c = 0; c < E; ++c) w[c] += src[c];
  }
  if (!live) return;
  unsigned char* yp = (unsigned char*)p.y + (plane * p.y_plane + e0) * YES;
  // the recurrence over this thread's positions (more than one batch: rows re-read, L1 / L2 hits)
  for (int j0 = 0; j0 < nj; j0 += BOX_BATCH) {
    if (nj > BOX_BATCH) load_rows(j0, va, vb);
#pragma unroll
    for (int j = 0; j < BOX_BATCH; ++j) {
      const int64_t i = r0 + j0 + j;
      if (j0 + j < nj && i < p.lo) {
        unsigned char* o = yp + i * p.inner * YES;
        if constexpr (YDT == DT_BF16) {
          unsigned q[E / 2];
#pragma unroll
          for (int c = 0; c < E / 2; ++c)
            q[c] = (unsigned)f32_to_bf16_bits((float)(w[2 * c] * p.scale)) |
                   ((unsigned)f32_to_bf16_bits((float)(w[2 * c + 1] * p.scale)) << 16);
          if constexpr (E == 8) *reinterpret_cast<u32x4*>(o) = u32x4{q[0], q[1], q[2], q[3]};
          else *reinterpret_cast<u32x2*>(o) = u32x2{q[0], q[1]};
        } else {
#pragma unroll
          for (int c = 0; c < E; c += 4)
            *reinterpret_cast<f32x4*>(o + c * 4) = f32x4{(float)(w[c] * p.scale), (float)(w[c + 1] * p.scale),
                                                         (float)(w[c + 2] * p.scale), (float)(w[c + 3] * p.scale)};
        }
#pragma unroll
        for (int c = 0; c < E; ++c) w[c] += (double)raw_elem<XDT>(vb[j], c) - (double)raw_elem<XDT>(va[j], c);
      }
    }
  }
}

}  // namespace clarus

using namespace clarus;

extern "C" size_t clarus_hip_boxmean_workspace(int64_t n, int64_t h, int64_t w, int64_t c, int64_t k1, int64_t k2) {
  (void)k2;
  if (n <= 0 || h <= 0 || w <= 0 || c <= 0 || k1 < 1 || k1 > h) return 0;
  return (size_t)(n * (h - k1 + 1) * w * c) * sizeof(float);
}

extern "C" int clarus_hip_boxmean(const void* x, int32_t x_dtype, void* out, int32_t o_dtype, int64_t n, int64_t h,
                                  int64_t w, int64_t c, int64_t k1, int64_t k2, void* scratch, size_t scratch_bytes,
                                  void* stream) {
  clear_error();
  CLARUS_REQUIRE(x && out && scratch, "boxmean: null operand");
  CLARUS_REQUIRE(n > 0 && h > 0 && w > 0 && c > 0, "boxmean: empty problem");
  CLARUS_REQUIRE(k1 >= 1 && k1 <= h && k2 >= 1 && k2 <= w, "boxmean: window %lldx%lld outside the %lldx%lld map",
                 (long long)k1, (long long)k2, (long long)h, (long long)w);
  CLARUS_REQUIRE((x_dtype == DT_BF16 || x_dtype == DT_F32) && (o_dtype == DT_BF16 || o_dtype == DT_F32),
                 "boxmean: bad dtype");
  CLARUS_REQUIRE(c % 8 == 0, "boxmean: channels must be a multiple of 8");
  CLARUS_REQUIRE(aligned(x, 16) && aligned(out, 16) && aligned(scratch, 16), "boxmean: 16-byte alignment");
  CLARUS_REQUIRE(n * h * w * c < ((int64_t)1 << 40) && h < (1 << 30) && w < (1 << 30), "boxmean: problem too large");
  const size_t need = clarus_hip_boxmean_workspace(n, h, w, c, k1, k2);
  CLARUS_REQUIRE(scratch_bytes >= need, "boxmean: scratch holds %zu bytes, needs %zu", scratch_bytes, need);
  const int64_t oh = h - k1 + 1;
  hipStream_t s = (hipStream_t)stream;
  // one 1-D pass over `outer` planes of L x inner elements
  auto pass = [&](const void* src, int sdt, void* dst, int ddt, int64_t L, int64_t k, int64_t inner, int64_t outer,
                  double scale) -> bool {
    BoxPass q{};
    q.x = src;
    q.y = dst;
    q.L = L;
    q.k = k;
    q.lo = L - k + 1;
    q.inner = inner;
    q.outer = outer;
    q.y_plane = q.lo * inner;
    // T threads per line block. A thread reads T partial sums (T x 64 B) in the exchange and
    // ~4 k / T rows of 16 B: the two balance at T ~ sqrt(k). T is raised so no lane group of a
    // workgroup is idle (T >= 256 / lane groups in a row), and doubled once more when the GPU
    // would have fewer than ~128 K threads.
    const int E = sdt == DT_BF16 ? 8 : 4;
    const int64_t groups = cdiv(inner, E);
    const int64_t lines = outer * cdiv(q.lo, k) * groups;
    int T0 = 1;
    while ((int64_t)(2 * T0) * (2 * T0) <= k) T0 *= 2;
    int T = T0;
    while (T < 256 && T * groups < 256) T *= 2;
    if (T == T0 && T < 256 && lines * T < 131072) T *= 2;
    // long windows take more threads while each keeps >= 6 positions (NAFNet-w64 720p, cold, us:
    // level 0, k = 384, 128.7 -> 117.4; level 1, k = 192, 62.5 -> 60.9); at 3 positions per
    // thread (k = 96, 48) the exchange outweighs the rows: 35.1 -> 47.7 and 24.9 -> 35.7
    while (T < 256 && lines * T < 262144 && cdiv(k, (int64_t)(2 * T)) >= 6) T *= 2;
    q.T = T;
    q.R = (int)cdiv(k, T);
    q.QW = 256 / T;
    q.nblk = (int)cdiv(q.lo, k);
    q.nqg = (int)cdiv(cdiv(inner, E), q.QW);
    q.scale = scale;
    const int64_t blocks = outer * q.nblk * q.nqg;
    if (blocks >= ((int64_t)1 << 31)) return false;
    // rows per batch: 8, the rows reloaded for the recurrence when R > 8; all R rows kept in
    // registers (one wave per SIMD) where that measured faster, us: bf16 rows with R = 24 (NAFNet
    // level 0, vertical pass) 64.0 vs 70-74, fp32 rows with R = 12 (level 1, horizontal) 28.3 vs
    // 30.4; not kept: bf16 R = 12 (level 1 vertical) 39.1 vs 30-31, fp32 R = 24 64.1 vs 59.4
    const int nb = (sdt == DT_BF16 && q.R > 16 && q.R <= 24) ? 24 : (sdt == DT_F32 && q.R > 8 && q.R <= 16) ? 16 : 8;
#define CLARUS_BOX_LAUNCH(NB_)                                                                             \
  if (sdt == DT_BF16) hipLaunchKernelGGL((box_pass_kernel<DT_BF16, DT_F32, NB_>), dim3((unsigned)blocks), dim3(256), 0, s, q); \
  else if (ddt == DT_BF16) hipLaunchKernelGGL((box_pass_kernel<DT_F32, DT_BF16, NB_>), dim3((unsigned)blocks), dim3(256), 0, s, q); \
  else hipLaunchKernelGGL((box_pass_kernel<DT_F32, DT_F32, NB_>), dim3((unsigned)blocks), dim3(256), 0, s, q);
    if (nb == 8) { CLARUS_BOX_LAUNCH(8) }
    else if (nb == 16) { CLARUS_BOX_LAUNCH(16) }
    else { CLARUS_BOX_LAUNCH(24) }
#undef CLARUS_BOX_LAUNCH
    return true;
  };
  // vertical: planes are images, lines the (x, c) columns; horizontal: planes are V rows
  CLARUS_REQUIRE(pass(x, x_dtype, scratch, DT_F32, h, k1, w * c, n, 1.0), "boxmean: too many workgroups");
  CLARUS_REQUIRE(pass(scratch, DT_F32, out, o_dtype, w, k2, c, n * oh, 1.0 / ((double)k1 * (double)k2)),
                 "boxmean: too many workgroups");
  return check_launch("boxmean");
}

// LDS-tiled form for dilation 1. A workgroup owns a slice of channels and walks tiles of TH x tw output
// pixels. A lane owns one output column of the tile and 8 input channels (with a gate 4 of each half,
// and the gate is formed in the lane; without one 8 consecutive), so cq lanes serve a column's slice of
// 8 cq input channels and tw = 256 / cq columns fit a workgroup; cq is chosen per channel count so that
// few lanes idle (144 channels: 18 lanes x 14 columns, not 2 x 64 of 128). The lane keeps its 72 taps and
// 8 biases in registers and walks its column down the tile: per input row the pixels left, at and right
// of the column come from LDS (the next row's reads issued before this row's FMAs) and feed the up to 3
// outputs whose window holds that row. Per output the sum runs bias, then ky outer, kx inner (the order
// of dwconv3x3_kernel).
// Copies. The tile's input with a one-pixel halo ((TH + 2) x (tw + 2) pixels) is copied global -> LDS
// once by direct 16-byte copies, pixels outside the image from a zero page; with NBUF = 2 the next tile's
// copies go out before the current tile is computed. With a gate a pixel's two halves are swapped in LDS
// when its column is odd, so neighbouring columns read both bank halves.
// Stores are buffer stores whose range ends at the tile's last image row and which drop lanes outside the
// image, so every wave issues the same stores per tile and the wait for the next tile's copies can leave
// them in flight.
// XCD-aware dealing: workgroup L runs on XCD L mod 8, which gets a contiguous eighth of the tiles (all
// slices), so the halo rows and columns that neighbouring tiles share, and the 128-byte lines that
// neighbouring slices share, are read into one L2 mostly once. A multiple of 8 slices is dealt by slice
// instead, XCD = slice mod 8: the same sharing of halos, and the eighths stay in step whatever the tile
// count (a whole NAFNet block at 90 x 160, 512 channels: 150.6 us against 153.9 by eighths). Eighths against
// 64 consecutive tiles per XCD and round (the GPU sweeping top to bottom): Restormer's block 983 / 998 us.
// Bound: HBM for bf16 without a gate or with SimpleGate (C in and out, 2C in and C out); with the GELU gate
// VALU work comes near it (18 FMAs, 6 bf16 unpacks and ~25 slots of GELU per output). Measured (us, 720 x
// 1280 bf16, before -> now): 288 channels no gate 547 (one thread per pixel and 8 channels) -> 251, 4.2 TB/s;
// 144 no gate 254 (register windows along rows) -> 114, 4.6 TB/s; SimpleGate 128 -> 64 90 -> 81, 4.4 TB/s
// (tiles dealt round-robin over the XCDs before); GELU gate 256 -> 128 280 -> 206; fp32 144 491 -> 211.
template <int XDT, int TH>
struct DwTile {
  static constexpr int ROWS = TH + 2;
  static constexpr int UL = XDT == DT_BF16 ? 1 : 2;               // 16-byte units per lane and pixel
  static constexpr int COPIES = ((ROWS * 288 + 255) / 256) * UL;  // copies per lane: (tw + 2) cq <= 288
  static constexpr int BYTES = COPIES * 256 * 16;
};
static __device__ __attribute__((aligned(256))) unsigned char g_dw_zero[256];
typedef float f32x4_u __attribute__((ext_vector_type(4), aligned(4)));  // taps and bias need no alignment

struct DwTileP {
  int cq, tw, nslices, streams;            // lanes per column, columns, slices, tile streams per dealing unit
  int xw;                                  // dealing units: 8 XCDs, or 1 (dealt by slice)
  int tiles_y, tiles_x, ptiles;
  unsigned mag_u, mag_c;                   // ceil(2^19 / (units per pixel)), ceil(2^19 / (tw + 2))
};

template <int XDT, int GATE, int TH, int NBUF, int ODT>
__global__ void __launch_bounds__(256, 2) dw_tile_kernel(const DwP p, const DwTileP g) {
  using G = DwTile<XDT, TH>;
  constexpr int XES = XDT == DT_BF16 ? 2 : 4, OES = ODT == DT_BF16 ? 2 : 4;
  constexpr int SPR = (GATE == 0 && ODT == DT_F32) ? 2 : 1;  // stores per output row of a lane
  constexpr int EU = 16 / XES;                                // channels per 16-byte unit
  __shared__ __attribute__((aligned(16))) unsigned char tile[NBUF][G::BYTES];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int col = (int)threadIdx.x / g.cq, l = (int)threadIdx.x - col * g.cq;
  const int cout = (int)p.cout, cin = (int)p.cin;
  const int sc = (GATE ? 4 : 8) * g.cq;          // output channels of a slice
  const int xcd = blockIdx.x & (g.xw - 1), local = blockIdx.x / g.xw;
  const int slice = local % g.nslices;
  const int cs = slice * sc;
  const int c0 = cs + l * (GATE ? 4 : 8);        // first output channel of the lane
  const bool active = c0 < cout && col < g.tw;   // cout % 8 == 0: all of the lane's channels or none
  float wt[2][9][4], bs[2][4];                   // [half][tap][channel]; lanes past cout hold its last ones
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int ci = min(c0, cout - (GATE ? 4 : 8)) + h * (GATE ? cout : 4);
#pragma unroll
    for (int t = 0; t < 9; ++t) {
      const f32x4_u a = *reinterpret_cast<const f32x4_u*>(p.w + (int64_t)t * cin + ci);
#pragma unroll
      for (int i = 0; i < 4; ++i) wt[h][t][i] = a[i];
    }
    f32x4_u b = {0.f, 0.f, 0.f, 0.f};
    if (p.b) b = *reinterpret_cast<const f32x4_u*>(p.b + ci);
#pragma unroll
    for (int i = 0; i < 4; ++i) bs[h][i] = b[i];
  }
  const int H = (int)p.h, W = (int)p.w_;
  const unsigned char* X = (const unsigned char*)p.x;
  const int upp = g.cq * G::UL, colw = g.tw + 2;   // 16-byte units per pixel, halo columns
  auto tile_pos = [&](int t, int& img, int& y0, int& x0) __attribute__((always_inline)) {
    img = t / (g.tiles_y * g.tiles_x);
    const int rem = t - img * g.tiles_y * g.tiles_x;
    const int ty = rem / g.tiles_x;
    y0 = ty * TH;
    x0 = (rem - ty * g.tiles_x) * g.tw;
  };
  // copy j of a lane fills unit u = (wave + 4 j) * 64 + lane of the LDS image: pixel u / upp of the halo
  // tile and unit u % upp of its channels (with a gate unit k of slot 0 / 1 is half (k's slot) ^ (column % 2))
  // off: byte offset of each copy from the halo tile's first pixel; rc: its row << 8 | column. Units that hold
  // no pixel or channel: offset 0, column 255
  unsigned off[G::COPIES], rc[G::COPIES];
#pragma unroll
  for (int j = 0; j < G::COPIES; ++j) {
    const unsigned u = (unsigned)((wave + 4 * j) * 64 + lane);
    const int pix = (int)(__umul24(u, g.mag_u) >> 19), k = (int)u - __mul24(pix, upp);
    const int r = (int)(__umul24((unsigned)pix, g.mag_c) >> 19), c = pix - __mul24(r, colw);
    int kk = k, seg = 0;
    if constexpr (GATE != 0) {
      const int hu = upp >> 1, slot = k >= hu ? 1 : 0;
      kk = k - slot * hu;
      seg = slot ^ (c & 1);
    }
    const int cc = cs + kk * EU;
    const bool real = cc < cout && r < G::ROWS;
    off[j] = real ? (unsigned)(((r * W + c) * cin + cc + seg * cout) * XES) : 0u;
    rc[j] = real ? (unsigned)(r << 8 | c) : 255u;
  }
  auto issue = [&](int t, unsigned char* dst) __attribute__((always_inline)) {
    int img, y0, x0;
    tile_pos(t, img, y0, x0);
    const unsigned char* base = X + ((((int64_t)img * H + y0 - 1) * W + x0 - 1) * cin) * XES;
    const bool inside = y0 >= 1 && y0 + TH < H && x0 >= 1 && x0 + g.tw < W;  // the whole halo tile is
#pragma unroll
    for (int j = 0; j < G::COPIES; ++j) {
      const unsigned char* src = base + off[j];
      if (!inside) {
        const int c = (int)(rc[j] & 255u), yy = y0 - 1 + (int)(rc[j] >> 8), xx = x0 - 1 + c;
        if (c == 255 || (unsigned)yy >= (unsigned)H || (unsigned)xx >= (unsigned)W) src = g_dw_zero;
      }
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                       (__attribute__((address_space(3))) void*)(dst + (wave + 4 * j) * 1024), 16, 0, 0);
    }
  };
  const int lcol = min(col, g.tw - 1);            // lanes past the last column read the last one
  const int rpitch = colw * upp * 16;
  typedef typename std::conditional<XDT == DT_BF16, u32x2, u32x4>::type Raw4;  // 4 channels as loaded
  auto load_row = [&](const unsigned char* cur, int row, Raw4 (&q)[3][2]) __attribute__((always_inline)) {
#pragma unroll
    for (int dx = 0; dx < 3; ++dx) {
      const unsigned char* px = cur + row * rpitch + (lcol + dx) * upp * 16;
      if constexpr (GATE != 0) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
          q[dx][h] = *reinterpret_cast<const Raw4*>(px + ((h ^ ((lcol + dx) & 1)) * (upp >> 1)) * 16 + l * 4 * XES);
      } else if constexpr (XDT == DT_BF16) {
        const u32x4 v = *reinterpret_cast<const u32x4*>(px + l * 16);
        q[dx][0] = Raw4{v[0], v[1]};
        q[dx][1] = Raw4{v[2], v[3]};
      } else {
        q[dx][0] = *reinterpret_cast<const Raw4*>(px + l * 32);
        q[dx][1] = *reinterpret_cast<const Raw4*>(px + l * 32 + 16);
      }
    }
  };
  // this dealing unit's tiles [lo, hi), every `streams`-th of them this workgroup's
  const int lo = (int)((int64_t)g.ptiles * xcd / g.xw), hi = (int)((int64_t)g.ptiles * (xcd + 1) / g.xw);
  int t = lo + local / g.nslices;
  if (NBUF == 2 && t < hi) issue(t, tile[0]);
  for (int it = 0; t < hi; ++it, t += g.streams) {
    unsigned char* cur = tile[NBUF == 2 ? (it & 1) : 0];
    if constexpr (NBUF == 2) {
      // this tile's copies are older than the previous tile's stores
      if (it == 0) wait_vmcnt<0>(); else wait_vmcnt<TH * SPR>();
      __syncthreads();  // copies landed; every wave is done with the other buffer
      if (t + g.streams < hi) issue(t + g.streams, tile[(it & 1) ^ 1]);
    } else {
      issue(t, cur);
      wait_vmcnt<0>();
      __syncthreads();
    }
    int img, y0, x0;
    tile_pos(t, img, y0, x0);
    const int xo = x0 + col;
    // output rows y0 .. of this image, TH of them or up to its last (the host checks the range's size)
    const int64_t orow = (int64_t)W * cout * OES;
    const __amdgpu_buffer_rsrc_t orc = buf_rsrc_n((unsigned char*)p.out + ((int64_t)img * H + y0) * orow,
                                                  (uint32_t)(min(TH, H - y0) * orow));
    const int ocol = (active && xo < W) ? (xo * cout + c0) * OES : 0x7ffffff0;
    float acc[3][2][4];
    // [row parity][dx][half]: bf16: the row being summed and the next; fp32: the row (registers)
    constexpr int AHEAD = XDT == DT_BF16 ? 1 : 0;
    Raw4 q[1 + AHEAD][3][2];
    if constexpr (AHEAD != 0) load_row(cur, 0, q[0]);
    static_for<G::ROWS>([&](auto IR) __attribute__((always_inline)) {  // input row y0 - 1 + ir
      constexpr int ir = IR.value;
      if constexpr (ir + AHEAD < G::ROWS) load_row(cur, ir + AHEAD, q[(ir + 1) & AHEAD]);
      if constexpr (ir < TH) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[ir % 3][h][i] = bs[h][i];
      }
      float v[3][2][4];
#pragma unroll
      for (int dx = 0; dx < 3; ++dx)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const Raw4 r = q[ir & AHEAD][dx][h];
          if constexpr (XDT == DT_BF16) {
            v[dx][h][0] = __uint_as_float(r[0] << 16);
            v[dx][h][1] = __uint_as_float(r[0] & 0xffff0000u);
            v[dx][h][2] = __uint_as_float(r[1] << 16);
            v[dx][h][3] = __uint_as_float(r[1] & 0xffff0000u);
          } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) v[dx][h][i] = __uint_as_float(r[i]);
          }
        }
      static_for<3>([&](auto KY) __attribute__((always_inline)) {  // outputs whose window holds this row
        constexpr int ky = 2 - KY.value, o = ir - ky;
        if constexpr (o >= 0 && o < TH) {
#pragma unroll
          for (int dx = 0; dx < 3; ++dx)
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
              for (int i = 0; i < 4; ++i)
                acc[o % 3][h][i] = fmaf(wt[h][ky * 3 + dx][i], v[dx][h][i], acc[o % 3][h][i]);
        }
      });
      if constexpr (ir >= 2) {
        constexpr int o = ir - 2;  // output row y0 + o is complete
        const int oo = ocol == 0x7ffffff0 ? ocol : ocol + o * (int)orow;
        float(&a)[2][4] = acc[o % 3];
        if constexpr (GATE != 0) {
          float r[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) r[i] = GATE == 1 ? a[0][i] * a[1][i] : gelu_erf(a[0][i]) * a[1][i];
          if constexpr (ODT == DT_BF16)
            __builtin_amdgcn_raw_buffer_store_b64(u32x2{pack2_bf16(r[0], r[1]), pack2_bf16(r[2], r[3])}, orc, oo, 0, 0);
          else
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, f32x4{r[0], r[1], r[2], r[3]}), orc, oo, 0, 0);
        } else {
          if (p.act == ACT_GELU) {
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
              for (int i = 0; i < 4; ++i) a[h][i] = gelu_erf(a[h][i]);
          }
          if constexpr (ODT == DT_BF16) {
            __builtin_amdgcn_raw_buffer_store_b128(u32x4{pack2_bf16(a[0][0], a[0][1]), pack2_bf16(a[0][2], a[0][3]),
                                                         pack2_bf16(a[1][0], a[1][1]), pack2_bf16(a[1][2], a[1][3])},
                                                   orc, oo, 0, 0);
          } else {
            __builtin_amdgcn_raw_buffer_store_b128(
                __builtin_bit_cast(u32x4, f32x4{a[0][0], a[0][1], a[0][2], a[0][3]}), orc, oo, 0, 0);
            __builtin_amdgcn_raw_buffer_store_b128(
                __builtin_bit_cast(u32x4, f32x4{a[1][0], a[1][1], a[1][2], a[1][3]}), orc, oo, 16, 0);
          }
        }
      }
    });
    if constexpr (NBUF == 1) __syncthreads();  // every wave is done with the tile before the next copies land
  }
}

// Lanes per column, columns and slices of dw_tile_kernel for `units` lane units of channels (4 output
// channels with a gate, else 8), and its tile height, returned. A workgroup takes as long for a tile
// whatever lanes idle: the cost counts tiles (at least the two workgroups per CU that run at once) times a tile's
// rows. cq is even with a gate (16-byte copies of halves) and at least 16 where the channels reach it:
// 256 bytes of a pixel or more per slice (us, 720p bf16 without a gate, 9 lanes -> 18: 288 channels
// 296 -> 250, 144 channels 131 -> 114). Heights: bf16 6 rows, or 2 where 6 leave CUs without a tile
// (32 x 42, 512 channels, gate: 8.7 -> 6.9 us); fp32, whose 6-row tile fills half a CU's LDS, 2 rows
// (90 x 160: 1152 channels 35.2 -> 30.0, 2048 with a GELU gate 69.0 -> 51.5).
static int dw_tile_shape(int64_t units, int64_t n, int64_t H, int64_t W, bool gate, bool f32, DwTileP& g) {
  const int64_t cus = device_cus();
  double best = 1e300;
  int th = 2;
  const int lo = (int)std::min<int64_t>(gate ? units + (units & 1) : units, 16);
  for (int cq = std::max(lo, 2); cq <= 26; ++cq) {
    const int tw = 256 / cq;
    if ((gate && cq % 2) || (tw + 2) * cq > 288) continue;
    const int64_t nsl = cdiv(units, cq);
    for (int t = 2; t <= (f32 ? 2 : 6); t += 4) {
      const double tiles = (double)nsl * (double)(n * cdiv(H, t) * cdiv(W, tw));
      if (t == 2 && !f32 && nsl * n * cdiv(H, 6) * cdiv(W, tw) >= cus) continue;
      const double cost = std::max(tiles / (2.0 * (double)cus), 1.0) * (t + 3.0) * (1.0 + 0.5 / tw);
      if (cost < best * 0.999) {
        best = cost;
        th = t;
        g.cq = cq;
        g.tw = tw;
        g.nslices = (int)nsl;
      }
    }
  }
  return th;
}

// Dilation 1 on the per-pixel kernel all the same: more than 256 input channels (it splits those over workgroups) of
// few pixels, where a launch is one chain of latencies and the tiled kernel's, copy, barrier and walk, is the longer.
// fp32, whose tiles have one buffer: up to 4096 pixels and 2^21 outputs, with a gate 3000 and 1.25 million (us, per
// pixel / tiled: 45 x 61, 288 channels 5.7 / 6.6, gate 384 -> 192 5.5 / 6.7; 24 x 49, GELU gate 2048 -> 1024 8.1 / 10.1; past
// the lines 64 x 64, 576 channels 9.9 / 8.6, 45 x 61 gate 1152 -> 576 12.0 / 9.0). bf16 without a gate: 6-row tiles of
// which only up to an eighth of the CUs get a second (45 x 61, 1152 channels 8.0 / 8.9; 64 x 64, 1024, three
// eighths: 9.1 / 9.1).
static bool dw_per_pixel(int64_t pixels, int64_t c, int64_t cout, bool gate, bool f32, int th, int64_t tiles) {
  if (c <= 256) return false;
  if (f32) return gate ? pixels <= 3000 && pixels * cout <= 1250000 : pixels <= 4096 && pixels * cout <= (1 << 21);
  const int64_t cus = device_cus();
  return !gate && th == 6 && pixels <= 6144 && tiles > cus && 8 * tiles <= 9 * cus;
}

extern "C" int clarus_hip_dwconv3x3(const void* x, int32_t x_dtype, const float* w, const float* bias, void* out,
                                    int32_t o_dtype, int64_t n, int64_t h, int64_t wd, int64_t c, int32_t dil,
                                    int32_t gate, int32_t act, void* stream) {
  clear_error();
  CLARUS_REQUIRE(x && w && out, "dwconv3x3: null operand");
  CLARUS_REQUIRE(n > 0 && h > 0 && wd > 0 && c > 0, "dwconv3x3: empty problem");
  CLARUS_REQUIRE((x_dtype == DT_BF16 || x_dtype == DT_F32) && (o_dtype == DT_BF16 || o_dtype == DT_F32),
                 "dwconv3x3: bad dtype");
  CLARUS_REQUIRE(gate >= 0 && gate <= 2 && (act == 0 || (act == ACT_GELU && gate == 0)) && dil >= 1,
                 "dwconv3x3: bad gate / act / dilation");
  const int64_t cout = gate ? c / 2 : c;
  CLARUS_REQUIRE((gate == 0 || c % 2 == 0) && cout % 8 == 0, "dwconv3x3: output channels must be a multiple of 8");
  CLARUS_REQUIRE(n * h * wd * (cout / 8) < ((int64_t)1 << 31) && n * h * wd * c < ((int64_t)1 << 40),
                 "dwconv3x3: problem too large for 32-bit pixel indexing");
  CLARUS_REQUIRE(aligned(x, 16) && aligned(out, 16), "dwconv3x3: 16-byte alignment");
  DwP p{x, w, bias, out, n, h, wd, c, cout, dil, gate, act, x_dtype, o_dtype};
  // workgroups: channel slices x pixel chunks of 32, persistent with every workgroup resident
  // (a grid-stride loop over more workgroups than fit leaves a tail of late starters)
  const int64_t nslices = cdiv(cout, DW_SLICE);
  const int64_t chunks = cdiv(n * h * wd, 32);
  hipStream_t s = (hipStream_t)stream;
#define DW_LAUNCH(XDT, G)                                                                                       \
  do {                                                                                                          \
    auto fn = &dwconv3x3_kernel<XDT, G>;                                                                        \
    static const int per_cu = [&] {                                                                             \
      int k = 0;                                                                                                \
      if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&k, reinterpret_cast<const void*>(fn), 256, 0) !=       \
              hipSuccess ||                                                                                     \
          k < 1)                                                                                                \
        k = 1;                                                                                                  \
      return k;                                                                                                 \
    }();                                                                                                        \
    const int64_t cap = std::max<int64_t>(1, (int64_t)device_cus() * per_cu / nslices);                                        \
    const unsigned blocks = (unsigned)(nslices * std::min<int64_t>(chunks, cap));                               \
    hipLaunchKernelGGL(fn, dim3(blocks), dim3(256), 0, s, p);                                                   \
  } while (0)
  // LDS-tiled kernel: every call with dilation 1 whose tile rows fit 2^31-byte buffer ranges and whose
  // tile count fits 30 bits (it needs no alignment of taps and bias); the per-pixel kernel keeps dilated
  // taps, whose halo would be larger than the tile, images past those ranges, and what dw_per_pixel names.
  {
    DwTileP g{};
    const int th = dw_tile_shape(cdiv(cout, gate ? 4 : 8), n, h, wd, gate != 0, x_dtype == DT_F32, g);
    const int64_t ptiles = n * cdiv(h, th) * cdiv(wd, g.tw);
    if (dil == 1 && (th + 2) * (wd + 2) * c * 4 < ((int64_t)1 << 31) && ptiles < ((int64_t)1 << 30) &&
        !dw_per_pixel(n * h * wd, c, cout, gate != 0, x_dtype == DT_F32, th, g.nslices * ptiles)) {
      g.tiles_y = (int)cdiv(h, th);
      g.tiles_x = (int)cdiv(wd, g.tw);
      g.ptiles = (int)ptiles;
      const unsigned upp = (unsigned)g.cq * (x_dtype == DT_BF16 ? 1 : 2);
      g.mag_u = ((1u << 19) + upp - 1) / upp;
      g.mag_c = ((1u << 19) + (unsigned)g.tw + 1) / ((unsigned)g.tw + 2);
#define DW_TILE(XDT, G, TH, NBUF, ODT)                                                                          \
  do {                                                                                                          \
    auto fn = &dw_tile_kernel<XDT, G, TH, NBUF, ODT>;                                                           \
    static const int per_cu = [&] {                                                                             \
      int k = 0;                                                                                                \
      if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&k, reinterpret_cast<const void*>(fn), 256, 0) !=       \
              hipSuccess ||                                                                                     \
          k < 1)                                                                                                \
        k = 1;                                                                                                  \
      return k;                                                                                                 \
    }();                                                                                                        \
    g.xw = g.nslices % 8 ? 8 : 1;                                                                               \
    const int64_t cap = std::max<int64_t>(1, (int64_t)device_cus() * per_cu / (g.xw * g.nslices));             \
    g.streams = (int)std::min<int64_t>(cdiv(ptiles, g.xw), cap);                                                \
    hipLaunchKernelGGL(fn, dim3((unsigned)(g.xw * g.nslices * g.streams)), dim3(256), 0, s, p, g);              \
  } while (0)
#define DW_TILE_G(XDT, TH, NBUF, ODT)                                                                           \
  do {                                                                                                          \
    if (gate == 0) DW_TILE(XDT, 0, TH, NBUF, ODT);                                                              \
    else if (gate == 1) DW_TILE(XDT, 1, TH, NBUF, ODT);                                                         \
    else DW_TILE(XDT, 2, TH, NBUF, ODT);                                                                        \
  } while (0)
      note_kernel("dw_tile_kernel gate=%d th=%d cq=%d tw=%d", gate, th, g.cq, g.tw);
      if (x_dtype == DT_BF16 && th == 6) {
        if (o_dtype == DT_BF16) DW_TILE_G(DT_BF16, 6, 2, DT_BF16); else DW_TILE_G(DT_BF16, 6, 2, DT_F32);
      } else if (x_dtype == DT_BF16) {
        if (o_dtype == DT_BF16) DW_TILE_G(DT_BF16, 2, 2, DT_BF16); else DW_TILE_G(DT_BF16, 2, 2, DT_F32);
      } else {
        if (o_dtype == DT_BF16) DW_TILE_G(DT_F32, 2, 1, DT_BF16); else DW_TILE_G(DT_F32, 2, 1, DT_F32);
      }
#undef DW_TILE_G
#undef DW_TILE
      return check_launch("dwconv3x3");
    }
  }
  note_kernel("dwconv3x3_kernel gate=%d dil=%d", gate, (int)dil);
  if (x_dtype == DT_BF16) {
    if (gate == 1) DW_LAUNCH(DT_BF16, 1); else if (gate == 2) DW_LAUNCH(DT_BF16, 2); else DW_LAUNCH(DT_BF16, 0);
  } else {
    if (gate == 1) DW_LAUNCH(DT_F32, 1); else if (gate == 2) DW_LAUNCH(DT_F32, 2); else DW_LAUNCH(DT_F32, 0);
  }
#undef DW_LAUNCH
  return check_launch("dwconv3x3");
}
