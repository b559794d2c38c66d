// gemm_rowwide_kernel: short rows (16 < K <= 96) against all of W^T at once, for bf16 weights.
//
//   out[q, :] = act(pro(a[q, :]) . W + bias) * scale * out_scale + res[q, :]
//
// The LayerNorm GEMMs of Restormer and FFTformer (K = 48 / 96 -> N = 144 .. 576 channels) and the LayerNorm-
// multiply projection (fp32 correlation rows, K = 96 -> 48). HBM bound: A in, N channels out. The streaming
// kernels walk W^T 64 or 128 channels at a time, so A was read and normalised 2 to 5 times and a wave held
// one 16-pixel block; here a wave takes 32 pixels, normalises their rows once in registers, keeps them as
// hi + lo bf16 operands (the same operand mode: fp32-accurate products) and runs through all channel tiles.
//   * MFMA 32x32x16 with W^T as the A operand and the pixels as columns. Rows of W^T are permuted so that a
//     lane accumulates 16 consecutive channels of its pixel (two 16-byte stores of bf16). Accumulators start
//     from the bias.
//   * W^T sits in LDS in fragment order (one 1 KiB run per tile and 16-k step), the bias, scale and LN-mul
//     vectors beside it: at most 60 KiB of W^T per workgroup, more channels go to further workgroups of the
//     same XCD, so the rows they share come into one L2 once.
//   * A lane loads 8 consecutive k of its pixel per step straight into registers, the next tile's rows before
//     the current tile's products; occupancy hides the rest (bf16 rows: 4 waves per SIMD).
//   * Two channel tiles leave through LDS as 128-byte runs per pixel (16-byte stores straight from the
//     accumulators: N = 256 181 us, through LDS 117 us).
// Measured (us, 720 x 1280 bf16 rows, LayerNorm, before -> now): K = 48 -> 144 250 -> 85, -> 256 222 -> 118
// (4.7 TB/s), -> 288 368 -> 142; 360 x 640, K = 96 -> 288 140 -> 51, -> 576 215 -> 102; LN-multiply fp32 96 -> 48
// with a residual 511 -> 173 (4.1 TB/s); 24 x 49 rows, K = 48 -> 144 11.2 -> 6.5.
#include <algorithm>

#include "capi.hpp"
#include "gemm_kernel.hpp"
#include "gemm_rowwide_dispatch.hpp"

namespace clarus {
namespace {

typedef __attribute__((ext_vector_type(16))) float f32x16;

struct RwP {
  GemmP g;
  int ntc, nch;  // channel tiles per chunk, chunks
};

constexpr int RW_W_MAX = 60 * 1024;
constexpr int RW_LDS_MAX = 160 * 1024;  // of a CU
constexpr int RW_ST_ROW = 128 + 16;  // bytes per pixel of a wave's store tile (not linear)

template <int PRO, int TA, int KS, bool LIN>
__global__ void __launch_bounds__(256, LIN ? 2 : TA == DT_F32 ? 3 : KS <= 4 ? 4 : 3) gemm_rowwide_kernel(const RwP rp) {
  const GemmP& p = rp.g;
  constexpr bool LNMUL = PRO == PRO_LNMUL;
  constexpr bool SPLIT = PRO != PRO_NONE || TA == DT_F32;
  constexpr int AES = TA == DT_BF16 ? 2 : 4;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  const int ntc = rp.ntc;
  unsigned char* wl = lds;
  float* bl = (float*)(lds + (size_t)ntc * KS * 1024);  // bias, scale [32 ntc], then lnw, lnb [16 KS]
  float* sl = bl + 32 * ntc;
  float* lw = sl + 32 * ntc;
  float* lb = lw + 16 * KS;
  const int st_row = LIN ? (int)p.n * 2 : RW_ST_ROW;
  unsigned char* st = (unsigned char*)(lb + 16 * KS) + (threadIdx.x >> 6) * (32 * st_row);  // the wave's store tile
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int lp = lane & 31, lh = lane >> 5;
  const int K = (int)p.k, N = (int)p.n;
  const int xcd = blockIdx.x & 7, local = blockIdx.x >> 3;  // the grid is a multiple of 8 chunks
  const int chunk = local % rp.nch;
  const int n0 = chunk * ntc * 32;
  const int nt = min(ntc, (N - n0 + 31) / 32);
  for (int e = threadIdx.x; e < nt * KS * 64; e += 256) {
    const int l = e & 63, ts = e >> 6, T = ts / KS, s = ts - T * KS;
    const int r = l & 31;
    const int row = n0 + 32 * T + 16 * ((r >> 2) & 1) + 4 * (r >> 3) + (r & 3), k = 16 * s + 8 * (l >> 5);
    u32x4 v = {0u, 0u, 0u, 0u};
    if (row < N && k < K) v = *reinterpret_cast<const u32x4*>((const unsigned short*)p.wt + (int64_t)row * K + k);
    *reinterpret_cast<u32x4*>(wl + e * 16) = v;
  }
  for (int e = threadIdx.x; e < 32 * ntc; e += 256) {
    const bool in = n0 + e < N;
    bl[e] = in && p.bias ? p.bias[n0 + e] : 0.f;
    sl[e] = (in && p.scale ? p.scale[n0 + e] : 1.f) * p.out_scale;
  }
  if constexpr (LNMUL) {
    for (int e = threadIdx.x; e < 16 * KS; e += 256) {
      lw[e] = e < K ? p.lnw[e] : 0.f;
      lb[e] = e < K ? p.lnb[e] : 0.f;
    }
  }
  __syncthreads();

  const bool plain = !p.scale && p.out_scale == 1.0f;
  const float invk = 1.0f / (float)K;
  const int64_t tiles = (p.m + 31) / 32;
  const int64_t wpx = (int64_t)(gridDim.x >> 3) / rp.nch * 4;  // waves per XCD on one chunk
  RawFrag<TA> raw[KS];
  u32x4 mraw[LNMUL ? KS : 1];
  auto load_rows = [&](int64_t t) __attribute__((always_inline)) {
    const int64_t q = min(t * 32 + lp, p.m - 1);  // rows past M repeat the last one and are not stored
    const unsigned char* ap = (const unsigned char*)p.a + q * p.lda * AES;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const int k = 16 * s + 8 * lh;
      raw[s] = k < K ? raw_load<TA>(ap + k * AES) : raw_zero<TA>();
      if constexpr (LNMUL)
        mraw[s] = k < K ? *reinterpret_cast<const u32x4*>((const unsigned short*)p.m2 + q * p.ldm2 + k) : u32x4{0u, 0u, 0u, 0u};
    }
  };
  int64_t t = ((int64_t)(local / rp.nch) * 4 + wave) * 8 + xcd;
  const int64_t step = wpx * 8;
  constexpr bool AHEAD = !LNMUL;  // the fp32 rows and the multiplier of one tile fill the registers
  if (AHEAD && t < tiles) load_rows(t);
  for (; t < tiles; t += step) {
    if constexpr (!AHEAD) load_rows(t);
    // ---- the rows as operands
    bf16x8 hi[KS], lo[SPLIT ? KS : 1];
    if constexpr (PRO == PRO_NONE && TA == DT_BF16) {
#pragma unroll
      for (int s = 0; s < KS; ++s) hi[s] = __builtin_bit_cast(bf16x8, raw[s].q);
    } else {
      float mean = 0.f, rstd = 1.f;
      if constexpr (PRO != PRO_NONE) {  // exact two-pass statistics from the registers
        if (p.pro != PRO_RMS) {
          float sum = 0.f;
#pragma unroll
          for (int s = 0; s < KS; ++s) {
            const f32x8 a = raw_f32<TA>(raw[s]);
#pragma unroll
            for (int i = 0; i < 8; ++i) sum += a.v[i];
          }
          mean = (sum + __shfl_xor(sum, 32, 64)) * invk;
        }
        float ss = 0.f;
#pragma unroll
        for (int s = 0; s < KS; ++s) {
          const f32x8 a = raw_f32<TA>(raw[s]);
          float part = 0.f;
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            const float d = a.v[i] - mean;
            part = fmaf(d, d, part);
          }
          ss += 16 * s + 8 * lh < K ? part : 0.f;
        }
        rstd = rsqrtf((ss + __shfl_xor(ss, 32, 64)) * invk + p.ln_eps);
      }
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        f32x8 a = raw_f32<TA>(raw[s]);
        if constexpr (PRO != PRO_NONE) {
#pragma unroll
          for (int i = 0; i < 8; ++i) a.v[i] = (a.v[i] - mean) * rstd;
        }
        if constexpr (LNMUL) {
          const int k = 16 * s + 8 * lh;
          const f32x8 w8 = load8<DT_F32>(lw + k), b8 = load8<DT_F32>(lb + k);
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            float m0 = __uint_as_float(mraw[s][i] << 16), m1 = __uint_as_float(mraw[s][i] & 0xffff0000u);
            if (p.m2_act == ACT_GELU) { m0 = gelu_erf(m0); m1 = gelu_erf(m1); }
            a.v[2 * i] = (a.v[2 * i] * w8.v[2 * i] + b8.v[2 * i]) * m0;
            a.v[2 * i + 1] = (a.v[2 * i + 1] * w8.v[2 * i + 1] + b8.v[2 * i + 1]) * m1;
          }
        }
        // k past K: W^T is zero there, the operand must be finite
        if (16 * s + 8 * lh >= K) a = zero8();
        split_bf16(a, hi[s], lo[SPLIT ? s : 0]);
      }
    }
    const int64_t q = t * 32 + lp;
    const bool live = q < p.m;
    if (AHEAD && t + step < tiles) load_rows(t + step);
    if constexpr (LIN) {
      // ---- two channel tiles at a time (independent product chains) into the wave's store tile, then its
      // 32 dense rows as one run of memory
      for (int T = 0; T < nt; T += 2) {
        const int T1 = min(T + 1, nt - 1);  // an odd count computes its last tile twice
        const unsigned char* w0 = wl + ((size_t)T * KS * 64 + lane) * 16;
        const unsigned char* w1 = wl + ((size_t)T1 * KS * 64 + lane) * 16;
        f32x16 acc[2];
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const f32x4 b = *reinterpret_cast<const f32x4*>(bl + 32 * (h ? T1 : T) + 16 * lh + 4 * j);
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[h][4 * j + i] = b[i];
          }
#pragma unroll
        for (int s = 0; s < KS; ++s) {
          const bf16x8 a0 = *reinterpret_cast<const bf16x8*>(w0 + s * 1024), a1 = *reinterpret_cast<const bf16x8*>(w1 + s * 1024);
          acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a0, hi[s], acc[0], 0, 0, 0);
          acc[1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a1, hi[s], acc[1], 0, 0, 0);
          if constexpr (SPLIT) {
            acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a0, lo[s], acc[0], 0, 0, 0);
            acc[1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a1, lo[s], acc[1], 0, 0, 0);
          }
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int c = 32 * (h ? T1 : T) + 16 * lh;
          unsigned char* op = st + lp * st_row + c * 2;
          if (c + 8 <= N)
            *reinterpret_cast<u32x4*>(op) = u32x4{pack2_bf16(acc[h][0], acc[h][1]), pack2_bf16(acc[h][2], acc[h][3]),
                                                  pack2_bf16(acc[h][4], acc[h][5]), pack2_bf16(acc[h][6], acc[h][7])};
          if (c + 16 <= N)
            *reinterpret_cast<u32x4*>(op + 16) = u32x4{pack2_bf16(acc[h][8], acc[h][9]), pack2_bf16(acc[h][10], acc[h][11]),
                                                       pack2_bf16(acc[h][12], acc[h][13]), pack2_bf16(acc[h][14], acc[h][15])};
        }
      }
      unsigned char* op = (unsigned char*)p.c + t * 32 * st_row;
      const int bytes = (int)min((int64_t)32, p.m - t * 32) * st_row;
      for (int i = lane * 16; i < bytes; i += 1024)
        *reinterpret_cast<u32x4*>(op + i) = *reinterpret_cast<const u32x4*>(st + i);
      continue;
    }
    // ---- channel tiles
    for (int T = 0; T < (LIN ? 0 : nt); ++T) {
      const int c0 = n0 + 32 * T + 16 * lh;  // the lane's 16 channels
      const int left = N - c0;               // of which this many exist (a multiple of 8)
      f32x16 acc;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const f32x4 b = *reinterpret_cast<const f32x4*>(bl + 32 * T + 16 * lh + 4 * j);
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[4 * j + i] = b[i];
      }
      u32x4 rr[4];
      if (p.has_res) {
        const int64_t ro = q * p.ldr + c0;
        if (p.r_dt == DT_BF16) {
#pragma unroll
          for (int j = 0; j < 2; ++j)
            rr[j] = live && left >= 8 * (j + 1) ? *reinterpret_cast<const u32x4*>((const unsigned short*)p.res + ro + 8 * j)
                                                : u32x4{0u, 0u, 0u, 0u};
        } else {
#pragma unroll
          for (int j = 0; j < 4; ++j)
            rr[j] = live && left >= 4 * (j + 1) ? *reinterpret_cast<const u32x4*>((const float*)p.res + ro + 4 * j)
                                                : u32x4{0u, 0u, 0u, 0u};
        }
      }
      const unsigned char* wt = wl + ((size_t)T * KS * 64 + lane) * 16;
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const bf16x8 w = *reinterpret_cast<const bf16x8*>(wt + s * 1024);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w, hi[s], acc, 0, 0, 0);
        if constexpr (SPLIT) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w, lo[s], acc, 0, 0, 0);
      }
      float v[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) v[i] = acc[i];
      if (p.act == ACT_GELU) {
#pragma unroll
        for (int i = 0; i < 16; ++i) v[i] = gelu_erf(v[i]);
      }
      if (!plain) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const f32x4 sc = *reinterpret_cast<const f32x4*>(sl + 32 * T + 16 * lh + 4 * j);
#pragma unroll
          for (int i = 0; i < 4; ++i) v[4 * j + i] *= sc[i];
        }
      }
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
      if (p.c_dt == DT_BF16) {
        const u32x4 o0 = u32x4{pack2_bf16(v[0], v[1]), pack2_bf16(v[2], v[3]), pack2_bf16(v[4], v[5]), pack2_bf16(v[6], v[7])};
        const u32x4 o1 = u32x4{pack2_bf16(v[8], v[9]), pack2_bf16(v[10], v[11]), pack2_bf16(v[12], v[13]), pack2_bf16(v[14], v[15])};
        unsigned char* op = st + lp * RW_ST_ROW + (T & 1) * 64 + lh * 32;
        *reinterpret_cast<u32x4*>(op) = o0;
        *reinterpret_cast<u32x4*>(op + 16) = o1;
        if (!(T & 1) && T + 1 < nt) continue;
        const int seg = lane & 7, cs = n0 + 32 * (T & ~1) + 8 * seg;
        const bool cok = cs < N && (seg < 4 || (T & 1));
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int px = 8 * j + (lane >> 3);
          const u32x4 w = *reinterpret_cast<const u32x4*>(st + px * RW_ST_ROW + seg * 16);
          const int64_t qq = t * 32 + px;
          if (cok && qq < p.m) *reinterpret_cast<u32x4*>((unsigned short*)p.c + qq * p.ldc + cs) = w;
        }
      } else if (live) {
        float* op = (float*)p.c + q * p.ldc + c0;
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (left >= 4 * (j + 1))
            *reinterpret_cast<f32x4*>(op + 4 * j) = f32x4{v[4 * j], v[4 * j + 1], v[4 * j + 2], v[4 * j + 3]};
      }
    }
  }
}

// dynamic LDS of a workgroup: W^T, vectors, the four waves' store tiles
template <int KS, bool LIN>
int rw_lds(int ntc, int n) {
  return ntc * KS * 1024 + (64 * ntc + 32 * KS) * 4 + 4 * 32 * (LIN ? n * 2 : RW_ST_ROW);
}

template <int PRO, int TA, int KS, bool LIN>
void launch_rw(RwP& p, hipStream_t s) {
  auto fn = &gemm_rowwide_kernel<PRO, TA, KS, LIN>;
  static const bool set = [&] {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize, RW_LDS_MAX);
    return true;
  }();
  (void)set;
  const GemmP& g = p.g;
  const int lds = rw_lds<KS, LIN>(p.ntc, (int)g.n);
  static OccupancyMemo occ;
  const int per_cu = occ.get(reinterpret_cast<const void*>(fn), 256, lds);
  const int64_t cap = std::max<int64_t>(1, (int64_t)device_cus() * per_cu / (8 * p.nch));
  const int64_t groups = std::min<int64_t>(cdiv(cdiv(g.m, 32), 4 * 8), cap);  // workgroups per XCD and chunk
  note_kernel("gemm_rowwide_kernel pro=%d a=%s ks=%d tiles=%d chunks=%d lin=%d", g.pro, TA == DT_BF16 ? "bf16" : "f32",
              KS, p.ntc, p.nch, (int)LIN);
  hipLaunchKernelGGL(fn, dim3((unsigned)(8 * p.nch * groups)), dim3(256), lds, s, p);
}

template <int PRO, int TA, int KS>
void choose_rw(const GemmP& g, hipStream_t s) {
  RwP p{};
  p.g = g;
  const int64_t cus = device_cus();
  const int nt = (int)cdiv(g.n, 32);
  const int most = RW_W_MAX / (KS * 1024) & ~1;  // an even count: chunks start on 128-byte lines of the row
  if constexpr (TA == DT_BF16 && KS <= 4) {
    // rows whose length is no multiple of 128 bytes: stored tile by tile as one run, so that no 128-byte line
    // is written in two parts (us, 720 x 1280, K = 48: N = 288 174 -> 142, N = 144 93 -> 85); the tile's store
    // buffer takes LDS, which costs more than it gives at K = 96 (360 x 640, N = 288: 48 -> 61) and where the
    // row groups alone leave CUs idle. The store tiles of four waves have to fit LDS beside W^T (K = 48: N < 456)
    if (nt <= most && rw_lds<KS, true>(nt, (int)g.n) <= RW_LDS_MAX && g.c_dt == DT_BF16 && g.ldc == g.n &&
        g.n % 64 != 0 && g.n > 64 && !g.has_res && g.act == ACT_NONE && !g.scale && g.out_scale == 1.0f && cdiv(g.m, 128) >= cus) {
      p.nch = 1;
      p.ntc = nt;
      return launch_rw<PRO, TA, KS, true>(p, s);
    }
  }
  // channel chunks: as few as LDS allows, one more where that deals the tiles out evenly (18 tiles as 3 x 6,
  // not 10 + 8), and more of them while the row groups leave CUs idle (50 x 60 rows, K = 96, N = 512)
  auto even = [&](int nch) { return (int)cdiv(nt, 2 * nch) * 2; };
  int nch = (int)cdiv(nt, most);
  if (even(nch + 1) * (nch + 1) < even(nch) * nch) ++nch;
  while (cdiv(g.m, 128) * nch < cus && even(nch) > 2) ++nch;
  p.ntc = nch == 1 ? nt : even(nch);
  p.nch = (int)cdiv(nt, p.ntc);
  launch_rw<PRO, TA, KS, false>(p, s);
}

template <int PRO, int TA>
bool pick_rw(const GemmP& g, hipStream_t s) {
  switch ((g.k + 15) / 16) {
    case 2: choose_rw<PRO, TA, 2>(g, s); return true;
    case 3: choose_rw<PRO, TA, 3>(g, s); return true;
    case 4: choose_rw<PRO, TA, 4>(g, s); return true;
    case 5: choose_rw<PRO, TA, 5>(g, s); return true;
    case 6: choose_rw<PRO, TA, 6>(g, s); return true;
    default: return false;
  }
}

}  // namespace

bool gemm_rowwide_fits(const GemmP& p, int a_dt, int w_dt) {
  if (w_dt != DT_BF16 || p.k <= 16 || p.k > 96 || p.n % 8 || p.n > (1 << 20) || p.vec_out != 2 ||
      (p.has_res && p.vec_res != 2) || (p.act != ACT_NONE && p.act != ACT_GELU) || p.c_mode != CM_ROWS)
    return false;
  if (p.pro == PRO_LNMUL) return a_dt == DT_F32 && p.m2_dt == DT_BF16;
  return a_dt == DT_BF16 && (p.pro == PRO_NONE || p.pro == PRO_LN || p.pro == PRO_RMS);
}

bool launch_gemm_rowwide(const GemmP& p, int a_dt, hipStream_t s) {
  if (p.pro == PRO_LNMUL) return pick_rw<PRO_LNMUL, DT_F32>(p, s);
  if (p.pro == PRO_NONE) return pick_rw<PRO_NONE, DT_BF16>(p, s);
  return pick_rw<PRO_LN, DT_BF16>(p, s);
}

}  // namespace clarus
