// Kernels of the decoder layer around the paged attention for gfx950: RMSNorm (with the
// residual add before it), SwiGLU, and linear layers on a few rows (a decode step's one
// token per sequence) with the norm, the residual add or SwiGLU fused in.
//
// All of them are bound by memory or, on a few rows, by latency:
//   rms_norm / swiglu  one pass over their operands, 16 bytes per lane and access; the
//                      formulas as torch operators take nine and two passes.
//   linear_rows        streams each weight matrix once.  On 1 .. 64 rows a library GEMM is
//                      set by its launch and its serial walk along K; here the waves of a
//                      workgroup split K, so every weight load of a wave is in flight at
//                      once, and q / k / v, or gate / up, go in one launch.
#include <string.h>

#include "ivakv_tile.h"

namespace ivakv {
namespace {

template <int DT>
__device__ inline void unpack8(const Chunk16& c, float (&f)[8]) {
  using E = typename Traits<DT>::E;
  typedef E E8 __attribute__((ext_vector_type(8)));
  const E8 e = __builtin_bit_cast(E8, c);
#pragma unroll
  for (int i = 0; i < 8; ++i) f[i] = (float)e[i];
}

template <int DT>
__device__ inline Chunk16 pack8(const float (&f)[8]) {
  Chunk16 c;
#pragma unroll
  for (int i = 0; i < 4; ++i) c.w[i] = Traits<DT>::pack2(f[2 * i], f[2 * i + 1]);
  return c;
}

// x rounded to the element type, as a float.
template <int DT>
__device__ inline float round_e(float x) {
  return (float)Traits<DT>::from_float(x);
}

__device__ inline float wave_sum(float v) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o);
  return v;
}

// silu(u) * g, rounded once by the caller.
__device__ inline float silu_mul(float u, float g) {
  return u * __builtin_amdgcn_rcpf(1.f + exp2_fast(-1.4426950408889634f * u)) * g;
}

// ---------------------------------------------------------------------------
// RMSNorm
// ---------------------------------------------------------------------------

// A wave normalizes one row of NC * 64 16-byte chunks (chunks past the row are masked):
// out = round(round(x / sqrt(mean(x^2) + eps)) * w), with x = round(x + residual) first
// when there is a residual, stored to `sum`.  The row stays in registers between the sum
// of squares and the store, so it is read once.  8192 rows of 1024 (bf16, from HBM): 8.2 us =
// 4.1 TB/s against 66 us for nine torch operators, with the residual 13.5 us = 5.0 TB/s against
// 74 us for ten; 16 rows 2.8 us (launch and one round trip) against 24 us.
template <int DT, int NC>
__global__ __launch_bounds__(256) void rms_norm_kernel(const void* x, const void* residual,
                                                       const void* weight, void* sum, void* out,
                                                       int64_t rows, int d, float eps) {
  using E = typename Traits<DT>::E;
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  const int n = d >> 3;
  const int64_t base = row * d;
  Chunk16 cx[NC], cr[NC], cw[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int64_t o = base + 8 * min(lane + 64 * c, n - 1);
    cx[c] = *reinterpret_cast<const Chunk16*>(static_cast<const E*>(x) + o);
    if (residual) cr[c] = *reinterpret_cast<const Chunk16*>(static_cast<const E*>(residual) + o);
  }
#pragma unroll
  for (int c = 0; c < NC; ++c)
    if (weight)
      cw[c] = *reinterpret_cast<const Chunk16*>(static_cast<const E*>(weight) +
                                                8 * min(lane + 64 * c, n - 1));
  float f[NC][8];
  float ss = 0.f;
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    unpack8<DT>(cx[c], f[c]);
    const bool in = lane + 64 * c < n;
    if (residual) {
      float r[8];
      unpack8<DT>(cr[c], r);
#pragma unroll
      for (int i = 0; i < 8; ++i) f[c][i] = round_e<DT>(f[c][i] + r[i]);
      if (in)
        *reinterpret_cast<Chunk16*>(static_cast<E*>(sum) + base + 8 * (lane + 64 * c)) = pack8<DT>(f[c]);
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) ss += in ? f[c][i] * f[c][i] : 0.f;
  }
  const float inv = 1.f / sqrtf(wave_sum(ss) / (float)d + eps);
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    if (lane + 64 * c >= n) continue;
    float y[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) y[i] = f[c][i] * inv;
    if (weight) {
      float w[8];
      unpack8<DT>(cw[c], w);
#pragma unroll
      for (int i = 0; i < 8; ++i) y[i] = round_e<DT>(y[i]) * w[i];
    }
    *reinterpret_cast<Chunk16*>(static_cast<E*>(out) + base + 8 * (lane + 64 * c)) = pack8<DT>(y);
  }
}

constexpr int kNormMaxChunks = 16;  // per lane: rows of up to 8192 elements

template <int DT>
void launch_rms_norm(const void* x, const void* residual, const void* weight, void* sum, void* out,
                     int64_t rows, int d, float eps, hipStream_t stream) {
  const dim3 grid((unsigned)((rows + 3) / 4));
  const int nc = cdiv(d >> 3, 64);
#define IVAKV_NORM(NC)                                                                           \
  rms_norm_kernel<DT, NC><<<grid, 256, 0, stream>>>(x, residual, weight, sum, out, rows, d, eps)
  if (nc <= 1) IVAKV_NORM(1);
  else if (nc <= 2) IVAKV_NORM(2);
  else if (nc <= 4) IVAKV_NORM(4);
  else if (nc <= 8) IVAKV_NORM(8);
  else IVAKV_NORM(kNormMaxChunks);
#undef IVAKV_NORM
}

// ---------------------------------------------------------------------------
// SwiGLU
// ---------------------------------------------------------------------------

// out = silu(up) * gate over n8 16-byte chunks: each thread takes two chunks, 256 apart so that
// a wave's accesses stay contiguous, all four loads before the first store.  8192 x 4096
// bf16: 30 - 32 us = 6.3 - 6.6 TB/s against 61 - 64 us for silu and product as two torch
// operators.
template <int DT>
__global__ __launch_bounds__(256) void swiglu_kernel(const Chunk16* up, const Chunk16* gate,
                                                     Chunk16* out, int64_t n8) {
  const int64_t i0 = (int64_t)blockIdx.x * 512 + threadIdx.x, i1 = i0 + 256;
  if (i0 >= n8) return;
  const bool two = i1 < n8;
  const int64_t j1 = two ? i1 : i0;
  const Chunk16 u0 = up[i0], u1 = up[j1], g0 = gate[i0], g1 = gate[j1];
  auto one = [&](const Chunk16& uc, const Chunk16& gc) IVAKV_INLINE -> Chunk16 {
    float u[8], g[8];
    unpack8<DT>(uc, u);
    unpack8<DT>(gc, g);
#pragma unroll
    for (int i = 0; i < 8; ++i) u[i] = silu_mul(u[i], g[i]);
    return pack8<DT>(u);
  };
  out[i0] = one(u0, g0);
  if (two) out[i1] = one(u1, g1);
}

// ---------------------------------------------------------------------------
// Linear layers on a few rows
// ---------------------------------------------------------------------------

constexpr int kLinearBlocks = 4;  // blocks of 64 k in one load set of a wave

// How linear_rows normalizes its rows: not, into LDS before the products, or by scaling the
// sums after them.
enum Norm { kNoNorm = 0, kNormLds = 1, kNormFold = 2 };

enum Epilogue { kPlain = 0, kResidual = 1, kSwiglu = 2 };

struct LinearArgs {
  const void* x;        // [m][ldx]
  int64_t ldx;
  int m, k;
  const void* w[3];     // [n][k] each
  void* out[3];         // [m][n] each
  int n[3];
  int t0, t1, tiles;    // 16-column tiles of w[0], of w[0] and w[1], of all (kSwiglu: of one)
  const void* residual; // [m][n[0]] (kResidual)
  const void* norm_w;   // [k] or null
  float eps;
};

// y[m][n] = x[m][k] . w[n][k]^T on MT tiles of 16 rows.  A workgroup computes tiles of 16
// columns (kSwiglu: the tile of gate and of up) a grid apart, its WAVES waves each a
// contiguous part of k in blocks of 64: per block and lane (ln = column, lq) two 16-byte
// chunks at k = 16 lq and 16 lq + 8, so a column's 128 bytes are read by four lanes side by
// side; the rows use the same order of k, which a sum does not see.  w is the MFMA's A
// operand, x its B operand, so lane (ln, lq) ends with columns 4 lq .. 4 lq + 3 of row ln.
// The waves' sums meet in LDS in a fixed order.
//
// ONE: a wave's part of k is one load set (k <= 64 U WAVES), so its part of x stays in
// registers for all its tiles and the next tile's weights are loaded before this tile's
// sums meet.  Otherwise the sets alternate along k and x is read again (L2) per tile.
//
// NORM (MT 1): x is RMS-normalized, each workgroup for itself (the rows are L2 hits).
//   kNormLds   into LDS rows of k + 8 elements (the pad spreads the rows over the banks), the
//              wave's first weight loads issued before that.
//   kNormFold  (bf16) the products take x * norm_w, rounded once, and the sums are scaled by
//              the rows' 1 / rms at the end; each wave sums the squares of its part of k, so
//              nothing waits for whole rows.  16 rows: q / k / v 7.0 -> 5.5 us, gate / up 9.0 ->
//              7.1; one row 4.3 -> 4.8 and 6.0 -> 6.6, so up to kNormLdsRows rows stay with LDS.
//              In fp16 the product could overflow where the normalized row does not.
//
// 16 rows, bf16, weights from HBM, against the library's products (us): q / k / v (3 x 1024
// x 1024) 4.6, with the norm 5.5, against 3 x 5.6; 1024 x 1024 with residual 4.0 against
// 5.6 + 2.4; gate / up (2 x 4096 x 1024) with norm and SwiGLU 7.1 against 2 x 7.6 + 5.2 + 21;
// 1024 x 4096 10.3 against 14.4 (64 column tiles reach 64 CUs, whose loads bound it: 7.6 at
// one row); 32000 x 1024 18.3 against 19.3.
template <int DT, int MT, int WAVES, int NORM, int EPI, bool ONE>
__global__ __launch_bounds__(64 * WAVES) void linear_rows_kernel(LinearArgs a) {
  using Tr = Traits<DT>;
  using E = typename Tr::E;
  constexpr int NT = EPI == kSwiglu ? 2 : 1;
  constexpr int U = kLinearBlocks;
  constexpr int NCN = WAVES / 2;    // norm: 16-byte chunks of a row per lane (k <= 256 WAVES)
  constexpr bool FOLD = NORM == kNormFold;
  constexpr bool NORM_LDS = NORM == kNormLds;
  static_assert(!FOLD || (ONE && MT == 1), "the folded norm keeps its rows in registers");
  extern __shared__ Chunk16 smem[];
  const int lane = threadIdx.x & 63, ln = lane & 15, lq = lane >> 4;
  const int wave = uni(threadIdx.x >> 6);
  const int k = a.k, m = a.m;
  const int nb = k >> 6;
  const int per = (nb + WAVES - 1) / WAVES;
  const int b0 = wave * per, b1 = min(b0 + per, nb);
  const int last = max(b1 - 1, 0);

  // Matrix and column tile of flat tile t.
  auto locate = [&](int t, int& seg, int& tile) IVAKV_INLINE {
    seg = 0;
    tile = t;
    if constexpr (EPI == kPlain) {
      if (t >= a.t1) {
        tile = t - a.t1;
        seg = 2;
      } else if (t >= a.t0) {
        tile = t - a.t0;
        seg = 1;
      }
    }
  };
  Chunk16 wv[2][NT][U][2];
  auto load_w = [&](int set, int t, int b) IVAKV_INLINE {
    int seg, tile;
    locate(t, seg, tile);
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const E* wp = static_cast<const E*>(a.w[NT == 2 ? j : seg]) + (int64_t)(16 * tile + ln) * k + 16 * lq;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const E* p = wp + 64 * min(b + u, last);
        wv[set][j][u][0] = load_nt<Chunk16>(p);
        wv[set][j][u][1] = load_nt<Chunk16>(p + 8);
      }
    }
  };
  if constexpr (!FOLD) load_w(0, blockIdx.x, b0);

  const int xs = k + 8;  // LDS row of the normalized x
  if constexpr (NORM_LDS) {
    E* xn = reinterpret_cast<E*>(smem);
    const int n8 = k >> 3;
    for (int r = wave; r < m; r += WAVES) {
      const E* xr = static_cast<const E*>(a.x) + r * a.ldx;
      Chunk16 cx[NCN], cw[NCN];
#pragma unroll
      for (int c = 0; c < NCN; ++c) {
        const int i = 8 * min(lane + 64 * c, n8 - 1);
        cx[c] = *reinterpret_cast<const Chunk16*>(xr + i);
        if (a.norm_w) cw[c] = *reinterpret_cast<const Chunk16*>(static_cast<const E*>(a.norm_w) + i);
      }
      float f[NCN][8], ss = 0.f;
#pragma unroll
      for (int c = 0; c < NCN; ++c) {
        unpack8<DT>(cx[c], f[c]);
#pragma unroll
        for (int i = 0; i < 8; ++i) ss += lane + 64 * c < n8 ? f[c][i] * f[c][i] : 0.f;
      }
      const float inv = 1.f / sqrtf(wave_sum(ss) / (float)k + a.eps);
#pragma unroll
      for (int c = 0; c < NCN; ++c) {
        if (lane + 64 * c >= n8) continue;
#pragma unroll
        for (int i = 0; i < 8; ++i) f[c][i] *= inv;
        if (a.norm_w) {
          float wn[8];
          unpack8<DT>(cw[c], wn);
#pragma unroll
          for (int i = 0; i < 8; ++i) f[c][i] = round_e<DT>(f[c][i]) * wn[i];
        }
        *reinterpret_cast<Chunk16*>(xn + r * xs + 8 * (lane + 64 * c)) = pack8<DT>(f[c]);
      }
    }
    __syncthreads();
  }

  const E* xp[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const int r = min(16 * t + ln, m - 1);  // rows past m repeat the last; never stored
    xp[t] = NORM_LDS ? reinterpret_cast<const E*>(smem) + r * xs + 16 * lq
                 : static_cast<const E*>(a.x) + r * a.ldx + 16 * lq;
  }
  f32x4 acc[MT][NT];
  Chunk16 xv[ONE ? MT : 1][U][2];
  auto load_x = [&](int t, int b) IVAKV_INLINE {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const E* p = xp[t] + 64 * min(b + u, last);
      xv[ONE ? t : 0][u][0] = *reinterpret_cast<const Chunk16*>(p);
      xv[ONE ? t : 0][u][1] = *reinterpret_cast<const Chunk16*>(p + 8);
    }
  };
  auto compute = [&](int set, int b) IVAKV_INLINE {
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      if constexpr (!ONE) load_x(t, b);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (b + u >= b1) continue;
#pragma unroll
        for (int j = 0; j < NT; ++j) {
          acc[t][j] = Tr::qk(wv[set][j][u][0], xv[ONE ? t : 0][u][0], acc[t][j]);
          acc[t][j] = Tr::qk(wv[set][j][u][1], xv[ONE ? t : 0][u][1], acc[t][j]);
        }
      }
    }
  };
  if constexpr (ONE) {
#pragma unroll
    for (int t = 0; t < MT; ++t) load_x(t, b0);
  }
  Chunk16 nw[FOLD ? U : 1][2];
  if constexpr (FOLD) {
    load_w(0, blockIdx.x, b0);
    if (a.norm_w) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const E* p = static_cast<const E*>(a.norm_w) + 16 * lq + 64 * min(b0 + u, last);
        nw[u][0] = *reinterpret_cast<const Chunk16*>(p);
        nw[u][1] = *reinterpret_cast<const Chunk16*>(p + 8);
      }
    }
  }

  // Sums over the waves, in two LDS buffers used in turn (one barrier per tile): tile t of
  // the rows by wave t.  With NORM they lie behind the normalized rows or the rows' sums of
  // squares.
  f32x4* red0 = reinterpret_cast<f32x4*>(smem) + (NORM_LDS ? (m * xs + 7) / 8 : FOLD ? 4 * WAVES : 0);
  float* s_ss = reinterpret_cast<float*>(smem);  // FOLD: [WAVES][16]
  if constexpr (FOLD) {
    float ss = 0.f;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      float part = 0.f;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const bf16x2 x2 = __builtin_bit_cast(bf16x2, xv[0][u][j].w[i]);
          part = __builtin_amdgcn_fdot2_f32_bf16(x2, x2, part, false);  // exact products, fp32 sum
          if (a.norm_w) {
            const bf16x2 w2 = __builtin_bit_cast(bf16x2, nw[u][j].w[i]);
            xv[0][u][j].w[i] = Tr::pack2((float)x2[0] * (float)w2[0], (float)x2[1] * (float)w2[1]);
          }
        }
      }
      ss += b0 + u < b1 ? part : 0.f;
    }
    ss += __shfl_xor(ss, 16);
    ss += __shfl_xor(ss, 32);
    if (lane < 16) s_ss[wave * 16 + lane] = ss;  // (published by the first sums' barrier)
  }
  auto finish = [&](int par, int t_flat) IVAKV_INLINE {
    f32x4* red = red0 + par * (MT * NT * WAVES * 64);
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int j = 0; j < NT; ++j) red[((t * NT + j) * WAVES + wave) * 64 + lane] = acc[t][j];
    __syncthreads();
    const int row = 16 * wave + ln;
    if (wave >= MT || row >= m) return;
    f32x4 s[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      s[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int u = 0; u < WAVES; ++u) s[j] += red[((wave * NT + j) * WAVES + u) * 64 + lane];
    }
    if constexpr (FOLD) {
      float ss = 0.f;
#pragma unroll
      for (int u = 0; u < WAVES; ++u) ss += s_ss[u * 16 + ln];
      const float inv = 1.f / sqrtf(ss / (float)k + a.eps);
#pragma unroll
      for (int j = 0; j < NT; ++j) s[j] *= inv;
    }
    int seg, tile;
    locate(t_flat, seg, tile);
    const int n = a.n[seg], col = 16 * tile + 4 * lq;
    if constexpr (EPI == kSwiglu) {
#pragma unroll
      for (int r = 0; r < 4; ++r) s[0][r] = silu_mul(s[1][r], s[0][r]);
    }
    if constexpr (EPI == kResidual) {
      typedef E E4 __attribute__((ext_vector_type(4)));
      const E4 rs = *reinterpret_cast<const E4*>(static_cast<const E*>(a.residual) + (int64_t)row * n + col);
#pragma unroll
      for (int r = 0; r < 4; ++r) s[0][r] += (float)rs[r];
    }
    Chunk8 o;
    o.w[0] = Tr::pack2(s[0][0], s[0][1]);
    o.w[1] = Tr::pack2(s[0][2], s[0][3]);
    *reinterpret_cast<Chunk8*>(static_cast<E*>(a.out[seg]) + (int64_t)row * n + col) = o;
  };
  auto clear = [&]() IVAKV_INLINE {
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int j = 0; j < NT; ++j) acc[t][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  };

  const int step = gridDim.x;
  if constexpr (ONE) {
    for (int t = blockIdx.x; t < a.tiles; t += 2 * step) {
      clear();
      if (t + step < a.tiles) load_w(1, t + step, b0);
      compute(0, b0);
      finish(0, t);
      if (t + step < a.tiles) {
        clear();
        if (t + 2 * step < a.tiles) load_w(0, t + 2 * step, b0);
        compute(1, b0);
        finish(1, t + step);
      }
    }
  } else {
    int par = 0;
    for (int t = blockIdx.x; t < a.tiles; t += step, par ^= 1) {
      clear();
      if (t != (int)blockIdx.x) load_w(0, t, b0);
      for (int b = b0; b < b1; b += 2 * U) {
        if (b + U < b1) load_w(1, t, b + U);
        compute(0, b);
        if (b + U < b1) {
          if (b + 2 * U < b1) load_w(0, t, b + 2 * U);
          compute(1, b + U);
        }
      }
      finish(par, t);
    }
  }
}

constexpr int kLinearMaxRows = 32;
constexpr int kLinearNormRows = 16;
constexpr int kLinearNormMaxK = 2048;
constexpr int kNormLdsRows = 4;

// Workgroups of a launch, each taking tiles a grid apart: four of 4 waves per CU, or two of 8.
// The CUs hold that many at once in the plain and residual instances; the SwiGLU ones (two
// matrices' loads in registers) run at half of it, and the rest follow as those end.
constexpr int kLinearWaves = 256 * 16;

template <int DT, int MT, int WAVES, int NORM, int EPI, bool ONE>
void launch_linear_one(const LinearArgs& a, hipStream_t stream) {
  size_t smem = (size_t)2 * MT * (EPI == kSwiglu ? 2 : 1) * WAVES * 64 * sizeof(f32x4);
  if (NORM == kNormLds) smem += ((size_t)a.m * (a.k + 8) + 7) / 8 * 16;
  if (NORM == kNormFold) smem += (size_t)64 * WAVES;
  if (smem > 64 * 1024) {  // (the size depends on m and k: the whole LDS is asked for)
    static std::atomic<uint64_t> done{0};
    allow_lds(reinterpret_cast<const void*>(&linear_rows_kernel<DT, MT, WAVES, NORM, EPI, ONE>),
              160 * 1024, done);
  }
  const int wgs = a.tiles < kLinearWaves / WAVES ? a.tiles : kLinearWaves / WAVES;
  linear_rows_kernel<DT, MT, WAVES, NORM, EPI, ONE><<<dim3((unsigned)wgs), 64 * WAVES, smem, stream>>>(a);
}

template <int DT, int MT, int WAVES, int NORM, int EPI>
void launch_linear(const LinearArgs& a, hipStream_t stream) {
  if (NORM || (MT == 1 && a.k <= 64 * kLinearBlocks * WAVES))
    launch_linear_one<DT, MT, WAVES, NORM, EPI, MT == 1>(a, stream);
  else
    launch_linear_one<DT, MT, WAVES, NORM, EPI, NORM != kNoNorm>(a, stream);
}

template <int DT, int MT, int WAVES, int NORM>
void launch_linear_e(const LinearArgs& a, int epi, hipStream_t stream) {
  if (epi == kSwiglu) launch_linear<DT, MT, WAVES, NORM, kSwiglu>(a, stream);
  else if (epi == kPlain) launch_linear<DT, MT, WAVES, NORM, kPlain>(a, stream);
  else if constexpr (NORM == kNoNorm) launch_linear<DT, MT, WAVES, NORM, kResidual>(a, stream);
}

template <int DT, int WAVES>
void launch_linear_m(const LinearArgs& a, bool norm, int epi, hipStream_t stream) {
  if (norm && DT == IVAKV_BF16 && a.m > kNormLdsRows)
    launch_linear_e<DT, 1, WAVES, DT == IVAKV_BF16 ? kNormFold : kNormLds>(a, epi, stream);
  else if (norm) launch_linear_e<DT, 1, WAVES, kNormLds>(a, epi, stream);
  else if (a.m <= 16) launch_linear_e<DT, 1, WAVES, kNoNorm>(a, epi, stream);
  else launch_linear_e<DT, 2, WAVES, kNoNorm>(a, epi, stream);
}

template <int DT>
void launch_linear_w(const LinearArgs& a, bool norm, int epi, hipStream_t stream) {
  if (a.k <= 1024) launch_linear_m<DT, 4>(a, norm, epi, stream);
  else launch_linear_m<DT, 8>(a, norm, epi, stream);
}

int check_16bit(const char* name, int dtype) {
  if (dtype != IVAKV_F16 && dtype != IVAKV_BF16)
    return fail(IVAKV_E_DTYPE, "%s: takes fp16 or bf16 (dtype %d)", name, dtype);
  return IVAKV_OK;
}

}  // namespace
}  // namespace ivakv

using namespace ivakv;

extern "C" int ivakv_rms_norm(const void* x, const void* residual, const void* weight, void* sum,
                              void* out, int64_t rows, int d, float eps, int dtype,
                              hipStream_t stream) {
  const char* name = "ivakv_rms_norm";
  const int st = check_16bit(name, dtype);
  if (st != IVAKV_OK) return st;
  if (rows < 0 || d <= 0) return fail(IVAKV_E_ARG, "%s: bad sizes rows=%lld d=%d", name, (long long)rows, d);
  if (d % 8 != 0 || d > 512 * kNormMaxChunks)
    return fail(IVAKV_E_SHAPE, "%s: d %d must be a multiple of 8 up to %d", name, d, 512 * kNormMaxChunks);
  if ((rows + 3) / 4 > 0x7fffffff) return fail(IVAKV_E_SHAPE, "%s: launch too large", name);
  if (rows == 0) return IVAKV_OK;
  if (!x || !out || (residual && !sum)) return fail(IVAKV_E_ARG, "%s: null pointer argument", name);
  if (!aligned16(x) || !aligned16(out) || !aligned16(residual) || !aligned16(weight) || !aligned16(sum))
    return fail(IVAKV_E_ARG, "%s: pointers must be 16-byte aligned", name);
  if (dtype == IVAKV_F16) launch_rms_norm<IVAKV_F16>(x, residual, weight, sum, out, rows, d, eps, stream);
  else launch_rms_norm<IVAKV_BF16>(x, residual, weight, sum, out, rows, d, eps, stream);
  return launch_status(name);
}

extern "C" int ivakv_swiglu(const void* up, const void* gate, void* out, int64_t n, int dtype,
                            hipStream_t stream) {
  const char* name = "ivakv_swiglu";
  const int st = check_16bit(name, dtype);
  if (st != IVAKV_OK) return st;
  if (n < 0) return fail(IVAKV_E_ARG, "%s: bad size %lld", name, (long long)n);
  if (n % 8 != 0) return fail(IVAKV_E_SHAPE, "%s: n %lld must be a multiple of 8", name, (long long)n);
  const int64_t n8 = n / 8, wgs = (n8 + 511) / 512;
  if (wgs > 0x7fffffff) return fail(IVAKV_E_SHAPE, "%s: launch too large", name);
  if (n == 0) return IVAKV_OK;
  if (!up || !gate || !out) return fail(IVAKV_E_ARG, "%s: null pointer argument", name);
  if (!aligned16(up) || !aligned16(gate) || !aligned16(out))
    return fail(IVAKV_E_ARG, "%s: pointers must be 16-byte aligned", name);
  const Chunk16* u = static_cast<const Chunk16*>(up);
  const Chunk16* g = static_cast<const Chunk16*>(gate);
  Chunk16* o = static_cast<Chunk16*>(out);
  if (dtype == IVAKV_F16) swiglu_kernel<IVAKV_F16><<<dim3((unsigned)wgs), 256, 0, stream>>>(u, g, o, n8);
  else swiglu_kernel<IVAKV_BF16><<<dim3((unsigned)wgs), 256, 0, stream>>>(u, g, o, n8);
  return launch_status(name);
}

extern "C" int ivakv_linear_rows(const void* x, int64_t ldx, int m, int k, const void* w0, int n0,
                                 void* out0, const void* w1, int n1, void* out1, const void* w2,
                                 int n2, void* out2, const void* residual, int norm,
                                 const void* norm_weight, float eps, int epilogue, int dtype,
                                 hipStream_t stream) {
  const char* name = "ivakv_linear_rows";
  const int st = check_16bit(name, dtype);
  if (st != IVAKV_OK) return st;
  if (m < 0 || k <= 0 || n0 <= 0 || n1 < 0 || n2 < 0 || ldx < k || epilogue < kPlain || epilogue > kSwiglu)
    return fail(IVAKV_E_ARG, "%s: bad sizes m=%d k=%d n=%d,%d,%d ldx=%lld epilogue=%d", name, m, k, n0,
                n1, n2, (long long)ldx, epilogue);
  if (m > kLinearMaxRows || k % 64 != 0 || n0 % 16 != 0 || n1 % 16 != 0 || n2 % 16 != 0 || ldx % 8 != 0)
    return fail(IVAKV_E_SHAPE, "%s: takes m <= %d rows, k in multiples of 64, n of 16, ldx of 8 "
                "(m=%d k=%d n=%d,%d,%d ldx=%lld)", name, kLinearMaxRows, m, k, n0, n1, n2, (long long)ldx);
  if (norm && (m > kLinearNormRows || k > kLinearNormMaxK || epilogue == kResidual))
    return fail(IVAKV_E_SHAPE, "%s: the fused norm takes m <= %d, k <= %d and no residual (m=%d k=%d)",
                name, kLinearNormRows, kLinearNormMaxK, m, k);
  if (n2 > 0 && n1 == 0) return fail(IVAKV_E_ARG, "%s: a third matrix without a second", name);
  if (epilogue == kSwiglu && (n1 != n0 || n2 != 0))
    return fail(IVAKV_E_SHAPE, "%s: SwiGLU takes two matrices of one size", name);
  if (epilogue == kResidual && n1 != 0) return fail(IVAKV_E_SHAPE, "%s: a residual takes one matrix", name);
  if (m == 0) return IVAKV_OK;
  if (!x || !w0 || !out0 || (n1 && (!w1 || (!out1 && epilogue != kSwiglu))) || (n2 && (!w2 || !out2)) ||
      (epilogue == kResidual && !residual))
    return fail(IVAKV_E_ARG, "%s: null pointer argument", name);
  if (!aligned16(x) || !aligned16(w0) || !aligned16(w1) || !aligned16(w2) || !aligned16(out0) ||
      !aligned16(out1) || !aligned16(out2) || !aligned16(residual) || !aligned16(norm_weight))
    return fail(IVAKV_E_ARG, "%s: pointers must be 16-byte aligned", name);
  LinearArgs a;
  a.x = x;
  a.ldx = ldx;
  a.m = m;
  a.k = k;
  a.w[0] = w0;
  a.w[1] = w1;
  a.w[2] = w2;
  a.out[0] = out0;
  a.out[1] = out1;
  a.out[2] = out2;
  a.n[0] = n0;
  a.n[1] = n1;
  a.n[2] = n2;
  a.t0 = n0 / 16;
  a.t1 = a.t0 + n1 / 16;
  a.residual = residual;
  a.norm_w = norm_weight;
  a.eps = eps;
  a.tiles = epilogue == kSwiglu ? a.t0 : a.t1 + n2 / 16;
  if (dtype == IVAKV_F16) launch_linear_w<IVAKV_F16>(a, norm != 0, epilogue, stream);
  else launch_linear_w<IVAKV_BF16>(a, norm != 0, epilogue, stream);
  return launch_status(name);
}

extern "C" int ivakv_block_decode(const char* args, hipStream_t stream) {
  const char* name = "ivakv_block_decode";
  if (!args) return fail(IVAKV_E_ARG, "%s: null args", name);
  ivakv_block_decode_args a;
  memcpy(&a, args, sizeof(a));
  const int dtype = (int)a.dtype;
  int st = check_16bit(name, dtype);
  if (st != IVAKV_OK) return st;
  if (a.batch < 0 || a.batch > kLinearMaxRows || a.d_model <= 0 || a.d_model > 1 << 20 ||
      a.num_q_heads <= 0 || a.num_q_heads > 1 << 16 || a.num_kv_heads <= 0 ||
      a.num_kv_heads > a.num_q_heads || a.head_dim <= 0 || a.head_dim > 256 || a.hidden <= 0 ||
      a.hidden > 1 << 24)
    return fail(IVAKV_E_ARG, "%s: bad sizes", name);
  if (a.batch == 0) return IVAKV_OK;
  const int m = (int)a.batch, d = (int)a.d_model;
  const int nq = (int)(a.num_q_heads * a.head_dim), nkv = (int)(a.num_kv_heads * a.head_dim);
  const int hidden = (int)a.hidden;
  // The intermediate rows, each 256-byte aligned in the scratch.
  char* base = static_cast<char*>(a.scratch);
  int64_t used = 0;
  auto take = [&](int n) -> void* {
    void* p = base + used;
    used += ((int64_t)m * n * 2 + 255) & ~(int64_t)255;
    return p;
  };
  void *q = take(nq), *k = take(nkv), *v = take(nkv), *o = take(nq), *x1 = take(d), *h = take(hidden),
       *y = take(d);
  if (!base || !aligned16(base) || used > a.scratch_bytes)
    return fail(IVAKV_E_WORKSPACE, "%s: %lld bytes of scratch (16-byte aligned) required, got %lld", name,
                (long long)used, (long long)(base ? a.scratch_bytes : 0));
  const int in_norm = m <= kLinearNormRows && d <= kLinearNormMaxK;
  const void* y1 = in_norm ? a.x : y;
  if (!in_norm) {
    st = ivakv_rms_norm(a.x, nullptr, a.norm1, nullptr, y, m, d, (float)a.eps1, dtype, stream);
    if (st != IVAKV_OK) return st;
  }
  st = ivakv_linear_rows(y1, d, m, d, a.wq, nq, q, a.wk, nkv, k, a.wv, nkv, v, nullptr, in_norm,
                         a.norm1, (float)a.eps1, kPlain, dtype, stream);
  if (st != IVAKV_OK) return st;
  const int hq = (int)a.num_q_heads, hkv = (int)a.num_kv_heads, hd = (int)a.head_dim;
  if (a.fp8)
    st = ivakv_decode_append_attn_fp8(q, k, v, a.k_pool, a.v_pool, static_cast<float*>(a.k_scale),
                                      static_cast<float*>(a.v_scale), a.block_tables, a.context_lens, o,
                                      a.workspace, (size_t)a.workspace_bytes, m, hq, hkv, hd,
                                      (int)a.block_size, (int)a.max_blocks, (int)a.num_pages,
                                      (float)a.scale, (int)a.window, (int)a.n_sink, dtype, stream);
  else
    st = ivakv_decode_append_attn(q, k, v, a.k_pool, a.v_pool, a.block_tables, a.context_lens, o,
                                  a.workspace, (size_t)a.workspace_bytes, m, hq, hkv, hd,
                                  (int)a.block_size, (int)a.max_blocks, (int)a.num_pages,
                                  (float)a.scale, (int)a.window, (int)a.n_sink, dtype, stream);
  if (st != IVAKV_OK) return st;
  st = ivakv_linear_rows(o, nq, m, nq, a.wo, d, x1, nullptr, 0, nullptr, nullptr, 0, nullptr, a.x, 0,
                         nullptr, 0.f, kResidual, dtype, stream);
  if (st != IVAKV_OK) return st;
  const void* y2 = in_norm ? x1 : y;
  if (!in_norm) {
    st = ivakv_rms_norm(x1, nullptr, a.norm2, nullptr, y, m, d, (float)a.eps2, dtype, stream);
    if (st != IVAKV_OK) return st;
  }
  st = ivakv_linear_rows(y2, d, m, d, a.wgate, hidden, h, a.wup, hidden, nullptr, nullptr, 0, nullptr,
                         nullptr, in_norm, a.norm2, (float)a.eps2, kSwiglu, dtype, stream);
  if (st != IVAKV_OK) return st;
  return ivakv_linear_rows(h, hidden, m, hidden, a.wdown, d, a.out, nullptr, 0, nullptr, nullptr, 0, nullptr,
                           x1, 0, nullptr, 0.f, kResidual, dtype, stream);
}
