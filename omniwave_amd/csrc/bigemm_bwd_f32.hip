// fp32 backward building blocks: the same steps as bigemm_bwd.hip for fp32 activations.  The C-ABI
// launchers of bigemm_bwd.hip call these when dtype is OW_DTYPE_F32.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "ow_common.h"
#include "ow_device.h"

namespace ow {
namespace {

constexpr float kLn2f = 0.6931471805599453f;

unsigned grid_for(int64_t n) { return static_cast<unsigned>((n + 255) / 256); }

__device__ __forceinline__ float weight_at(const void* p, int64_t i, int dtype) {
  if (dtype == OW_DTYPE_F32) return static_cast<const float*>(p)[i];
  const uint16_t u = static_cast<const uint16_t*>(p)[i];
  return dtype == OW_DTYPE_BF16 ? BF16::to_f32(u) : F16::to_f32(u);
}

__device__ __forceinline__ int64_t slot_row_f32(const int32_t* tok, int64_t k, int32_t q_s, int32_t n_tok) {
  const int64_t tile = k >> 4;
  const int64_t b = tile / q_s;
  const int32_t s = static_cast<int32_t>(tile - b * q_s);
  const int32_t tk = tok[s * kG + static_cast<int32_t>(k & 15)];
  return (tk >= 0 && tk < n_tok) ? b * n_tok + tk : -1;
}

__global__ void __launch_bounds__(256) gather_f32_kernel(const float* x, const float* dy, const float* rscale,
                                                         const int32_t* tok, const int32_t* chan, float* xt,
                                                         float* dyt, int64_t slots, int32_t n_tok, int32_t channels,
                                                         int32_t q_s, int32_t d, int64_t total) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= total) return;
  const int32_t c = static_cast<int32_t>(i % d);
  const int64_t qk = i / d;
  const int64_t k = qk % slots;
  const int32_t q = static_cast<int32_t>(qk / slots);
  const int64_t row = slot_row_f32(tok, k, q_s, n_tok);
  const int32_t ch = chan[q * d + c];
  float xv = 0.0f, dv = 0.0f;
  if (row >= 0 && ch >= 0 && ch < channels) {
    xv = x[row * channels + ch] * (rscale ? rscale[row] : 1.0f);
    dv = dy[row * channels + ch];
  }
  xt[i] = xv;
  dyt[i] = dv;
}

__global__ void __launch_bounds__(256) gate_f32_kernel(const float* u, const float* v, const float* dz, float* z,
                                                       float* du, float* dv, int64_t n) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= n) return;
  const float up = u[i], vp = v[i], g = dz[i];
  const float s = 1.0f / (1.0f + exp2f(up));
  z[i] = up * vp * s;
  du[i] = g * vp * s * (1.0f - kLn2f * up * (1.0f - s));
  dv[i] = g * up * s;
}

__global__ void __launch_bounds__(256) scatter_f32_kernel(const float* dxt, const int32_t* tok, const int32_t* chan,
                                                          float* g, int64_t slots, int32_t n_tok, int32_t channels,
                                                          int32_t q_s, int32_t d, int64_t total) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= total) return;
  const int32_t c = static_cast<int32_t>(i % d);
  const int64_t qk = i / d;
  const int64_t k = qk % slots;
  const int32_t q = static_cast<int32_t>(qk / slots);
  const int64_t row = slot_row_f32(tok, k, q_s, n_tok);
  const int32_t ch = chan[q * d + c];
  if (row >= 0 && ch >= 0 && ch < channels) g[row * channels + ch] = dxt[i];
}

// dx = (dout) + r g - x r^3 / C sum_c(g x), one row per LPR lanes of 4 channels each (C % 4 == 0,
// 16-byte aligned rows, VEC), or one per wave with one channel per lane step.
template <int LPR, bool VEC>
__global__ void __launch_bounds__(256) rmsnorm_bwd_f32_kernel(const float* __restrict__ x, const float* __restrict__ g,
                                                              const float* __restrict__ rscale,
                                                              const float* __restrict__ dout, float* __restrict__ dx,
                                                              int64_t rows, int32_t channels, int32_t residual) {
  constexpr int RPB = 256 / LPR, W = VEC ? 4 : 1;
  typedef float vec __attribute__((ext_vector_type(W)));
  const int64_t row = static_cast<int64_t>(blockIdx.x) * RPB + threadIdx.x / LPR;
  const int sub = threadIdx.x % LPR;
  if (row >= rows) return;  // whole groups of LPR lanes leave together
  auto at = [&](const float* p, int c) { return *reinterpret_cast<const vec*>(p + row * channels + c); };
  float r = 1.0f, coef = 0.0f;
  if (rscale) {
    r = rscale[row];
    float dot = 0.0f;
    for (int c = W * sub; c < channels; c += W * LPR) {
      const vec xv = at(x, c), gv = at(g, c);
#pragma unroll
      for (int k = 0; k < W; ++k) dot = fmaf(gv[k], xv[k], dot);
    }
    for (int m = LPR / 2; m > 0; m >>= 1) dot += __shfl_xor(dot, m);
    coef = dot * r * r * r / static_cast<float>(channels);
  }
  for (int c = W * sub; c < channels; c += W * LPR) {
    vec v = r * at(g, c) - coef * at(x, c);
    if (residual) v += at(dout, c);
    *reinterpret_cast<vec*>(dx + row * channels + c) = v;
  }
}

struct FoldF32Args {
  const void* b_u;
  const void* b_v;
  const void* b_o;
  const float* norm_w;
  const float* gamma;
  const int32_t* chan;
  float* bu;
  float* buT;
  float* bv;
  float* bvT;
  float* bo;
  float* boT;
  int32_t wdtype, q_c, d, rd, channels;
};

__global__ void __launch_bounds__(256) fold_f32_kernel(FoldF32Args a, int64_t total) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= total) return;
  const int32_t e = static_cast<int32_t>(i % a.rd);
  const int64_t qc = i / a.rd;
  const int32_t c = static_cast<int32_t>(qc % a.d);
  const int32_t q = static_cast<int32_t>(qc / a.d);
  const int32_t ch = a.chan[q * a.d + c];
  const bool ok = ch >= 0 && ch < a.channels;
  const float w = ok ? (a.norm_w ? a.norm_w[ch] : 1.0f) : 0.0f;
  const float gm = ok ? (a.gamma ? a.gamma[ch] : 1.0f) : 0.0f;
  const int64_t cd = (static_cast<int64_t>(q) * a.d + c) * a.rd + e;
  const int64_t ec = (static_cast<int64_t>(q) * a.rd + e) * a.d + c;
  const float u = weight_at(a.b_u, cd, a.wdtype) * w * kNegLog2e;
  const float v = weight_at(a.b_v, cd, a.wdtype) * w * kNegLn2;
  const float o = weight_at(a.b_o, ec, a.wdtype) * gm;
  a.bu[cd] = u;
  a.buT[ec] = u;
  a.bv[cd] = v;
  a.bvT[ec] = v;
  a.bo[ec] = o;
  a.boT[cd] = o;
}

// out[t][i][c] = sum_j M1[i][j] in1[t][j][c] (+ M2[i][j] in2[t][j][c]): one thread per (tile,
// column) holds the column's 16 values and forms its 16 outputs, the matrices from scalar
// registers, so each value is read once (a thread per output read it 16 times).  Bound by
// memory: 25,088 slots x 4 groups x 64 channels, one input, 33 -> 10.5 us.
template <bool TWO>
__global__ void __launch_bounds__(256) tile_mix_f32_kernel(const float* __restrict__ in1, const float* __restrict__ m1,
                                                           const float* __restrict__ in2, const float* __restrict__ m2,
                                                           float* __restrict__ out, int64_t columns, int32_t d) {
  const int64_t idx = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (idx >= columns) return;
  const int64_t tile = idx / d;
  const int64_t base = tile * kG * d + (idx - tile * d);
  float v[kG], w[TWO ? kG : 1];
#pragma unroll
  for (int j = 0; j < kG; ++j) v[j] = in1[base + static_cast<int64_t>(j) * d];
  if constexpr (TWO) {
#pragma unroll
    for (int j = 0; j < kG; ++j) w[j] = in2[base + static_cast<int64_t>(j) * d];
  }
#pragma unroll
  for (int i = 0; i < kG; ++i) {
    float acc = 0.0f;
#pragma unroll
    for (int j = 0; j < kG; ++j) acc = fmaf(m1[i * kG + j], v[j], acc);
    if constexpr (TWO) {
#pragma unroll
      for (int j = 0; j < kG; ++j) acc = fmaf(m2[i * kG + j], w[j], acc);
    }
    out[base + static_cast<int64_t>(i) * d] = acc;
  }
}

// partial[i][j][w] = sum over tiles t = w, w + n_waves, ... of sum_c in1[t][i][c] in2[t][j][c]
// on the fp32 16x16x4 MFMA: lane (row l16, h) holds channels 16 s + 4 h .. + 3 of its row, and
// product j of a 16-channel step takes component j of both operands.  Bound by memory (each tile
// is read once, 64-byte pieces of 16 rows per instruction), so with few waves the loads of two
// tiles are in flight before the first product (D, the compile-time d; 0: any, one step at a
// time).  The same shape took 169 us with one serial dot product per output, 18 us now.
template <bool VEC, int D>
__global__ void __launch_bounds__(256) tile_outer_f32_kernel(const float* __restrict__ in1, const float* __restrict__ in2,
                                                             float* __restrict__ partial, int64_t n_tiles, int32_t d) {
  const int lane = threadIdx.x & 63, l16 = lane & 15, h = lane >> 4;
  const int64_t wave = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
  const int64_t n_waves = static_cast<int64_t>(gridDim.x) * 4;
  auto load = [&](const float* p) {
    if constexpr (VEC) {
      return *reinterpret_cast<const f32x4*>(p);
    } else {
      return f32x4{p[0], p[1], p[2], p[3]};
    }
  };
  const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
  f32x4 acc = zero;  // sum over tiles; a tile's own sum is formed apart, so the fp32 chains stay short
  auto mma = [&](const f32x4& a, const f32x4& b, f32x4& c) {
#pragma unroll
    for (int j = 0; j < 4; ++j) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j], b[j], c, 0, 0, 0);
  };
  if constexpr (D > 0) {
    constexpr int N = D / 16;
    for (int64_t t = wave; t < n_tiles; t += 2 * n_waves) {
      const bool two = t + n_waves < n_tiles;
      const int64_t b0 = (t * kG + l16) * D + 4 * h, b1 = ((two ? t + n_waves : t) * kG + l16) * D + 4 * h;
      f32x4 u[2][N], v[2][N];
#pragma unroll
      for (int c = 0; c < N; ++c) {
        u[0][c] = load(in1 + b0 + 16 * c);
        v[0][c] = load(in2 + b0 + 16 * c);
      }
#pragma unroll
      for (int c = 0; c < N; ++c) {
        u[1][c] = load(in1 + b1 + 16 * c);
        v[1][c] = load(in2 + b1 + 16 * c);
      }
      f32x4 s[2] = {zero, zero};
#pragma unroll
      for (int c = 0; c < N; ++c) {
        mma(u[0][c], v[0][c], s[0]);
        mma(u[1][c], v[1][c], s[1]);
      }
      mfma_drain();
      acc += two ? s[0] + s[1] : s[0];
    }
  } else {
    for (int64_t t = wave; t < n_tiles; t += n_waves) {
      const int64_t base = (t * kG + l16) * d + 4 * h;
      f32x4 s = zero;
      for (int c = 0; c < d; c += 16) mma(load(in1 + base + c), load(in2 + base + c), s);
      mfma_drain();
      acc += s;
    }
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) partial[static_cast<int64_t>((4 * h + k) * kG + l16) * n_waves + wave] = acc[k];
}

}  // namespace

int bwd_gather_f32(const float* x, const float* dy, const float* rscale, const int32_t* tok, const int32_t* chan,
                   float* xt, float* dyt, int64_t slots, int32_t n_tok, int32_t channels, int32_t q_s, int32_t q_c,
                   int32_t d, hipStream_t s) {
  const int64_t total = static_cast<int64_t>(q_c) * slots * d;
  hipLaunchKernelGGL(gather_f32_kernel, dim3(grid_for(total)), dim3(256), 0, s, x, dy, rscale, tok, chan, xt, dyt,
                     slots, n_tok, channels, q_s, d, total);
  return hip_status(hipGetLastError(), "gather_f32_kernel launch");
}

int bwd_gate_f32(const float* u, const float* v, const float* dz, float* z, float* du, float* dv, int64_t n,
                 hipStream_t s) {
  hipLaunchKernelGGL(gate_f32_kernel, dim3(grid_for(n)), dim3(256), 0, s, u, v, dz, z, du, dv, n);
  return hip_status(hipGetLastError(), "gate_f32_kernel launch");
}

int bwd_scatter_f32(const float* dxt, const int32_t* tok, const int32_t* chan, float* g, int64_t slots,
                    int32_t n_tok, int32_t channels, int32_t q_s, int32_t q_c, int32_t d, hipStream_t s) {
  const int64_t total = static_cast<int64_t>(q_c) * slots * d;
  hipLaunchKernelGGL(scatter_f32_kernel, dim3(grid_for(total)), dim3(256), 0, s, dxt, tok, chan, g, slots, n_tok,
                     channels, q_s, d, total);
  return hip_status(hipGetLastError(), "scatter_f32_kernel launch");
}

int bwd_rmsnorm_f32(const float* x, const float* g, const float* rscale, const float* dout, float* dx, int64_t rows,
                    int32_t channels, int32_t residual, hipStream_t s) {
  auto launch = [&](auto lpr, auto vec) {
    constexpr int L = decltype(lpr)::value;
    hipLaunchKernelGGL((rmsnorm_bwd_f32_kernel<L, decltype(vec)::value>),
                       dim3(static_cast<unsigned>((rows * L + 255) / 256)), dim3(256), 0, s, x, g, rscale, dout, dx, rows,
                       channels, residual);
  };
  const std::integral_constant<bool, true> vec;
  const bool aligned = channels % 4 == 0 && aligned16(x) && aligned16(g) && aligned16(dx) && (!residual || aligned16(dout));
  if (!aligned)
    launch(std::integral_constant<int, 64>{}, std::integral_constant<bool, false>{});
  else if (channels <= 128)  // a row in one step of half a wave
    launch(std::integral_constant<int, 32>{}, vec);
  else
    launch(std::integral_constant<int, 64>{}, vec);
  return hip_status(hipGetLastError(), "rmsnorm_bwd_f32_kernel launch");
}

int fold_weights_f32(const void* b_u, const void* b_v, const void* b_o, int32_t wdtype, const float* norm_w,
                     const float* gamma, const int32_t* chan, int32_t channels, int32_t q_c, int32_t d, int32_t rd,
                     float* bu, float* buT, float* bv, float* bvT, float* bo, float* boT, hipStream_t s) {
  FoldF32Args a{b_u, b_v, b_o, norm_w, gamma, chan, bu, buT, bv, bvT, bo, boT, wdtype, q_c, d, rd, channels};
  const int64_t total = static_cast<int64_t>(q_c) * d * rd;
  hipLaunchKernelGGL(fold_f32_kernel, dim3(grid_for(total)), dim3(256), 0, s, a, total);
  return hip_status(hipGetLastError(), "fold_f32_kernel launch");
}

int tile_mix_f32(const float* in1, const float* m1, const float* in2, const float* m2, float* out, int64_t n_tiles,
                 int32_t d, hipStream_t s) {
  const int64_t columns = n_tiles * d;
  if (in2)
    hipLaunchKernelGGL(tile_mix_f32_kernel<true>, dim3(grid_for(columns)), dim3(256), 0, s, in1, m1, in2, m2, out,
                       columns, d);
  else
    hipLaunchKernelGGL(tile_mix_f32_kernel<false>, dim3(grid_for(columns)), dim3(256), 0, s, in1, m1, in2, m2, out,
                       columns, d);
  return hip_status(hipGetLastError(), "tile_mix_f32_kernel launch");
}

int tile_outer_f32(const float* in1, const float* in2, float* partial, int32_t n_waves, int64_t n_tiles, int32_t d,
                   hipStream_t s) {
  const dim3 grid(static_cast<unsigned>(n_waves / 4));
  const bool vec = aligned16(in1) && aligned16(in2);
  if (vec && d == 64)
    hipLaunchKernelGGL((tile_outer_f32_kernel<true, 64>), grid, dim3(256), 0, s, in1, in2, partial, n_tiles, d);
  else if (vec && d == 128)
    hipLaunchKernelGGL((tile_outer_f32_kernel<true, 128>), grid, dim3(256), 0, s, in1, in2, partial, n_tiles, d);
  else
    hipLaunchKernelGGL((tile_outer_f32_kernel<false, 0>), grid, dim3(256), 0, s, in1, in2, partial, n_tiles, d);
  return hip_status(hipGetLastError(), "tile_outer_f32_kernel launch");
}

}  // namespace ow
