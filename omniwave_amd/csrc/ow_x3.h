// fp32 operands on the bf16 matrix cores: every fp32 value is the sum of three bf16 values
// (v = v0 + v1 + v2, each the nearest bf16 of what is left: 3 x 8 significand bits, so a value
// is held to its 24 bits), and a product of two such operands is the six bf16 products whose
// weight is above 2^-24:
//     a b = a0 b0 + (a0 b1 + a1 b0) + (a0 b2 + a1 b1 + a2 b0)      (fp32 accumulation)
// What is left out (a1 b2, a2 b1, a2 b2) is below 2^-25 of the product.  The bf16 MFMAs have 16
// times the rate of the fp32 ones, so six of them cost 0.375 of one fp32 product.
//
// Range: up to fp32's largest value (x3_split2).  Parts end at bf16's smallest subnormal, so an
// operand below about 2^-110 is held to 2^-134 instead of 24 bits (gradients from an upstream of
// 2^-112: 5e-7 off, 2^-116: 7e-6).  An infinite operand makes its token group's results NaN (its
// parts are not all infinite), never another group's.
#pragma once

#include "ow_device.h"

namespace ow {

// One operand of a 32x32x16 product (8 values per lane) as its three bf16 parts.
struct X3 {
  u32x4 p[3];
};

// Two fp32 values -> their three parts, packed (first value in the low half).  The largest values
// (from 3.3962e38 on) round up to infinity in bf16; kWhole keeps them: the first part is at most
// bf16's largest and the second holds the rest.  It is for the caller's tensors (weights: x3_part); for the
// sums in between, where those values are infinite, it would cost 2% of the whole kernels.
constexpr float kMostBf16 = 3.38953139e38f;  // 0x7f7f0000
template <bool kWhole = false>
__device__ __forceinline__ void x3_split2(float a, float b, uint32_t& p0, uint32_t& p1, uint32_t& p2) {
  if constexpr (kWhole)
    p0 = BF16::pack2(__builtin_amdgcn_fmed3f(a, -kMostBf16, kMostBf16), __builtin_amdgcn_fmed3f(b, -kMostBf16, kMostBf16));
  else
    p0 = BF16::pack2(a, b);
  const float a1 = a - __uint_as_float(p0 << 16), b1 = b - __uint_as_float(p0 & 0xffff0000u);
  p1 = BF16::pack2(a1, b1);
  p2 = BF16::pack2(a1 - __uint_as_float(p1 << 16), b1 - __uint_as_float(p1 & 0xffff0000u));
}

template <bool kWhole = false, class V>
__device__ __forceinline__ X3 x3_split8(V v) {  // v(j), j = 0..7
  X3 r;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    uint32_t a, b, c;
    x3_split2<kWhole>(v(2 * q), v(2 * q + 1), a, b, c);
    r.p[0][q] = a;
    r.p[1][q] = b;
    r.p[2][q] = c;
  }
  return r;
}

// Part n of a folded weight, taken off it (only the first is cut off, so that NaN stays NaN).
__device__ __forceinline__ uint16_t x3_part(double& v, int n) {
  const float f = static_cast<float>(v);
  const uint16_t b = BF16::from_f32(n == 0 ? __builtin_amdgcn_fmed3f(f, -kMostBf16, kMostBf16) : f);
  v -= static_cast<double>(BF16::to_f32(b));
  return b;
}

// Accumulator registers 8s..8s+7 as an operand (K step s of the next product).
__device__ __forceinline__ X3 x3_kstep(const f32x16& acc, int s) {
  return x3_split8([&](int j) { return acc[8 * s + j]; });
}

// c + a b, smallest products first.
__device__ __forceinline__ f32x16 x3_mma(const X3& a, const X3& b, f32x16 c) {
  c = BF16::mma32(a.p[2], b.p[0], c);
  c = BF16::mma32(a.p[1], b.p[1], c);
  c = BF16::mma32(a.p[0], b.p[2], c);
  c = BF16::mma32(a.p[1], b.p[0], c);
  c = BF16::mma32(a.p[0], b.p[1], c);
  return BF16::mma32(a.p[0], b.p[0], c);
}

// The same with the five smaller products in a sum of their own: one rounding at the size of the
// sum per product instead of six (long chains, where those roundings are the error).
__device__ __forceinline__ void x3_mma_apart(const X3& a, const X3& b, f32x16& hi, f32x16& lo) {
  lo = BF16::mma32(a.p[2], b.p[0], lo);
  lo = BF16::mma32(a.p[1], b.p[1], lo);
  lo = BF16::mma32(a.p[0], b.p[2], lo);
  lo = BF16::mma32(a.p[1], b.p[0], lo);
  lo = BF16::mma32(a.p[0], b.p[1], lo);
  hi = BF16::mma32(a.p[0], b.p[0], hi);
}

// The two token groups of a pair share a product's 32 rows and columns but not its K steps: each
// group's product is formed apart, with the same token matrix in every lane, and its half of the
// result taken.  (A zero in the other group's place would be as many products, but 0 x NaN and
// 0 x Inf are NaN, and the groups of a pair can belong to different images.)
// lane & 15 = token (columns): group 0 in lanes without bit 4.
__device__ __forceinline__ f32x16 pair_columns(bool group0, const f32x16& p0, const f32x16& p1) {
  f32x16 r;
#pragma unroll
  for (int i = 0; i < 16; ++i) r[i] = group0 ? p0[i] : p1[i];
  return r;
}
// rows = tokens: group 0 in registers 0 to 7 (pair_token_row).
__device__ __forceinline__ f32x16 pair_rows_of(const f32x16& p0, const f32x16& p1) {
  f32x16 r;
#pragma unroll
  for (int i = 0; i < 16; ++i) r[i] = i < 8 ? p0[i] : p1[i];
  return r;
}

}  // namespace ow
