// fp32 backward of the channel side on the bf16 matrix cores (three-part operands, ow_x3.h): the
// gradients of omniweave/ops/reference.py:120-173 (autograd there) in three kernels,
// for d, rd as the forward.  x r and dy are read where they lie, through the token and channel tables.
//
//   chan_x3     P_u = A_u X', P_v = A_v X', dW' = A_o^T dY, then per 32-row chunk of the expanded
//               dimension U', V', dZ and the gate backward: Z, dU', dV'
//   chan2_x3    dP_u = dU' B_u''^T, dP_v = dV' B_v''^T, W' = Z B_o'', from the registers they are
//               summed in the token-matrix gradients and dX' = A_u^T dP_u + A_v^T dP_v, stored at
//               its routed place
//   reduce_x3   dB_u'' = P_u^T dU', dB_v'' = P_v^T dV', dB_o'' = Z^T dW' over ranges of slots
//
// The split lies where the fewest values cross it that a wave's registers can't hold: at d = 128
// the operands of the first three products take 288 registers and the sums of the second three
// 192.  Each value that crosses is written once and read twice (chan2_x3, reduce_x3).
//
// 28x28x256, B = 32 (100,352 slots of 64 channels): 81 + 73 + 51 us, where fp32 products of the
// library around a gate kernel, gather, token mixings, per-tile outer products and the scatter took
// 485; the whole step 640 -> 310 us.  With routed tiles X', dY written by a gather kernel first (27
// us) the three took 80 + 72 + 51.  Errors against 64 bits over 4x4 to 56x56 images: dx 1.7e-7
// (2.6e-7 before), weights' 4.3e-7 (7.2e-7), token matrices' 4.3e-7 (5.5e-7).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "ow_common.h"
#include "ow_x3.h"

namespace ow {
namespace {

constexpr int kThreads = 256;
constexpr float kLn2f = 0.6931471805599453f;

struct PackBwdX3Args {
  const void* b[3];
  const float* norm_w;
  const float* gamma;
  const int32_t* chan;
  uint4* packed;
  int32_t wdtype, q_c, d, rd, channels;
  int64_t total;  // operand lanes: q_c * 2 * (rd / 32) * 3 * (d / 16) * 64
};

__device__ __forceinline__ double weight64(const void* p, int64_t i, int dtype) {
  if (dtype == OW_DTYPE_F32) return static_cast<const float*>(p)[i];
  const uint16_t u = static_cast<const uint16_t*>(p)[i];
  return dtype == OW_DTYPE_BF16 ? BF16::to_f32(u) : F16::to_f32(u);
}

// Per group: the chunks of chan_x3 (rows: 32 expanded rows, K: 16 channels a step), then those of
// chan2_x3 (rows: 32 channels, K: 16 expanded rows); a chunk holds B_u'', B_v'', B_o'', each d / 16
// fragments of three 1 KB parts.  Folds in fp64, as in the forward's packed weights.
__global__ void __launch_bounds__(kThreads) pack_bwd_x3_kernel(PackBwdX3Args p) {
  const int64_t idx = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
  if (idx >= p.total) return;
  const int lane = static_cast<int>(idx & 63), l32 = lane & 31, hh = lane >> 5;
  const int ks_n = p.d / 16, nch = p.rd / 32;
  int64_t rem = idx >> 6;
  const int f = static_cast<int>(rem % ks_n);
  rem /= ks_n;
  const int kind = static_cast<int>(rem % 3);
  rem /= 3;
  const int ec = static_cast<int>(rem % nch);
  rem /= nch;
  const int second = static_cast<int>(rem & 1);
  const int q = static_cast<int>(rem >> 1);
  const double fold = kind == 0 ? -1.4426950408889634 : kind == 1 ? -0.6931471805599453 : 1.0;
  const float* vec = kind < 2 ? p.norm_w : p.gamma;
  uint32_t w[3][4];
#pragma unroll
  for (int j2 = 0; j2 < 4; ++j2) {
    uint32_t part[3][2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int k = pair_token_row(2 * j2 + h, hh);
      const int c = second ? 32 * (f >> 1) + l32 : 16 * f + k;
      const int e = 32 * ec + (second ? 16 * (f & 1) + k : l32);
      const int gc = p.chan[q * p.d + c];
      const bool ok = gc >= 0 && gc < p.channels;
      double v = ok ? (vec ? fold * static_cast<double>(vec[gc]) : fold) : 0.0;
      const int64_t mat = static_cast<int64_t>(q) * p.d * p.rd;
      v *= weight64(p.b[kind], mat + (kind < 2 ? static_cast<int64_t>(c) * p.rd + e : static_cast<int64_t>(e) * p.d + c),
                    p.wdtype);
#pragma unroll
      for (int n = 0; n < 3; ++n) part[n][h] = x3_part(v, n);
    }
#pragma unroll
    for (int n = 0; n < 3; ++n) w[n][j2] = part[n][0] | (part[n][1] << 16);
  }
  uint4* dst = p.packed + (idx >> 6) * 3 * 64 + lane;
#pragma unroll
  for (int n = 0; n < 3; ++n) dst[64 * n] = uint4{w[n][0], w[n][1], w[n][2], w[n][3]};
}

struct ChanX3Args {
  const float* x;
  const float* dy;
  const float* rscale;  // NULL: 1
  const float* a_u;
  const float* a_v;
  const float* a_o;
  const uint8_t* packed;
  float* pu;
  float* pv;
  float* dw;
  float* z;
  float* du;
  float* dv;
  float* g;  // chan2_x3
  float* partial;
  const int32_t* tok;
  const int32_t* chan;
  int64_t slots;
  int32_t q_c, rd, n_tok, channels, q_s, batch;
};

// Row l32 % 16 of a token matrix (or of its transpose), 8 entries in the K order of the pair scheme.
__device__ __forceinline__ X3 token_operand(const float* m, bool transposed, int l32, int hh) {
  const int r = l32 & 15;
  return x3_split8<true>([&](int j) {
    const int k = pair_token_row(j, hh);
    return transposed ? m[k * kG + r] : m[r * kG + k];
  });
}

// A wave's pair of one group: its 32 rows of a [q_c][slots][width] matrix as a buffer (rows past
// the last slot read as zero and store nowhere; a wave without a pair has no rows at all).
struct PairRows {
  int64_t first;
  uint32_t rows;
  __device__ __forceinline__ __amdgpu_buffer_rsrc_t of(const float* p, int width) const {
    const uint16_t* base = uniform_ptr(reinterpret_cast<const uint16_t*>(p + first * width));
    return buffer_rsrc(base, rows * static_cast<uint32_t>(width) * 4u);
  }
};
__device__ __forceinline__ PairRows pair_rows(int64_t slots, int q, int64_t pair) {
  const int64_t s0 = 32 * pair;
  const bool any = s0 < slots;
  const int64_t left = slots - s0;
  return {static_cast<int64_t>(q) * slots + (any ? s0 : 0), any ? static_cast<uint32_t>(left < 32 ? left : 32) : 0u};
}

__device__ __forceinline__ float load1(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, static_cast<int>(off), 0, 0));
}
__device__ __forceinline__ f32x4 load4(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, static_cast<int>(off), 0, 0));
}
// Accumulator registers 4k .. 4k + 3 (consecutive rows 8k + 4hh ..) to one lane's row.
__device__ __forceinline__ void store4(__amdgpu_buffer_rsrc_t r, uint32_t off, const f32x16& v, int k) {
  const f32x4 t = {v[4 * k], v[4 * k + 1], v[4 * k + 2], v[4 * k + 3]};
  __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, t), r, static_cast<int>(off), 0, 0);
}

// Routed x and dy: a buffer from the first image of the workgroup's pairs on, of at most 1 GiB; a pad
// slot's row offset lies at 2 GiB and a pad channel's at 1 GiB, so what either asks for reads as zero
// without a branch.
constexpr int64_t kSpan = int64_t(1) << 30;
struct Routed {
  int64_t img0;
  __device__ __forceinline__ Routed(const ChanX3Args& a, int64_t pair0) : img0(2 * pair0 / a.q_s) {}
  __device__ __forceinline__ __amdgpu_buffer_rsrc_t of(const float* p, const ChanX3Args& a) const {
    const int64_t img = static_cast<int64_t>(a.n_tok) * a.channels, left = (a.batch - img0) * img * 4;
    return buffer_rsrc(p + img0 * img, static_cast<uint32_t>(left < kSpan ? left : kSpan));
  }
};
// The workgroup's 128 slots: byte offset of the row, row number (-1: pad) and RMSNorm scale.
struct SlotTables {
  uint32_t off[4][32];
  int32_t row[4][32];
  float scale[4][32];
  __device__ __forceinline__ void fill(const ChanX3Args& a, int64_t pair0, int64_t img0, int t) {
    const int64_t slot = 32 * pair0 + t;
    uint32_t o = kOffOut;
    int32_t r = -1;
    float s = 0.0f;
    if (slot < a.slots) {
      const int64_t b = (slot >> 4) / a.q_s;
      const int32_t tk = a.tok[((slot >> 4) - b * a.q_s) * kG + (slot & 15)];
      if (tk >= 0 && tk < a.n_tok) {
        o = static_cast<uint32_t>((b - img0) * a.n_tok + tk) * static_cast<uint32_t>(a.channels) * 4u;
        r = static_cast<int32_t>(b * a.n_tok + tk);
        s = a.rscale ? a.rscale[r] : 1.0f;
      }
    }
    off[t >> 5][t & 31] = o;
    row[t >> 5][t & 31] = r;
    scale[t >> 5][t & 31] = s;
  }
};
__device__ __forceinline__ uint32_t channel_offset(const ChanX3Args& a, int64_t i) {
  const int32_t ch = a.chan[i];
  return ch >= 0 && ch < a.channels ? 4u * static_cast<uint32_t>(ch) : static_cast<uint32_t>(kSpan);
}

// The weight chunks of one group and phase through two LDS buffers: every wave copies a quarter.
template <int KS>
struct ChunkRing {
  static constexpr int FR = 9 * KS, CP = FR / 4;
  const uint8_t* src;
  uint32_t lds, lane16;
  int wave;
  __device__ __forceinline__ void copy(int ec, int buf) const {
    const uint8_t* s = src + (static_cast<int64_t>(ec) * FR + wave * CP) * 1024;
#pragma unroll
    for (int i = 0; i < CP; ++i)
      copy_frag_to_lds_at(uniform_ptr(reinterpret_cast<const uint16_t*>(s + i * 1024)),
                          lds + static_cast<uint32_t>((buf * FR + wave * CP + i) * 1024), lane16);
  }
};
__device__ __forceinline__ X3 ring_frag(const u32x4* p) { return X3{{p[0], p[64], p[128]}}; }

// Workgroups are dispatched round-robin over the 8 XCDs: the q_c groups of one block of pairs lie 8
// apart, on one XCD, whose L2 then serves the rows that interleaved groups share (28x28x256 radix,
// B = 32, the whole step 380 -> 345 us; 7x7x1024 radix, B = 64, 370 -> 340; contiguous groups the
// same or a little less).
//
// Four waves, each a 32-slot pair, share a group's weight chunks (36 KB at d = 64, 72 KB at
// d = 128) through two LDS buffers, one barrier a chunk.  A chunk's copies have its predecessor's
// products to land in, and its stores its successor's.  The rows are read once and P_u, P_v,
// dW', Z, dU', dV' written once, as 16-byte pieces straight from the accumulators (lane = slot): at
// 28x28x256, B = 32 295 MB in 81 us, 70% of a copy's rate, beside 18% of the matrix cores' time.
// What keeps it from either is the rounds: 784 workgroups on 512 places.
template <int D>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(D == 64 ? 2 : 1, D == 64 ? 2 : 1)))
chan_x3_kernel(ChanX3Args a) {
  constexpr int KS = D / 16, MB = D / 32;
  using Ring = ChunkRing<KS>;
  __shared__ __attribute__((aligned(16))) u32x4 ring[2][Ring::FR * 64];
  __shared__ __attribute__((aligned(16))) SlotTables tab;
  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, hh = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int q = static_cast<int>(blockIdx.x / 8) % a.q_c;
  const int64_t block = static_cast<int64_t>(blockIdx.x) / (8 * a.q_c) * 8 + blockIdx.x % 8, pair0 = 4 * block;
  if (32 * pair0 >= a.slots) return;
  const PairRows rows = pair_rows(a.slots, q, pair0 + wave);
  const Routed routed(a, pair0);
  const int ne = a.rd / 32;
  const Ring copier{a.packed + static_cast<int64_t>(q) * 2 * ne * Ring::FR * 1024, lds_addr(&ring[0][0]),
                    16u * static_cast<uint32_t>(lane), wave};
  copier.copy(0, 0);

  if (tid < 128) tab.fill(a, pair0, routed.img0, tid);
  __syncthreads();
  const bool g0 = (lane & 16) == 0;
  X3 P[3][KS];  // P_u, P_v, dW' as K-step operands
  const f32x16 zero = {};
  auto load_rows = [&](const __amdgpu_buffer_rsrc_t& r, float(&v)[MB][16]) {
#pragma unroll
    for (int cb = 0; cb < MB; ++cb) {
      const uint32_t ch = channel_offset(a, q * D + 32 * cb + l32);
#pragma unroll
      for (int i = 0; i < 16; ++i) v[cb][i] = load1(r, tab.off[wave][pair_token_row(i, hh)] + ch);
    }
  };
  const uint32_t own = static_cast<uint32_t>(l32 * D + 4 * hh) * 4u;
  auto token_side = [&](const float(&raw)[MB][16], const X3& m, const __amdgpu_buffer_rsrc_t& out, X3(&op)[KS]) {
#pragma unroll
    for (int cb = 0; cb < MB; ++cb) {
      const f32x16 p0 = x3_mma(x3_split8<true>([&](int j) { return raw[cb][j]; }), m, zero);
      const f32x16 p1 = x3_mma(x3_split8<true>([&](int j) { return raw[cb][8 + j]; }), m, zero);
      mfma_drain();
      const f32x16 p = pair_columns(g0, p0, p1);
#pragma unroll
      for (int k = 0; k < 4; ++k) store4(out, own + static_cast<uint32_t>(32 * cb + 8 * k) * 4u, p, k);
      op[2 * cb] = x3_kstep(p, 0);
      op[2 * cb + 1] = x3_kstep(p, 1);
    }
  };
  {
    float x[MB][16], y[MB][16];  // all of a lane's loads in flight at once
    load_rows(routed.of(a.x, a), x);
    load_rows(routed.of(a.dy, a), y);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const float r = tab.scale[wave][pair_token_row(i, hh)];
#pragma unroll
      for (int cb = 0; cb < MB; ++cb) x[cb][i] *= r;
    }
    token_side(x, token_operand(a.a_u, false, l32, hh), rows.of(a.pu, D), P[0]);
    token_side(x, token_operand(a.a_v, false, l32, hh), rows.of(a.pv, D), P[1]);
    token_side(y, token_operand(a.a_o, true, l32, hh), rows.of(a.dw, D), P[2]);
  }
  const __amdgpu_buffer_rsrc_t rz = rows.of(a.z, a.rd), rdu = rows.of(a.du, a.rd), rdv = rows.of(a.dv, a.rd);
  const uint32_t wide = static_cast<uint32_t>(l32 * a.rd + 4 * hh) * 4u;
  wait_vmcnt<0>();
#pragma unroll 1
  for (int ec = 0; ec < ne; ++ec) {
    __syncthreads();  // chunk ec is there, and chunk ec - 1 has been read by every wave
    if (ec + 1 < ne) copier.copy(ec + 1, (ec + 1) & 1);
    const u32x4* fr = &ring[ec & 1][lane];
    f32x16 acc[3] = {zero, zero, zero};  // U', V', dZ: rows = expanded rows, lane = slot
#pragma unroll
    for (int f = 0; f < KS; ++f)
#pragma unroll
      for (int m = 0; m < 3; ++m) acc[m] = x3_mma(ring_frag(fr + (m * KS + f) * 192), P[m][f], acc[m]);
    mfma_drain();
    f32x16 z, du, dv;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const float up = acc[0][i], vp = acc[1][i], g = acc[2][i];
      const float s = __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(up));
      z[i] = up * vp * s;
      du[i] = g * vp * s * (1.0f - kLn2f * up * (1.0f - s));
      dv[i] = g * up * s;
    }
    wait_vmcnt<0>();  // the next chunk's copies; this chunk's stores follow
    const uint32_t o = wide + static_cast<uint32_t>(32 * ec) * 4u;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      store4(rz, o + 32u * k, z, k);
      store4(rdu, o + 32u * k, du, k);
      store4(rdv, o + 32u * k, dv, k);
    }
  }
}

// Pairs and weight chunks as above (245 MB in 73 us, 23% of the matrix cores' time, the same rounds;
// at d = 128 six registers are kept in spare accumulator registers).  Each lane reads its slot's rows of dU', dV', Z as 16-byte
// pieces, one chunk ahead; the sums have lane = slot and rows = channels, which are operands of
// the token-matrix gradients as they stand; dX' contracts the slots, so dP_u and dP_v go through
// LDS (rows of 36 floats: neither direction conflicts) to lane = channel.
template <int D>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(D == 64 ? 2 : 1, D == 64 ? 2 : 1)))
chan2_x3_kernel(ChanX3Args a) {
  constexpr int KS = D / 16, MB = D / 32, LD = 36;
  using Ring = ChunkRing<KS>;
  __shared__ __attribute__((aligned(16))) u32x4 ring[2][Ring::FR * 64];
  __shared__ __attribute__((aligned(16))) SlotTables tab;
  static_assert(sizeof(ring) >= 4 * (32 * LD + 768) * sizeof(float), "the epilogue's LDS fits the ring");
  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, hh = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int q = static_cast<int>(blockIdx.x / 8) % a.q_c;
  const int64_t block = static_cast<int64_t>(blockIdx.x) / (8 * a.q_c) * 8 + blockIdx.x % 8, pair0 = 4 * block;
  if (32 * pair0 >= a.slots) return;
  const PairRows rows = pair_rows(a.slots, q, pair0 + wave);
  const int ne = a.rd / 32;
  const Ring copier{a.packed + (static_cast<int64_t>(q) * 2 + 1) * ne * Ring::FR * 1024, lds_addr(&ring[0][0]),
                    16u * static_cast<uint32_t>(lane), wave};
  copier.copy(0, 0);
  const Routed routed(a, pair0);
  if (tid < 128) tab.fill(a, pair0, routed.img0, tid);

  const float* src[3] = {a.du, a.dv, a.z};
  __amdgpu_buffer_rsrc_t r[3] = {rows.of(src[0], a.rd), rows.of(src[1], a.rd), rows.of(src[2], a.rd)};
  const uint32_t wide = static_cast<uint32_t>(l32 * a.rd + 4 * hh) * 4u;
  f32x4 raw[3][4];
  auto load_chunk = [&](int m, int ec) {
#pragma unroll
    for (int t = 0; t < 4; ++t) raw[m][t] = load4(r[m], wide + static_cast<uint32_t>(32 * ec + 8 * t) * 4u);
  };
#pragma unroll
  for (int m = 0; m < 3; ++m) load_chunk(m, 0);
  const f32x16 zero = {};
  f32x16 acc[3][MB];  // dP_u, dP_v, W': rows = channels, lane = slot
#pragma unroll
  for (int m = 0; m < 3; ++m)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) acc[m][mb] = zero;
#pragma unroll 1
  for (int ec = 0; ec < ne; ++ec) {
    wait_vmcnt<0>();
    __syncthreads();  // chunk ec is there, and chunk ec - 1 has been read by every wave
    if (ec + 1 < ne) copier.copy(ec + 1, (ec + 1) & 1);
    const u32x4* fr = &ring[ec & 1][lane];
#pragma unroll
    for (int m = 0; m < 3; ++m) {
      X3 op[2];
#pragma unroll
      for (int s = 0; s < 2; ++s) op[s] = x3_split8([&](int j) { return raw[m][2 * s + (j >> 2)][j & 3]; });
      if (ec + 1 < ne) load_chunk(m, ec + 1);
#pragma unroll
      for (int f = 0; f < KS; ++f)
        acc[m][f >> 1] = x3_mma(ring_frag(fr + (m * KS + f) * 192), op[f & 1], acc[m][f >> 1]);
    }
  }
  mfma_drain();
  __syncthreads();  // the ring is free

  // dA_u = dP_u X'^T, dA_v = dP_v X'^T, dA_o = dY W'^T: 32x32 products of the pair's slots, of which
  // the two 16x16 blocks on the diagonal are its tiles.
  float* scratch = reinterpret_cast<float*>(&ring[0][0]) + wave * 32 * LD;
  f32x16 da[3];
  // x r (or dy) of the pair with lane = channel, through LDS to lane = slot: the operand of K step f.
  auto tiles = [&](const __amdgpu_buffer_rsrc_t& r, auto scaled, auto use) {
    float v[MB][16];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      const uint32_t ch = channel_offset(a, q * D + 32 * mb + l32);
#pragma unroll
      for (int i = 0; i < 16; ++i) v[mb][i] = load1(r, tab.off[wave][pair_token_row(i, hh)] + ch);
    }
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int t = pair_token_row(i, hh);
        scratch[t * LD + l32] = decltype(scaled)::value ? v[mb][i] * tab.scale[wave][t] : v[mb][i];
      }
      wave_lds_sync();
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const float* p = scratch + l32 * LD + 16 * s + 4 * hh;
        const f32x4 lo = *reinterpret_cast<const f32x4*>(p), hi = *reinterpret_cast<const f32x4*>(p + 8);
        use(2 * mb + s, x3_split8<true>([&](int j) { return j < 4 ? lo[j & 3] : hi[j & 3]; }));
      }
      wave_lds_sync();
    }
  };
  {
    f32x16 hi[2] = {zero, zero}, lo[2] = {zero, zero};
    tiles(routed.of(a.x, a), std::integral_constant<bool, true>{}, [&](int f, const X3& t) {
#pragma unroll
      for (int m = 0; m < 2; ++m) x3_mma_apart(x3_kstep(acc[m][f >> 1], f & 1), t, hi[m], lo[m]);
    });
    mfma_drain();
    da[0] = hi[0] + lo[0];
    da[1] = hi[1] + lo[1];
  }
  {
    f32x16 hi = zero, lo = zero;
    tiles(routed.of(a.dy, a), std::integral_constant<bool, false>{}, [&](int f, const X3& t) {
      x3_mma_apart(t, x3_kstep(acc[2][f >> 1], f & 1), hi, lo);
    });
    mfma_drain();
    da[2] = hi + lo;
  }
  float* sums = reinterpret_cast<float*>(&ring[0][0]) + 4 * 32 * LD;  // [wave][3][16][16]
#pragma unroll
  for (int m = 0; m < 3; ++m)
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      float v = lane & 16 ? da[m][8 + i] : da[m][i];
      v += __shfl_xor(v, 16);
      if (!(lane & 16)) sums[wave * 768 + m * 256 + pair_token_row(i, hh) * 16 + (l32 & 15)] = v;
    }

  const X3 au = token_operand(a.a_u, true, l32, hh), av = token_operand(a.a_v, true, l32, hh);
  int32_t row[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) row[i] = tab.row[wave][pair_token_row(i, hh)];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    f32x16 d0 = zero, d1 = zero;
#pragma unroll
    for (int m = 0; m < 2; ++m) {
#pragma unroll
      for (int k = 0; k < 4; ++k)
        *reinterpret_cast<f32x4*>(scratch + l32 * LD + 8 * k + 4 * hh) =
            f32x4{acc[m][mb][4 * k], acc[m][mb][4 * k + 1], acc[m][mb][4 * k + 2], acc[m][mb][4 * k + 3]};
      wave_lds_sync();
      float v[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) v[i] = scratch[pair_token_row(i, hh) * LD + l32];
      wave_lds_sync();
      const X3& t = m == 0 ? au : av;
      d0 = x3_mma(t, x3_split8([&](int j) { return v[j]; }), d0);
      d1 = x3_mma(t, x3_split8([&](int j) { return v[8 + j]; }), d1);
    }
    mfma_drain();
    const f32x16 dx = pair_rows_of(d0, d1);
    const int32_t ch = a.chan[q * D + 32 * mb + l32];
    if (ch >= 0 && ch < a.channels) {
#pragma unroll
      for (int i = 0; i < 16; ++i)
        if (row[i] >= 0) a.g[static_cast<int64_t>(row[i]) * a.channels + ch] = dx[i];
    }
  }
  __syncthreads();
  for (int i = tid; i < 768; i += kThreads)
    a.partial[(block * a.q_c + q) * 768 + i] = (sums[i] + sums[768 + i]) + (sums[1536 + i] + sums[2304 + i]);
}

// out[c] = the sum of partial[r][c] over the rows, c < 768, in fp64: 48 workgroups of 16 columns,
// 64 rows at a time (three workgroups of ow_sum_rows would take 49 rows one after the other at
// 28x28x256, B = 32, and their fp32 sum doubled the gradient's error).
__global__ void __launch_bounds__(1024) sum_token_grads_kernel(const float* p, int64_t rows, float* out) {
  __shared__ double part[64][17];
  const int c = threadIdx.x & 15, r0 = threadIdx.x >> 4;
  double s = 0.0;
#pragma unroll 4
  for (int64_t r = r0; r < rows; r += 64) s += static_cast<double>(p[r * 768 + 16 * blockIdx.x + c]);
  part[r0][c] = s;
  __syncthreads();
  for (int n = 32; n > 0; n >>= 1) {
    if (r0 < n) part[r0][c] += part[r0 + n][c];
    __syncthreads();
  }
  if (r0 == 0) out[16 * blockIdx.x + c] = static_cast<float>(part[0][c]);
}

struct ReduceX3Args {
  const float* narrow[3];  // P_u, P_v, dW' [q_c][slots][d]
  const float* wide[3];    // dU', dV', Z [q_c][slots][rd]
  float* partial;          // [ranges][3][q_c][d * rd]
  int64_t slots;
  int32_t q_c, ranges;
};

// One workgroup: a range of slots of one group and product, all of its d x rd outputs; a wave
// holds d x (rd / 4) of them.  Both operands have lane = column and the slots along K, so each
// value is read as it lies (two rows of 128 bytes per load) and split in the register it arrives
// in; the next 16 slots' loads are in flight during a step's products.  Bound by memory: at
// 28x28x256, B = 32 257 MB in 49 us, the copy's rate.
template <int D, int RD>
__global__ void __launch_bounds__(kThreads) reduce_x3_kernel(ReduceX3Args a) {
  constexpr int NB = D / 32, WB = RD / 128;
  const int lane = threadIdx.x & 63, l32 = lane & 31, hh = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
  int b = static_cast<int>(blockIdx.x);
  const int q = b % a.q_c;
  b /= a.q_c;
  const int kind = b % 3, range = b / 3;
  const int64_t steps = a.slots / 16;
  const int64_t first = steps * range / a.ranges, last = steps * (range + 1) / a.ranges;
  const float* np = a.narrow[kind] + (q * a.slots + 16 * first) * D + 8 * hh * D + l32;
  const float* wp = a.wide[kind] + (q * a.slots + 16 * first) * RD + 8 * hh * RD + 32 * WB * wave + l32;
  float n[NB][8], w[WB][8];
  auto load = [&] {
#pragma unroll
    for (int c = 0; c < NB; ++c)
#pragma unroll
      for (int j = 0; j < 8; ++j) n[c][j] = np[j * D + 32 * c];
#pragma unroll
    for (int c = 0; c < WB; ++c)
#pragma unroll
      for (int j = 0; j < 8; ++j) w[c][j] = wp[j * RD + 32 * c];
    np += 16 * D;
    wp += 16 * RD;
  };
  f32x16 acc[NB][WB];
#pragma unroll
  for (int i = 0; i < NB; ++i)
#pragma unroll
    for (int j = 0; j < WB; ++j) acc[i][j] = f32x16{};
  load();
  // The two orders of the operands give [d][rd] (lane = expanded row) and [rd][d] (lane = channel).
  auto run = [&](auto swapped) {
    constexpr bool kSwap = decltype(swapped)::value;
#pragma unroll 1
    for (int64_t s = first; s < last; ++s) {
      X3 no[NB], wo[WB];
#pragma unroll
      for (int c = 0; c < NB; ++c) no[c] = x3_split8([&](int j) { return n[c][j]; });
#pragma unroll
      for (int c = 0; c < WB; ++c) wo[c] = x3_split8([&](int j) { return w[c][j]; });
      if (s + 1 < last) load();
#pragma unroll
      for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int j = 0; j < WB; ++j)
          acc[i][j] = kSwap ? x3_mma(wo[j], no[i], acc[i][j]) : x3_mma(no[i], wo[j], acc[i][j]);
    }
    mfma_drain();
    float* out = a.partial + ((static_cast<int64_t>(range) * 3 + kind) * a.q_c + q) * D * RD;
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int j = 0; j < WB; ++j)
#pragma unroll
        for (int k = 0; k < 16; ++k) {
          const int rr = pair_token_row(k, hh), col = 32 * (WB * wave + j);
          if constexpr (kSwap)
            out[(col + rr) * D + 32 * i + l32] = acc[i][j][k];
          else
            out[(32 * i + rr) * RD + col + l32] = acc[i][j][k];
        }
  };
  if (kind == 2)
    run(std::integral_constant<bool, true>{});
  else
    run(std::integral_constant<bool, false>{});
}

int64_t blocks_of(int64_t slots, int32_t q_c) { return (slots + 127) / 128 * q_c; }

// Ranges of slots: about three workgroups a CU where the slots allow it, but no range below 256
// slots, whose operands are then six times the bytes of its partial sums (d = 64, rd = 128).
int64_t ranges_of(int64_t slots, int32_t q_c) {
  const int64_t want = (3 * static_cast<int64_t>(device_cus()) + 3 * q_c - 1) / (3 * q_c);
  return std::max<int64_t>(1, std::min<int64_t>(want, slots / 256));
}

bool shape_ok(int32_t d, int32_t rd) { return (d == 64 || d == 128) && (rd == 128 || rd == 256); }

}  // namespace
}  // namespace ow

extern "C" {

size_t ow_bwd_x3_packed_bytes(int32_t q_c, int32_t d, int32_t rd) {
  if (q_c < 1 || !ow::shape_ok(d, rd)) return 0;
  return static_cast<size_t>(q_c) * 6 * d * rd * 6;
}

int ow_pack_bwd_x3(const void* b_u, const void* b_v, const void* b_o, int32_t weight_dtype, const float* norm_weight,
                   const float* gamma, const int32_t* channel_index, int32_t channels, int32_t q_c, int32_t d,
                   int32_t rd, void* packed, size_t packed_bytes, void* stream) {
  OW_CHECK_SUPPORTED(ow::shape_ok(d, rd), "unsupported fp32 tile d=%d rd=%d", d, rd);
  OW_CHECK_ARG(q_c >= 1, "q_c must be >= 1");
  OW_CHECK_SUPPORTED(weight_dtype == OW_DTYPE_BF16 || weight_dtype == OW_DTYPE_F16 || weight_dtype == OW_DTYPE_F32,
                     "unsupported weight dtype %d", weight_dtype);
  OW_CHECK_ARG(b_u && b_v && b_o && channel_index && packed, "weight pointer is NULL");
  OW_CHECK_ARG(packed_bytes >= ow_bwd_x3_packed_bytes(q_c, d, rd), "packed buffer too small");
  OW_CHECK_ARG(ow::aligned16(packed), "packed must be 16-byte aligned");
  const int64_t total = static_cast<int64_t>(q_c) * 2 * (rd / 32) * 3 * (d / 16) * 64;
  ow::PackBwdX3Args p{{b_u, b_v, b_o}, norm_weight, gamma, channel_index, static_cast<uint4*>(packed), weight_dtype,
                      q_c, d, rd, channels, total};
  hipLaunchKernelGGL(ow::pack_bwd_x3_kernel, dim3(static_cast<unsigned>((total + 255) / 256)), dim3(ow::kThreads), 0,
                     static_cast<hipStream_t>(stream), p);
  if (int rc = ow::hip_status(hipGetLastError(), "pack_bwd_x3_kernel launch")) return rc;
  ow::clear_error();
  return OW_OK;
}

// A workgroup's offsets start at its first image: the images its 8 token groups can span.
int ow_bwd_x3_fits(int32_t n_tok, int32_t channels, int32_t q_s) {
  return q_s >= 1 && static_cast<int64_t>(8 / q_s + 2) * n_tok * channels * 4 < ow::kSpan;
}

int64_t ow_bwd_channel_x3_partials(int64_t slots, int32_t q_c) {
  return slots < 1 || q_c < 1 ? 0 : ow::blocks_of(slots, q_c);
}

int ow_bwd_channel_x3(const float* x, const float* dy, const float* rscale, const float* a_u, const float* a_v, const float* a_o,
                      const void* packed, size_t packed_bytes, float* pu, float* pv, float* dw, float* z, float* du,
                      float* dv, const int32_t* token_index, const int32_t* channel_index, int32_t batch, int32_t n_tok,
                      int32_t channels, int32_t q_s, int32_t q_c, int32_t d, int32_t rd, float* g, float* partial,
                      int64_t n_partial, float* d_a, void* stream) {
  const int64_t slots = static_cast<int64_t>(batch) * q_s * 16;
  OW_CHECK_SUPPORTED(ow::shape_ok(d, rd), "unsupported fp32 tile d=%d rd=%d", d, rd);
  OW_CHECK_ARG(batch >= 0, "batch must be >= 0 (got %d)", batch);
  OW_CHECK_ARG(q_c >= 1 && q_s >= 1 && n_tok >= 1 && channels >= 1, "sizes must be positive");
  OW_CHECK_ARG(packed && packed_bytes >= ow_bwd_x3_packed_bytes(q_c, d, rd), "packed weights missing or too small");
  OW_CHECK_SUPPORTED(ow_bwd_x3_fits(n_tok, channels, q_s), "images too large for 32-bit offsets");
  if (slots == 0) {
    ow::clear_error();
    return OW_OK;
  }
  OW_CHECK_ARG(x && dy && a_u && a_v && a_o && pu && pv && dw && z && du && dv && token_index && channel_index && g &&
                   partial && d_a,
               "tensor pointer is NULL");
  for (const void* p : {packed, static_cast<const void*>(pu),
                        static_cast<const void*>(pv), static_cast<const void*>(dw), static_cast<const void*>(z),
                        static_cast<const void*>(du), static_cast<const void*>(dv)})
    OW_CHECK_ARG(ow::aligned16(p), "tile buffers must be 16-byte aligned");
  const int64_t blocks = ow::blocks_of(slots, q_c);
  OW_CHECK_ARG(n_partial == blocks, "n_partial must be %lld", (long long)blocks);
  OW_CHECK_SUPPORTED(blocks + 8 * q_c < (int64_t(1) << 31) && static_cast<int64_t>(batch) * n_tok < (int64_t(1) << 31),
                     "too many slots for one launch");
  ow::ChanX3Args a{x, dy, rscale, a_u, a_v, a_o, static_cast<const uint8_t*>(packed), pu, pv, dw, z, du, dv, g, partial,
                   token_index, channel_index, slots, q_c, rd, n_tok, channels, q_s,
                   batch};
  const dim3 grid(static_cast<unsigned>((blocks / q_c + 7) / 8 * 8 * q_c)), threads(ow::kThreads);
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (d == 64)
    hipLaunchKernelGGL(ow::chan_x3_kernel<64>, grid, threads, 0, s, a);
  else
    hipLaunchKernelGGL(ow::chan_x3_kernel<128>, grid, threads, 0, s, a);
  if (int rc = ow::hip_status(hipGetLastError(), "chan_x3_kernel launch")) return rc;
  if (d == 64)
    hipLaunchKernelGGL(ow::chan2_x3_kernel<64>, grid, threads, 0, s, a);
  else
    hipLaunchKernelGGL(ow::chan2_x3_kernel<128>, grid, threads, 0, s, a);
  if (int rc = ow::hip_status(hipGetLastError(), "chan2_x3_kernel launch")) return rc;
  hipLaunchKernelGGL(ow::sum_token_grads_kernel, dim3(48), dim3(1024), 0, s, partial, blocks, d_a);
  if (int rc = ow::hip_status(hipGetLastError(), "sum_token_grads_kernel launch")) return rc;
  ow::clear_error();
  return OW_OK;
}

int64_t ow_bwd_param_reduce_x3_ranges(int64_t slots, int32_t q_c) {
  return slots < 1 || q_c < 1 ? 0 : ow::ranges_of(slots, q_c);
}

int ow_bwd_param_reduce_x3(const float* pu, const float* pv, const float* dw, const float* z, const float* du,
                           const float* dv, float* partial, int64_t ranges, int64_t slots, int32_t q_c, int32_t d,
                           int32_t rd, void* stream) {
  OW_CHECK_SUPPORTED(ow::shape_ok(d, rd), "unsupported fp32 tile d=%d rd=%d", d, rd);
  OW_CHECK_ARG(slots >= 16 && slots % 16 == 0, "slots must be a positive multiple of 16 (got %lld)", (long long)slots);
  OW_CHECK_ARG(q_c >= 1 && pu && pv && dw && z && du && dv && partial, "tensor pointer is NULL");
  OW_CHECK_ARG(ranges >= 1 && ranges <= slots / 16, "ranges must be in [1, slots / 16]");
  const int64_t blocks = ranges * 3 * q_c;
  OW_CHECK_SUPPORTED(blocks < (int64_t(1) << 31), "too many ranges");
  ow::ReduceX3Args a{{pu, pv, dw}, {du, dv, z}, partial, slots, q_c, static_cast<int32_t>(ranges)};
  const dim3 grid(static_cast<unsigned>(blocks)), threads(ow::kThreads);
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (d == 64 && rd == 128)
    hipLaunchKernelGGL((ow::reduce_x3_kernel<64, 128>), grid, threads, 0, s, a);
  else if (d == 64)
    hipLaunchKernelGGL((ow::reduce_x3_kernel<64, 256>), grid, threads, 0, s, a);
  else if (rd == 128)
    hipLaunchKernelGGL((ow::reduce_x3_kernel<128, 128>), grid, threads, 0, s, a);
  else
    hipLaunchKernelGGL((ow::reduce_x3_kernel<128, 256>), grid, threads, 0, s, a);
  if (int rc = ow::hip_status(hipGetLastError(), "reduce_x3_kernel launch")) return rc;
  ow::clear_error();
  return OW_OK;
}

}  // extern "C"
