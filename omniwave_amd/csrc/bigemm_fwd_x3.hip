// fp32 BiGEMM forward on the bf16 matrix cores (three-part operands, ow_x3.h): the operator of
// omniweave/ops/reference.py:120-173 with the block's RMSNorm prologue and residual epilogue
// (omniweave/models/block.py:83-108) for fp32 activations, any supported shape and route.
//
// A unit is one 32-token pair (two token groups) of one channel group, computed by the operand
// scheme of ow_device.h (32x32x16 products, accumulators reused as the next operand) with every
// operand in three bf16 parts and the groups' token products apart.  Every shape takes this one
// kernel: x is read and out written by the lane that owns the channel, so contiguous, strided and
// ragged groups differ only in the channel table.
//
// What bounds it: the products.  A d = 128, rd = 256 unit is 1,296 of them, 41,500 cycles of one
// SIMD; the chunk loop runs at 42 cycles a product (32 alone; the rest is the gate, the splits
// and the slices' barriers).  The operator at 14x14x512, B = 32, this kernel alone, takes 34.4 us
// (152 TFLOP/s of fp32 work; 832 units on 1,024 SIMDs), the block with its residual and statistics
// pass 38, against 180 us for fp32 FMAs staged through LDS, and the error against 64 bits falls
// (block 1.9e-7 rel-L2 against 2.3e-7, delta 2.9e-7 against 4.5e-7) since one fp32 addition takes
// a K step of 16 instead of one element.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "ow_common.h"
#include "ow_x3.h"

namespace ow {
namespace {

constexpr int kX3Threads = 256;
constexpr int64_t kX3Span = int64_t(1) << 30;  // addressable bytes from a workgroup's first image
constexpr int kX3HeadFloats = 3 * kG * kG;  // A_u, A_v, A_o row-major at the head of the packed weights

__device__ __forceinline__ float load_weight(const void* p, int64_t i, int dtype) {
  if (dtype == OW_DTYPE_F32) return static_cast<const float*>(p)[i];
  const uint16_t u = static_cast<const uint16_t*>(p)[i];
  return dtype == OW_DTYPE_BF16 ? BF16::to_f32(u) : F16::to_f32(u);
}

struct PackX3Args {
  const void* a[3];
  const void* b_u;
  const void* b_v;
  const void* b_o;
  const float* norm_w;
  const float* gamma;
  const int32_t* chan;
  uint8_t* packed;
  int32_t wdtype, q_c, d, rd, channels;
  int64_t total;  // operand lanes: q_c * (rd / 32) * 3 * (d / 16) * 64
};

// One thread per operand lane: the 8 folded values of a fragment's lane, in three parts.  The
// folds are formed in fp64, so the parts hold the exact product rounded once.
__global__ void __launch_bounds__(256) pack_x3_kernel(PackX3Args p) {
  const int64_t idx = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (idx < kX3HeadFloats)
    reinterpret_cast<float*>(p.packed)[idx] = load_weight(p.a[idx / (kG * kG)], idx % (kG * kG), p.wdtype);
  if (idx >= p.total) return;
  const int lane = static_cast<int>(idx & 63), l32 = lane & 31, hh = lane >> 5;
  const int ks_n = p.d / 16, nch = p.rd / 32;
  int64_t rem = idx >> 6;
  const int f = static_cast<int>(rem % ks_n);  // K step of B_u / B_v, (block, K half) of B_o
  rem /= ks_n;
  const int kind = static_cast<int>(rem % 3);
  rem /= 3;
  const int ec = static_cast<int>(rem % nch);
  const int q = static_cast<int>(rem / nch);
  const double fold = kind == 0 ? -1.4426950408889634 : kind == 1 ? -0.6931471805599453 : 1.0;
  const float* vec = kind < 2 ? p.norm_w : p.gamma;
  uint32_t w[3][4];
#pragma unroll
  for (int j2 = 0; j2 < 4; ++j2) {
    uint32_t part[3][2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int k = pair_token_row(2 * j2 + h, hh);  // kord of the slot
      int c, e;
      if (kind < 2) {
        c = 16 * f + k;
        e = 32 * ec + l32;
      } else {
        c = 32 * (f >> 1) + l32;
        e = 32 * ec + 16 * (f & 1) + k;
      }
      double v = fold;
      if (p.chan) {
        const int gc = p.chan[q * p.d + c];
        const bool ok = gc >= 0 && gc < p.channels;
        v = ok ? (vec ? v * static_cast<double>(vec[gc]) : v) : 0.0;
      }
      const int64_t mat = static_cast<int64_t>(p.d) * p.rd;
      const int64_t src = static_cast<int64_t>(q) * mat +
                          (kind < 2 ? static_cast<int64_t>(c) * p.rd + e : static_cast<int64_t>(e) * p.d + c);
      v *= static_cast<double>(load_weight(kind == 0 ? p.b_u : kind == 1 ? p.b_v : p.b_o, src, p.wdtype));
#pragma unroll
      for (int n = 0; n < 3; ++n) part[n][h] = x3_part(v, n);
    }
#pragma unroll
    for (int n = 0; n < 3; ++n) w[n][j2] = part[n][0] | (part[n][1] << 16);
  }
  uint4* dst = reinterpret_cast<uint4*>(p.packed + kX3HeadFloats * 4) + (idx >> 6) * 3 * 64 + lane;
#pragma unroll
  for (int n = 0; n < 3; ++n) dst[64 * n] = uint4{w[n][0], w[n][1], w[n][2], w[n][3]};
}

// The gate with silu(U) formed before V comes in: a large U V beside a vanishing sigmoid is zero,
// where (U V) s (silu_gate) overflows.
__device__ __forceinline__ float silu_first(float up, float vp) {
  return up * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(up)) * vp;
}

struct X3Args {
  const float* x;
  float* out;
  const float* row_scale;  // NULL: no RMSNorm, or the kernel forms the scales (norm)
  const uint8_t* packed;
  const int32_t* tok;
  const int32_t* chan;
  const float* drop_scale;  // [batch] per-image multiplier of delta (drop-path); NULL: none
  int32_t batch, n_tok, channels, q_s, q_c, residual;
  int32_t n_groups;  // batch * q_s token groups
  int32_t norm;      // S = 4: form the RMSNorm scales here
  float eps;
  int32_t interleaved;  // radix channel groups
};

// S waves share a pair, each with an S-th of the expanded dimension (W summed over them at the
// end); the workgroup's four waves hold 4 / S pairs of one channel group.  The weights of the
// group arrive as slices of one chunk's B_u, B_v or B_o fragments (for d = 128 and S = 4 halves
// of them) in a ring of three LDS stages, copied two slices ahead.
template <int D, int RD, int S>
__global__ void __launch_bounds__(kX3Threads) __attribute__((amdgpu_waves_per_eu(D == 64 && S < 4 ? 2 : 1, D == 64 && S < 4 ? 2 : 1)))
bigemm_fwd_x3_kernel(X3Args a) {
  constexpr int KS = D / 16, MB = D / 32, NE = RD / 32 / S;
  constexpr int HS = (D == 128 && S == 4) ? 2 : 1;  // slices per fragment kind
  constexpr int FR = 3 * KS / HS;                   // 1 KB fragments of one slice
  constexpr int STAGE = S * FR;
  constexpr int NS = 3 * NE * HS;                   // slices of one wave's chunks
  constexpr int CP = STAGE / 4;                     // copies per wave and slice
  constexpr int NP = 4 / S;                         // pairs of the workgroup
  constexpr bool PIPE = D == 128;
  static_assert(STAGE % 4 == 0 && (KS / HS) % 2 == 0, "slice split");
  __shared__ __attribute__((aligned(16))) u32x4 ring[3][STAGE * 64];
  __shared__ __attribute__((aligned(16))) uint32_t s_off[NP][32];  // byte offset of each token's row
  __shared__ __attribute__((aligned(16))) float s_scale[NP][32];

  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, hh = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int sub = wave % S, pl = wave / S;
  // Interleaved groups share the lines of x and out: the q_c groups of one block of pairs lie 8
  // workgroups apart, on one XCD (round-robin dispatch), whose L2 serves them (radix 1, B = 32:
  // 28x28x256 77 -> 60 us, 14x14x512 59 -> 52).  Contiguous groups share nothing, and an XCD then
  // reads one group's weights only where q_c divides 8 (the other order costs them 2 to 5%).
  const int bid = static_cast<int>(blockIdx.x);
  const int q = a.interleaved ? bid / 8 % a.q_c : bid % a.q_c;
  const int pair0 = (a.interleaved ? bid / (8 * a.q_c) * 8 + bid % 8 : bid / a.q_c) * NP;
  if (2 * pair0 >= a.n_groups) return;

  const uint16_t* planes = reinterpret_cast<const uint16_t*>(a.packed + kX3HeadFloats * 4) +
                           static_cast<int64_t>(q) * (RD / 32) * 9 * KS * kFragElems;
  const uint32_t lane16 = 16u * static_cast<uint32_t>(lane);
  // Slice n of a wave's sequence: U V O of each chunk, or (PIPE: one wave per SIMD, whose gate
  // runs beside the next chunk's U products) U0 V0, then U V of chunk m + 1 and O of chunk m, and
  // the last O.
  auto source = [&](int n) {  // chunk, kind and half of slice n, as the fragment offset of its start
    const int k = n / HS, half = n % HS;
    int e, kind;
    if constexpr (!PIPE) {
      e = k / 3;
      kind = k % 3;
    } else if (k < 2) {
      e = 0;
      kind = k;
    } else if (k == 3 * NE - 1) {
      e = NE - 1;
      kind = 2;
    } else {
      const int m = (k - 2) / 3;
      kind = (k - 2) % 3;
      e = kind == 2 ? m : m + 1;
    }
    return (e * 3 + kind) * 3 * KS + half * FR;
  };
  // This wave's CP fragments of a slice are contiguous in the packed weights and in the stage:
  // those from f0 of the stage on, of the chunks of wave f0 / FR of the pair.
  const int f0 = wave * CP;
  const uint8_t* own = reinterpret_cast<const uint8_t*>(
      uniform_ptr(planes + (static_cast<int64_t>(f0 / FR) * NE * 9 * KS + f0 % FR) * kFragElems));
  const uint32_t own_lds = lds_addr(&ring[0][0]) + static_cast<uint32_t>(f0) * 1024;
  auto copy_piece = [&](const uint8_t* src, int buf, int i) {
    copy_frag_to_lds_at(reinterpret_cast<const uint16_t*>(src + i * 1024), own_lds + (buf * STAGE + i) * 1024, lane16);
  };
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int i = 0; i < CP; ++i) copy_piece(own + source(s) * 1024, s, i);

  // x and out from the first image of the workgroup's pairs on, as buffers of at most 1 GiB: a pad
  // slot's row offset lies at 2 GiB, a pad channel's at 1 GiB, so what either asks for reads as
  // zero and stores nowhere, without a branch.
  const int img0 = 2 * pair0 / a.q_s;
  const int64_t img_elems = static_cast<int64_t>(a.n_tok) * a.channels;
  const int64_t left = (static_cast<int64_t>(a.batch) - img0) * img_elems * 4;
  const uint32_t span = static_cast<uint32_t>(left < kX3Span ? left : kX3Span);
  const __amdgpu_buffer_rsrc_t rx = buffer_rsrc(a.x + img0 * img_elems, span);
  const __amdgpu_buffer_rsrc_t ro = buffer_rsrc(a.out + img0 * img_elems, span);

  if (tid < 32 * NP) {
    const int t = tid & 31;
    const int g = 2 * (pair0 + (tid >> 5)) + (t >> 4);
    uint32_t off = kOffOut;
    float r = 0.0f;
    if (g < a.n_groups) {
      const int b = g / a.q_s, s = g - b * a.q_s;
      const int32_t tk = a.tok[s * kG + (t & 15)];
      if (tk >= 0 && tk < a.n_tok) {
        off = static_cast<uint32_t>((b - img0) * a.n_tok + tk) * static_cast<uint32_t>(a.channels) * 4u;
        r = a.row_scale ? a.row_scale[static_cast<int64_t>(b) * a.n_tok + tk] : 1.0f;
      }
    }
    s_off[tid >> 5][t] = off;
    s_scale[tid >> 5][t] = r;
  }
  const float* head = reinterpret_cast<const float*>(a.packed) + (l32 & 15) * kG + 4 * hh;
  auto token_operand = [&](int m) {  // row l32 % 16 of A_m in the K order of the pair scheme
    const float* p = head + m * kG * kG;
    const float4 lo = *reinterpret_cast<const float4*>(p), hi = *reinterpret_cast<const float4*>(p + 8);
    const float v[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
    return x3_split8<true>([&](int j) { return v[j]; });
  };
  const bool g0 = (lane & 16) == 0;
  __syncthreads();
  if constexpr (S == 4) {
    if (a.norm) {  // eight lanes a row, 128 bytes of it a step (a ragged row's last vector is cut off)
      const uint32_t base = s_off[0][tid >> 3];
      f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 8
      for (int c = 4 * (tid & 7); c < a.channels; c += 32) {
        const f32x4 v = __builtin_bit_cast(
            f32x4, __builtin_amdgcn_raw_buffer_load_b128(rx, static_cast<int>(base + 4u * static_cast<uint32_t>(c)), 0, 0));
#pragma unroll
        for (int k = 0; k < 4; ++k) acc[k] = c + k < a.channels ? fmaf(v[k], v[k], acc[k]) : acc[k];
      }
      float sum = (acc[0] + acc[1]) + (acc[2] + acc[3]);
#pragma unroll
      for (int m = 4; m > 0; m >>= 1) sum += __shfl_xor(sum, m);
      if ((tid & 7) == 0) s_scale[0][tid >> 3] = base == kOffOut ? 0.0f : 1.0f / sqrtf(sum / static_cast<float>(a.channels) + a.eps);
      __syncthreads();
    }
  }

  auto channel = [&](int mb) -> uint32_t {  // byte offset of the lane's channel of a 32-channel block
    const int32_t ch = a.chan[q * D + 32 * mb + l32];
    return ch >= 0 && ch < a.channels ? 4u * static_cast<uint32_t>(ch) : static_cast<uint32_t>(kX3Span);
  };
  // Row offsets of the lane's tokens kord(0..15), and x of one channel at them.
  uint32_t row[16];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const u32x4 v = *reinterpret_cast<const u32x4*>(&s_off[pl][8 * k + 4 * hh]);
#pragma unroll
    for (int j = 0; j < 4; ++j) row[4 * k + j] = v[j];
  }
  auto load_x = [&](uint32_t ch, float(&v)[16]) {
#pragma unroll
    for (int i = 0; i < 16; ++i)
      v[i] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rx, static_cast<int>(row[i] + ch), 0, 0));
  };

  // Token side: P_u, P_v of the pair as K-step operands.
  X3 Pu[KS], Pv[KS];
  const f32x16 zero = {};
  {
    const X3 au = token_operand(0), av = token_operand(1);
    float raw[MB][16];  // x of the pair: all 16 MB loads per lane in flight at once
#pragma unroll
    for (int cb = 0; cb < MB; ++cb) load_x(channel(cb), raw[cb]);
    float sc[16];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const f32x4 v = *reinterpret_cast<const f32x4*>(&s_scale[pl][8 * k + 4 * hh]);
#pragma unroll
      for (int j = 0; j < 4; ++j) sc[4 * k + j] = v[j];
    }
#pragma unroll
    for (int cb = 0; cb < MB; ++cb) {
      f32x16 pg[2][2];
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        const X3 xt = x3_split8<true>([&](int j) { return raw[cb][8 * g + j] * sc[8 * g + j]; });
        pg[0][g] = x3_mma(xt, au, zero);
        pg[1][g] = x3_mma(xt, av, zero);
      }
      mfma_drain();
      const f32x16 pu = pair_columns(g0, pg[0][0], pg[0][1]), pv = pair_columns(g0, pg[1][0], pg[1][1]);
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        Pu[2 * cb + s] = x3_kstep(pu, s);
        Pv[2 * cb + s] = x3_kstep(pv, s);
      }
    }
  }

  f32x16 W[MB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) W[mb] = zero;
  f32x16 U, V;
  X3 Z[2];
  // The stream of K steps: step i lies in slice i / SK, buffer (i / SK) % 3.  One wave per SIMD
  // (d = 128) hides nothing behind another wave, and its products form one dependent chain (32
  // cycles each), so everything else is placed between two products, in pieces that fit there:
  // the next step's fragment reads, one copy of the slice after next, and `side` work.  Left where
  // the compiler put them, in clumps between two steps, the same instructions took a d = 128 chunk
  // from 6,050 to 7,700 cycles (4,608 of products).
  constexpr int SK = KS / HS;  // K steps of one slice
  const uint32_t ring0 = lds_addr(&ring[0][0]) + static_cast<uint32_t>(sub * FR) * 1024 + lane16;
  const uint32_t ring1 = ring0 + 65536u;  // LDS offsets are 16 bits wide
  X3 fr[2];
  int n = 0;                      // slices made readable so far
  const uint8_t* ahead = nullptr; // this wave's part of the slice after next, copied during a slice's
  bool more = false;              // steps, and whether there is one
  auto fetch = [&](auto step) {
    constexpr int i = decltype(step)::value;
    if constexpr (i % SK == 0) {
      // Slice n is in its buffer, and slice n - 1 has been read by every wave.
      if (n + 1 >= NS)
        wait_vmcnt<0>();
      else
        wait_vmcnt<CP * (SK - 1) / SK>();  // copies of slice n + 1 issued by now
      __syncthreads();
      ++n;
    }
    constexpr int off = ((i / SK) % 3) * STAGE * 1024 + (i % SK) * 3072;
    X3& f = fr[i & 1];
    if constexpr (off + 2048 < 65536) {
      f.p[2] = lds_read_async<off + 2048>(ring0);
      f.p[1] = lds_read_async<off + 1024>(ring0);
      f.p[0] = lds_read_async<off>(ring0);
    } else {
      constexpr int o = off - 65536 < 0 ? 0 : off - 65536;
      const uint32_t base = off - 65536 < 0 ? ring1 - static_cast<uint32_t>(65536 - off) : ring1;
      f.p[2] = lds_read_async<o + 2048>(base);
      f.p[1] = lds_read_async<o + 1024>(base);
      f.p[0] = lds_read_async<o>(base);
    }
  };
  auto no = std::integral_constant<bool, false>{};
  auto yes = std::integral_constant<bool, true>{};
  // Steps [first, last): product(j, f, i) is the j-th of step i's six products (smallest first,
  // part 2 - j % 3 .. of the fragment), side(j, i) other work for three of the gaps.
  auto steps = [&](auto first, auto last, auto final, auto product, auto side) {
    static_for<decltype(first)::value, decltype(last)::value>([&](auto step) {
      constexpr int i = decltype(step)::value;
      X3& f = fr[i & 1];
      lds_wait<0>(f.p[2]);  // also: no read of this slice is in flight at the next barrier
      lds_wait<0>(f.p[1]);
      lds_wait<0>(f.p[0]);
      if constexpr (i % SK == 0) {
        more = n + 1 < NS;
        ahead = own + source(more ? n + 1 : 0) * 1024;
      }
      if constexpr (!(decltype(final)::value && i + 1 == decltype(last)::value))
        fetch(std::integral_constant<int, i + 1>{});
      static_for<0, 6>([&](auto j) {
        __builtin_amdgcn_sched_barrier(0);
        product(j, f, step);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (decltype(j)::value == 1) {
          if (more) {
#pragma unroll
            for (int c = CP * (i % SK) / SK; c < CP * (i % SK + 1) / SK; ++c) copy_piece(ahead, (i / SK + 2) % 3, c);
          }
        } else if constexpr (decltype(j)::value >= 2 && decltype(j)::value < 5) {
          side(std::integral_constant<int, decltype(j)::value - 2>{}, step);
        }
      });
    });
  };
  constexpr int kF[6] = {2, 1, 0, 1, 0, 0}, kOther[6] = {0, 1, 2, 0, 1, 0};  // parts of the six products
  auto u_step = [&](auto j, const X3& f, auto i) {
    constexpr int n = decltype(j)::value;
    U = BF16::mma32(f.p[kF[n]], Pu[decltype(i)::value % KS].p[kOther[n]], U);
  };
  auto v_step = [&](auto j, const X3& f, auto i) {
    constexpr int n = decltype(j)::value;
    V = BF16::mma32(f.p[kF[n]], Pv[decltype(i)::value % KS].p[kOther[n]], V);
  };
  auto w_step = [&](auto j, const X3& f, auto i) {
    constexpr int n = decltype(j)::value, k = decltype(i)::value % KS;
    W[k / 2] = BF16::mma32(Z[k % 2].p[kOther[n]], f.p[kF[n]], W[k / 2]);
  };
  auto idle = [](auto, auto) {};
  constexpr std::integral_constant<int, 0> i0{};
  constexpr std::integral_constant<int, KS> i1{};
  constexpr std::integral_constant<int, 2 * KS> i2{};
  constexpr std::integral_constant<int, 3 * KS> i3{};
  constexpr std::integral_constant<int, 4 * KS> i4{};
  constexpr std::integral_constant<int, 5 * KS> i5{};
  auto gate_all = [&] {
    f32x16 z;
#pragma unroll
    for (int i = 0; i < 16; ++i) z[i] = silu_first(U[i], V[i]);
    Z[0] = x3_kstep(z, 0);
    Z[1] = x3_kstep(z, 1);
  };
  // The residual's x of the blocks this wave will store, requested before the last W products (P
  // is dead by then, and its registers hold them).
  constexpr int NB = MB >= S ? MB / S : 1;
  float res[NB][16] = {};
  uint32_t och[NB];
  auto load_residual = [&] {
    if (sub * NB < MB) {
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        och[j] = channel(sub * NB + j);
        if (a.residual) load_x(och[j], res[j]);
      }
    }
  };
  fetch(i0);
  if constexpr (PIPE) {
    U = zero;
    V = zero;
    steps(i0, i1, no, u_step, idle);
    steps(i1, i2, no, v_step, idle);
    mfma_drain();
#pragma unroll 1
    for (int e = 0; e + 1 < NE; ++e) {
      const f32x16 u0 = U, v0 = V;
      U = zero;
      V = zero;
      // The gate of chunk e beside the U products of chunk e + 1: values 2k, 2k + 1 in K step k.
      // The empty asm keeps each piece in its gap (pure arithmetic moves across the scheduling
      // barriers before they apply).
      float den[2], num[2];
      auto pin = [](float(&v)[2]) { asm volatile("" : "+v"(v[0]), "+v"(v[1])); };
      steps(i2, i3, no, u_step, [&](auto j, auto i) {
        constexpr int k = decltype(i)::value - 2 * KS;
        if constexpr (decltype(j)::value == 0) {
          for (int h = 0; h < 2; ++h) den[h] = u0[2 * k + h];
          pin(den);
          for (int h = 0; h < 2; ++h) den[h] = 1.0f + __builtin_amdgcn_exp2f(den[h]);
        } else if constexpr (decltype(j)::value == 1) {
          pin(den);
          for (int h = 0; h < 2; ++h) num[h] = u0[2 * k + h] * __builtin_amdgcn_rcpf(den[h]) * v0[2 * k + h];  // as silu_first
        } else {
          pin(num);
          uint32_t p0, p1, p2;
          x3_split2(num[0], num[1], p0, p1, p2);
          asm volatile("" : "+v"(p0), "+v"(p1), "+v"(p2));
          Z[k / 4].p[0][k % 4] = p0;
          Z[k / 4].p[1][k % 4] = p1;
          Z[k / 4].p[2][k % 4] = p2;
        }
      });
      steps(i3, i4, no, v_step, idle);
      steps(i4, i5, no, w_step, idle);
      mfma_drain();
    }
    load_residual();
    gate_all();
    steps(i2, i3, yes, w_step, idle);
  } else {
    auto chunk = [&](auto final) {
      U = zero;
      V = zero;
      steps(i0, i1, no, u_step, idle);
      steps(i1, i2, no, v_step, idle);
      mfma_drain();
      if constexpr (decltype(final)::value) load_residual();
      gate_all();
      steps(i2, i3, final, w_step, idle);
    };
#pragma unroll 1
    for (int e = 0; e + 1 < NE; ++e) chunk(no);
    chunk(yes);
  }
  mfma_drain();

  // delta = A_o W, residual and routed store of one 32-channel block.
  const X3 ao = token_operand(2);
  float ds[2] = {1.0f, 1.0f};
  if (a.drop_scale) {
#pragma unroll
    for (int g = 0; g < 2; ++g) ds[g] = a.drop_scale[min(2 * (pair0 + pl) + g, a.n_groups - 1) / a.q_s];
  }
  auto store = [&](uint32_t ch, const f32x16& w, float(&xv)[16]) {
    const f32x16 d0 = x3_mma(ao, x3_kstep(w, 0), zero), d1 = x3_mma(ao, x3_kstep(w, 1), zero);
    mfma_drain();
    f32x16 dl = pair_rows_of(d0, d1);
    if (a.drop_scale) {
#pragma unroll
      for (int i = 0; i < 16; ++i) dl[i] *= ds[i >> 3];
    }
    if (a.residual) {
#pragma unroll
      for (int i = 0; i < 16; ++i) dl[i] += xv[i];
    }
#pragma unroll
    for (int i = 0; i < 16; ++i)
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(dl[i]), ro, static_cast<int>(row[i] + ch), 0, 0);
  };
  if constexpr (S == 1) {
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) store(och[mb], W[mb], res[mb]);
  } else {
    // The S waves' partial W through LDS (the ring is no longer read), summed in wave order; each
    // wave finishes its share of the 32-channel blocks.
    static_assert(sizeof(ring) >= 4 * MB * 16 * 64 * sizeof(float), "partial W fits the ring");
    f32x4* part = reinterpret_cast<f32x4*>(&ring[0][0]);
    __syncthreads();
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        part[((wave * MB + mb) * 4 + i) * 64 + lane] = f32x4{W[mb][4 * i], W[mb][4 * i + 1], W[mb][4 * i + 2], W[mb][4 * i + 3]};
    __syncthreads();
    if (sub * NB < MB) {
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        const int mb = sub * NB + j;
        f32x16 w;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          f32x4 v = part[((pl * S * MB + mb) * 4 + i) * 64 + lane];
#pragma unroll
          for (int s = 1; s < S; ++s) v += part[(((pl * S + s) * MB + mb) * 4 + i) * 64 + lane];
#pragma unroll
          for (int k = 0; k < 4; ++k) w[4 * i + k] = v[k];
        }
        store(och[j], w, res[j]);
      }
    }
  }
}

// With fewer units than four per CU the waves of a workgroup share one pair (or two) and its
// expanded dimension: a workgroup still holds one CU, and each unit is done sooner.  Measured on
// an earlier form of the loop at 14x14x512: B = 8 (208 units) 24 us split in four, 30 in two, 42
// whole; B = 16 (416) 41, 33, 44; B = 32 (832) 77, 60, 49.  d = 64 crosses at the same counts
// (28x28x256, 196 units: 12.8, 13.6, 17.9; 392: 21, 15, 18; 784: 38, 21, 20).
int x3_split(int64_t units) {
  const int64_t cus = device_cus();
  return units <= cus ? 4 : units <= 2 * cus ? 2 : 1;
}

template <int D, int RD>
int launch_x3(const X3Args& a, int32_t n_pairs, int split, hipStream_t stream) {
  const int64_t blocks = (n_pairs + 4 / split - 1) / (4 / split);
  const unsigned grid = static_cast<unsigned>((a.interleaved ? (blocks + 7) / 8 * 8 : blocks) * a.q_c);
  if (split == 4)
    hipLaunchKernelGGL((bigemm_fwd_x3_kernel<D, RD, 4>), dim3(grid), dim3(kX3Threads), 0, stream, a);
  else if (split == 2)
    hipLaunchKernelGGL((bigemm_fwd_x3_kernel<D, RD, 2>), dim3(grid), dim3(kX3Threads), 0, stream, a);
  else
    hipLaunchKernelGGL((bigemm_fwd_x3_kernel<D, RD, 1>), dim3(grid), dim3(kX3Threads), 0, stream, a);
  return hip_status(hipGetLastError(), "bigemm_fwd_x3_kernel launch");
}

}  // namespace

bool x3_fits(int32_t n_tok, int32_t channels, int32_t q_s) {
  return static_cast<int64_t>(8 / q_s + 2) * n_tok * channels * 4 < kX3Span;
}

size_t packed_bytes_x3(int32_t q_c, int32_t d, int32_t rd) {
  return static_cast<size_t>(kX3HeadFloats) * 4 + static_cast<size_t>(q_c) * 3 * d * rd * 6;
}

int pack_weights_x3(const void* a_u, const void* a_v, const void* a_o, const void* b_u, const void* b_v,
                    const void* b_o, int32_t weight_dtype, const float* norm_weight, const float* gamma,
                    const int32_t* channel_index, int32_t channels, int32_t q_c, int32_t d, int32_t rd, void* packed,
                    hipStream_t stream) {
  const int64_t total = static_cast<int64_t>(q_c) * (rd / 32) * 3 * (d / 16) * 64;  // >= kX3HeadFloats
  PackX3Args p{{a_u, a_v, a_o}, b_u, b_v, b_o, norm_weight, gamma, channel_index, static_cast<uint8_t*>(packed),
               weight_dtype, q_c, d, rd, channels, total};
  hipLaunchKernelGGL(pack_x3_kernel, dim3(static_cast<unsigned>((total + 255) / 256)), dim3(256), 0, stream, p);
  return hip_status(hipGetLastError(), "pack_x3_kernel launch");
}

// Split in four, a workgroup holds one pair and forms its rows' RMSNorm scales itself: 32 rows by
// 256 threads, read by the q_c workgroups of the pair from L2, against a launch of its own.
// 14x14x512, B = 8: 2.4 us more in this kernel against a pass of 4.3 and the gap before it; with
// whole pairs per wave four times the rows would wait for their reads, beside a pass of 6 us in 40.
bool x3_forms_scales(int32_t batch, int32_t q_s, int32_t q_c) {
  return x3_split((static_cast<int64_t>(batch) * q_s + 1) / 2 * q_c) == 4;
}

int launch_fwd_x3(const float* x, float* out, const float* row_scale, bool norm, float eps, bool interleaved, const void* packed,
                  const int32_t* tok, const int32_t* chan, int32_t batch, int32_t n_tok, int32_t channels, int32_t q_s,
                  int32_t q_c, int32_t d, int32_t rd, int32_t residual, const float* drop_scale, hipStream_t stream) {
  const int64_t groups = static_cast<int64_t>(batch) * q_s;
  if (groups >= (int64_t(1) << 31)) return fail(OW_ERR_UNSUPPORTED, "batch * token groups must be below 2^31");
  X3Args a{x, out, row_scale, static_cast<const uint8_t*>(packed), tok, chan, drop_scale, batch, n_tok, channels,
           q_s, q_c, residual, static_cast<int32_t>(groups), norm ? 1 : 0, eps, interleaved ? 1 : 0};
  const int32_t n_pairs = static_cast<int32_t>((groups + 1) / 2);
  // A workgroup's offsets start at its first image: the images its 8 token groups can span.
  if (!x3_fits(n_tok, channels, q_s)) return fail(OW_ERR_UNSUPPORTED, "images too large for 32-bit offsets");
  const int split = x3_split(static_cast<int64_t>(n_pairs) * q_c);
  if (d == 64 && rd == 128) return launch_x3<64, 128>(a, n_pairs, split, stream);
  if (d == 64 && rd == 256) return launch_x3<64, 256>(a, n_pairs, split, stream);
  if (d == 128 && rd == 128) return launch_x3<128, 128>(a, n_pairs, split, stream);
  if (d == 128 && rd == 256) return launch_x3<128, 256>(a, n_pairs, split, stream);
  return fail(OW_ERR_UNSUPPORTED, "unsupported fp32 tile d=%d rd=%d", d, rd);
}

}  // namespace ow
