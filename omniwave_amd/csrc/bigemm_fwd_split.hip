// BiGEMM forward for d = 128, rd = 256 at small sizes: one workgroup per 32-token pair and
// channel group, the expanded dimension split over its waves.
//
// Same math, operand packing and order of every sum as the persistent kernel
// (bigemm_fwd_persist.hip), whose results it reproduces bit for bit.  That kernel walks a unit of
// eight pairs through the eight 32-row chunks of the expanded dimension one after the other:
// 30000 cycles however few units there are, on as many CUs as there are units.  Here the four
// waves of a workgroup share one pair:
//   * wave w loads rows 8 w .. + 7 of the pair (whole rows where their RMSNorm sums or the
//     interleaved columns of strided groups need them) into the tile in LDS;
//   * each wave forms P for the whole pair, then U', V' and the gate Z of chunks w and w + 4,
//     their weights read straight into registers while the rows are on their way;
//   * Z (16 KB) goes through LDS, and wave w accumulates channel block w of W = Z B_o over all
//     chunks in order: the 32x32 blocks of W are independent, so no partial sums are added;
//   * block w of delta^T, staged through LDS, leaves as 16-byte pieces of the rows the wave
//     loaded (2-byte elements for strided groups).
// Bound by the latency of its loads and by the chain rows -> P -> Z -> W: at 7x7x1024 radix 1, B = 8
// waves wait for memory or LDS 47% of their time and the matrix cores are busy 2%.  Every instance
// uses all 256 registers of two waves per SIMD and spills four more (20 bytes of scratch a lane).
#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "ow_device.h"

namespace ow {
namespace {

constexpr int kD = 128;
constexpr int kRD = 256;
constexpr int kKS = kD / 16;
constexpr int kMB = kD / 32;
constexpr int kNCH = kRD / 32;
constexpr int kWaves = 4;
constexpr int kThreads = 64 * kWaves;
constexpr int kFrU = kKS;                 // B_u'^T fragments per chunk (B_v'^T the same), then 2 kMB of B_o
constexpr int kFrCh = 2 * kFrU + 2 * kMB;
constexpr int kLdo = kD + 8;              // output staging row stride (elements)
static_assert(kMB == kWaves && kNCH == 2 * kWaves, "a channel block and two chunks per wave");

struct SplitLds {
  uint16_t x[32 * kD];       // the pair's rows of this group, 16-byte piece p of row r at slot p ^ tile128_swz(r)
  u32x4 z[kNCH][2][64];      // the gate, chunk by chunk, as A operands of the W products
  uint16_t st[32 * kLdo];    // delta rows
  float rsc[32];
};

// NS: 1 for contiguous channel groups, else the channel stride of the strided groups (= q_c).
template <class Ty, int NS>
__global__ void __launch_bounds__(kThreads, 2) bigemm_fwd_split_kernel(PersistArgs a) {
  __shared__ __attribute__((aligned(16))) SplitLds sh;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int hh = lane >> 5, l32 = lane & 31, l16 = lane & 15;
  // The workgroups of an XCD (block b runs on XCD b % 8) see few groups when q_c divides 8, so its
  // L2 holds their weights.
  const int qc = static_cast<int>(blockIdx.x % static_cast<unsigned>(a.q_c));
  const uint32_t pair = blockIdx.x / static_cast<unsigned>(a.q_c);
  // This wave's rows 8 wave + 4 p + lane / 16 belong to one token group.
  const uint32_t n_groups = static_cast<uint32_t>(a.batch) * static_cast<uint32_t>(a.q_s);
  const uint32_t tg = 2 * pair + (wave >> 1);
  const int32_t img = static_cast<int32_t>(tg / static_cast<uint32_t>(a.q_s));
  const int32_t sg = static_cast<int32_t>(tg - static_cast<uint32_t>(img) * static_cast<uint32_t>(a.q_s));
  const bool real = tg < n_groups;

  int32_t tk[2], to[2];
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    const int ti = sg * kG + 8 * (wave & 1) + 4 * p + (lane >> 4);
    tk[p] = a.tok[ti];
    to[p] = a.out_tok ? a.out_tok[ti] : tk[p];
  }
  const float dsc = a.drop_scale ? a.drop_scale[real ? img : 0] : 1.0f;
  const int res = NS > 1 ? (a.chan[qc * kD] & (NS - 1)) : 0;

  // Weights: chunks w and w + 4 of B_u', B_v' now, the wave's blocks of B_o later.
  const u32x4* head = reinterpret_cast<const u32x4*>(a.packed);
  const u32x4 fAu = head[lane], fAv = head[64 + lane], fAo = head[128 + lane];
  const __amdgpu_buffer_rsrc_t rw =
      buffer_rsrc(a.packed + kHeadElems + static_cast<size_t>(qc) * kNCH * kFrCh * kFragElems, kNCH * kFrCh * 1024);
  auto frag = [&](int ec, int f) -> u32x4 {
    return __builtin_amdgcn_raw_buffer_load_b128(rw, 16 * lane, (ec * kFrCh + f) * 1024, 0);
  };
  u32x4 wf[2][2 * kFrU];
#pragma unroll
  for (int f = 0; f < 2 * kFrU; ++f) wf[0][f] = frag(wave, f);
  __builtin_amdgcn_sched_barrier(0);

  // The pair's rows.
  const uint32_t xbytes = static_cast<uint32_t>(static_cast<int64_t>(a.batch) * a.n_tok * a.channels * 2);
  const __amdgpu_buffer_rsrc_t rx = buffer_rsrc(a.x, xbytes);
  int32_t id[2], od[2];
  uint32_t off[2];
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    const bool ok = real & (tk[p] >= 0) & (tk[p] < a.n_tok);
    id[p] = ok ? img * a.n_tok + tk[p] : -1;
    od[p] = (ok & (to[p] >= 0) & (to[p] < a.n_tok)) ? img * a.n_tok + to[p] : -1;
    off[p] = ok ? static_cast<uint32_t>(id[p]) * static_cast<uint32_t>(a.channels * 2) + 16u * l16 : kOffOut;
  }
  float acc[2] = {0.0f, 0.0f};
  auto row_of = [&](int p) { return 8 * wave + 4 * p + (lane >> 4); };
  if constexpr (NS == 1) {
    u32x4 own[2];
#pragma unroll
    for (int p = 0; p < 2; ++p) own[p] = __builtin_amdgcn_raw_buffer_load_b128(rx, off[p] + 256u * qc, 0, 0);
    if (a.norm == kNormInline) {  // q_c <= 8: every piece of the rows, in the statistics pass's order
      u32x4 v[2][8];
#pragma unroll
      for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int j = 0; j < 8; ++j)
          v[p][j] = __builtin_amdgcn_raw_buffer_load_b128(rx, j < a.q_c ? off[p] + 256u * j : kOffOut, 0, 0);
#pragma unroll
      for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int j = 0; j < 8; ++j)
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[p] = Ty::dot2sq(v[p][j][e], acc[p]);
    }
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      const int r = row_of(p);
      *reinterpret_cast<u32x4*>(&sh.x[r * kD + ((l16 ^ tile128_swz(r)) * 8)]) = own[p];
    }
  } else {
    constexpr int M = 8 / NS;
    u32x4 v[2][NS];
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
      for (int j = 0; j < NS; ++j) v[p][j] = __builtin_amdgcn_raw_buffer_load_b128(rx, off[p] + 256u * j, 0, 0);
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      const int r = row_of(p);
#pragma unroll
      for (int j = 0; j < NS; ++j) {
        const StridedPack<M> e = strided_pack<M>(v[p][j], res);
        uint16_t* dst = &sh.x[r * kD + ((M * (l16 + 16 * j)) ^ (8 * tile128_swz(r)))];
        if constexpr (M == 1)
          *dst = static_cast<uint16_t>(e);
        else
          *reinterpret_cast<StridedPack<M>*>(dst) = e;
#pragma unroll
        for (int k = 0; k < 4; ++k) acc[p] = Ty::dot2sq(v[p][j][k], acc[p]);
      }
    }
  }
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    const float sum = group_sum<16>(acc[p]);  // all lanes take part; lane 15 of a row has the total
    if (l16 == 15) {
      float s = 1.0f;
      if (id[p] >= 0) {
        if (a.norm == kNormInline) {
          s = rms_scale<Ty>(sum / static_cast<float>(a.channels), a.eps);
          if (a.rs_out && qc == 0) a.rs_out[id[p]] = s;
        } else if (a.norm == kNormBuffer) {
          s = a.row_scale[id[p]];
        } else if (a.norm == kNormPartials) {
          float t = 0.0f;
          for (int q = 0; q < a.parts; ++q) t += a.row_scale[static_cast<int64_t>(id[p]) * a.parts + q];
          s = rms_scale<Ty>(t / static_cast<float>(a.channels), a.eps);
        }
      }
      sh.rsc[row_of(p)] = s;
    }
  }
#pragma unroll
  for (int f = 0; f < kFrU; ++f) wf[1][f] = frag(wave + kWaves, f);
  __syncthreads();

  // Token side of the pair (every wave the whole pair).
  u32x4 Pu[kKS], Pv[kKS];
  {
    u32x4 xk[kKS / 2][2];
    const uint32_t xb = lds_addr(sh.x);
    pair_xt_tr<kKS>([&](int r, int c) { return xb + 2u * static_cast<uint32_t>(r * kD + (c ^ (8 * tile128_swz(r)))); },
                    lane, xk);
    u32x4 bu = fAu, bv = fAv;
    if (a.norm != kNormNone) {
      const float* r8 = &sh.rsc[16 * ((lane >> 4) & 1) + 4 * hh];
      bu = scale8<Ty>(fAu, r8);
      bv = scale8<Ty>(fAv, r8);
    }
    pair_token_side_mma<Ty, kKS>(xk, bu, bv, lane, Pu, Pv);
  }
#pragma unroll
  for (int f = kFrU; f < 2 * kFrU; ++f) wf[1][f] = frag(wave + kWaves, f);

  u32x4 bo[kNCH][2];
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    f32x16 U = {}, V = {};
#pragma unroll
    for (int i = 0; i < kKS; ++i) {
      U = Ty::mma32(wf[c][i], Pu[i], U);
      V = Ty::mma32(wf[c][kFrU + i], Pv[i], V);
    }
    // Half the B_o fragments at a time, in the registers of a chunk's weights.
#pragma unroll
    for (int ec = 0; ec < kNCH / 2; ++ec)
#pragma unroll
      for (int j = 0; j < 2; ++j) bo[4 * c + ec][j] = frag(4 * c + ec, 2 * kFrU + 2 * wave + j);
    u32x4 Z[2];
#pragma unroll
    for (int k = 0; k < 16; k += 2)
      Z[k / 8][(k % 8) / 2] = Ty::pack2(silu_gate(U[k], V[k]), silu_gate(U[k + 1], V[k + 1]));
#pragma unroll
    for (int j = 0; j < 2; ++j) sh.z[wave + kWaves * c][j][lane] = Z[j];
  }
  __syncthreads();

  // W = Z B_o for channel block `wave`, then its delta^T: lane l32 = token row.
  f32x16 W[1] = {f32x16{}};
#pragma unroll
  for (int ec = 0; ec < kNCH; ++ec)
#pragma unroll
    for (int j = 0; j < 2; ++j) W[0] = Ty::mma32(sh.z[ec][j][lane], bo[ec][j], W[0]);
  mfma_drain();
  f32x16 dl[1];
  pair_output_t<Ty, 1>(W, fAo, lane, dl);
  mfma_drain();
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    *reinterpret_cast<u32x2*>(&sh.st[l32 * kLdo + 32 * wave + 8 * q + 4 * hh]) =
        u32x2{Ty::pack2(dl[0][4 * q], dl[0][4 * q + 1]), Ty::pack2(dl[0][4 * q + 2], dl[0][4 * q + 3])};
  }
  __syncthreads();

  // This wave's rows to memory.
  const __amdgpu_buffer_rsrc_t ro = buffer_rsrc(a.out, xbytes);
  u32x4 val[2];
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    const int r = row_of(p);
    val[p] = *reinterpret_cast<const u32x4*>(&sh.st[r * kLdo + 8 * l16]);
    if (a.drop_scale) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        val[p][e] = Ty::pack2(Ty::to_f32(lo16(val[p][e])) * dsc, Ty::to_f32(hi16(val[p][e])) * dsc);
    }
    if (a.residual) {
      const u32x4 x = *reinterpret_cast<const u32x4*>(&sh.x[r * kD + ((l16 ^ tile128_swz(r)) * 8)]);
#pragma unroll
      for (int e = 0; e < 4; ++e) val[p][e] = add_residual2<Ty>(x[e], val[p][e]);
    }
    if (a.stats_out) {
      float t = 0.0f;
#pragma unroll
      for (int e = 0; e < 4; ++e) t = Ty::dot2sq(val[p][e], t);
      t = group_sum<16>(t);
      if (l16 == 15 && od[p] >= 0) a.stats_out[static_cast<int64_t>(od[p]) * a.q_c + qc] = t;
    }
    if constexpr (NS == 1) {
      const uint32_t oo =
          od[p] >= 0 ? static_cast<uint32_t>(od[p]) * static_cast<uint32_t>(a.channels * 2) + 256u * qc + 16u * l16 : kOffOut;
      __builtin_amdgcn_raw_buffer_store_b128(val[p], ro, oo, 0, 0);
    } else {
      *reinterpret_cast<u32x4*>(&sh.st[r * kLdo + 8 * l16]) = val[p];
    }
  }
  if constexpr (NS > 1) {
    // Tile column t is channel res + t NS: lane l stores column 64 h + l of one row per instruction.
    wave_lds_sync();
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int32_t row = __builtin_amdgcn_readlane(od[k >> 2], 16 * (k & 3));
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int t = 64 * h + lane;
        const uint32_t ob = row >= 0 ? static_cast<uint32_t>(row) * static_cast<uint32_t>(a.channels * 2) +
                                           2u * static_cast<uint32_t>(res + t * NS)
                                     : kOffOut;
        __builtin_amdgcn_raw_buffer_store_b16(sh.st[(8 * wave + k) * kLdo + t], ro, ob, 0, 0);
      }
    }
  }
}

template <class Ty>
void launch_stride(const PersistArgs& a, dim3 g, hipStream_t stream) {
  switch (a.stride) {
    case 2: hipLaunchKernelGGL((bigemm_fwd_split_kernel<Ty, 2>), g, dim3(kThreads), 0, stream, a); break;
    case 4: hipLaunchKernelGGL((bigemm_fwd_split_kernel<Ty, 4>), g, dim3(kThreads), 0, stream, a); break;
    case 8: hipLaunchKernelGGL((bigemm_fwd_split_kernel<Ty, 8>), g, dim3(kThreads), 0, stream, a); break;
    default: hipLaunchKernelGGL((bigemm_fwd_split_kernel<Ty, 1>), g, dim3(kThreads), 0, stream, a); break;
  }
}

}  // namespace

// Up to two and a half pairs x groups per CU (640 on 256 CUs): two workgroups fit on a CU, and the
// second round of a larger launch takes as long as the persistent kernel (block, us, split against persistent, the latter with
// its statistics pass: 14x14x512 local B = 1: 7.0 / 17.0, B = 16 (416): 10.7 / 18.1, B = 20 (520):
// 14.5 / 18.2, B = 32 (832): 18.9 / 18.9; 7x7x1024 radix 1 B = 8 (128): 9.4 / 25.6, B = 32 (512):
// 17.8 / 25.8, B = 64 (1024): 31.2 / 27.2).
bool split_supported(int64_t n_groups, int32_t q_c) {
  return 2 * ((n_groups + 1) / 2 * q_c) <= 5 * static_cast<int64_t>(device_cus());
}

int launch_fwd_split(const PersistArgs& a, int32_t dtype, hipStream_t stream) {
  const int64_t blocks = (static_cast<int64_t>(a.batch) * a.q_s + 1) / 2 * a.q_c;
  if (blocks == 0) return OW_OK;
  if (blocks > 0x7fffffff) return fail(OW_ERR_UNSUPPORTED, "grid too large (%lld workgroups)", (long long)blocks);
  if (a.fp8) return fail(OW_ERR_UNSUPPORTED, "the split forward has no fp8 channel side");
  if (a.norm == kNormInline && a.stride == 1 && a.q_c > 8)
    return fail(OW_ERR_INVALID, "the split forward forms row scales of at most 1024 channels");
  if (a.stride != 1 && (a.stride != a.q_c || (a.stride != 2 && a.stride != 4 && a.stride != 8)))
    return fail(OW_ERR_UNSUPPORTED, "split forward: channel stride %d", a.stride);
  const dim3 g(static_cast<unsigned>(blocks));
  if (dtype == OW_DTYPE_BF16)
    launch_stride<BF16>(a, g, stream);
  else if (dtype == OW_DTYPE_F16)
    launch_stride<F16>(a, g, stream);
  else
    return fail(OW_ERR_UNSUPPORTED, "unsupported dtype %d", dtype);
  return hip_status(hipGetLastError(), "bigemm_fwd_split_kernel launch");
}

}  // namespace ow
