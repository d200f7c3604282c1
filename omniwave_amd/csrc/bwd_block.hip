// The whole 16-bit backward of a block as one call (ow_bwd_block): the launches of
// omniwave_amd/backward.py's kernels in order, over one workspace.  Host work is what it saves: a
// training step at a small batch was bound by a dozen separate calls and twice as many
// allocations (7x7x1024, one image: 265 us of host time a step for 95 us of kernels).
#include <hip/hip_runtime.h>

#include <cstdint>

#include "ow_common.h"
#include "ow_device.h"

namespace ow {
namespace {

// Parameter gradients from the fp32 buffer to the parameters' dtype.
template <class Ty>
__global__ void __launch_bounds__(256) cast_grads_kernel(const float* src, uint16_t* dst, int64_t n) {
  const int64_t i = (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x) * 4;
  if (i + 4 <= n) {
    const f32x4 v = *reinterpret_cast<const f32x4*>(src + i);
    *reinterpret_cast<u32x2*>(dst + i) = u32x2{Ty::pack2(v[0], v[1]), Ty::pack2(v[2], v[3])};
  } else {
    for (int64_t k = i; k < n; ++k) dst[k] = Ty::from_f32(src[k]);
  }
}

constexpr size_t kPage = size_t(2) << 20;

// Offsets of a backward's buffers in its workspace.
struct BwdPlan {
  int32_t q_s, q_c, d, rd;
  int64_t slots, rows;
  bool fused64, routed;
  size_t packed_bytes;
  int64_t n_part, n_red;
  size_t delta, rscale, small, xt, dyt, wpk, pu, pv, dw, z, du, dv, partial, red, gb, g, dxt, total;
};

// Whether the shape has kernels of its own (d = 64 in pairs of token groups, d = 128; no empty
// batch, whose sums have no rows), and the workspace layout.
bool bwd_plan(const OwPlan* plan, int32_t batch, int32_t rd, int32_t dtype, int32_t flags, bool drop, bool scales,
              BwdPlan& p) {
  if (!plan || batch < 1 || (dtype != OW_DTYPE_BF16 && dtype != OW_DTYPE_F16) || plan->spatial_tile != kG) return false;
  if (ow_plan_dims(plan, &p.q_s, &p.q_c) != OW_OK) return false;
  p.d = plan->channel_tile;
  p.rd = rd;
  p.slots = static_cast<int64_t>(batch) * p.q_s * kG;
  p.rows = static_cast<int64_t>(batch) * plan->height * plan->width;
  p.fused64 = p.d == 64;
  if (p.fused64 ? p.slots % 32 != 0 : p.d != 128) return false;
  p.packed_bytes = ow_bwd_packed_bytes(p.q_c, p.d, rd);
  if (p.packed_bytes == 0) return false;
  // Group q is channels [d q, d q + d): the kernels read x / dy and write g themselves.
  p.routed = plan->channels == p.q_c * p.d && (plan->radix_level == 0 || p.q_c == 1);
  p.n_part = p.fused64 ? ow_bwd_fused_partials(p.slots, p.q_c, rd) : ow_bwd_channel_partials(p.slots, p.q_c);
  p.n_red = p.fused64 ? ow_bwd_param_reduce64_partials(p.slots, p.q_c, rd)
                      : ow_bwd_param_reduce128_partials(p.slots, p.q_c, rd);
  const size_t c = static_cast<size_t>(plan->channels), tile = static_cast<size_t>(p.q_c) * p.slots * p.d * 2,
               wide = static_cast<size_t>(p.q_c) * p.slots * rd * 2, map = static_cast<size_t>(p.rows) * c * 2,
               mat = static_cast<size_t>(p.d) * rd * 4;
  size_t at = 0;
  auto take = [&](size_t bytes) {
    // Large buffers lie at multiples of 2 MiB from the workspace's start (the start itself need not
    // be one): at 56x56x128, B = 128 the step takes 1.6% longer with the three 103 MB operand sets
    // packed end to end.
    const size_t unit = bytes >= kPage ? kPage : 256;
    const size_t o = (at + unit - 1) / unit * unit;
    at = o + bytes;
    return o;
  };
  const bool norm = flags & OW_FUSE_NORM;
  p.delta = take(drop ? map : 0);
  p.rscale = take(norm && !scales ? static_cast<size_t>(p.rows) * 4 : 0);
  p.small = take((2 * c + 768) * 4);
  p.wpk = take(p.packed_bytes);
  p.xt = take(p.routed ? 0 : tile);
  p.dyt = take(p.routed ? 0 : tile);
  p.dxt = take(p.routed ? 0 : tile);
  p.pu = take(tile);
  p.pv = take(tile);
  p.dw = take(tile);
  p.z = take(p.fused64 ? 0 : wide);
  p.du = take(p.fused64 ? 0 : wide);
  p.dv = take(p.fused64 ? 0 : wide);
  p.partial = take(static_cast<size_t>(p.n_part) * 768 * 4);
  p.red = take(static_cast<size_t>(p.n_red) * 3 * mat);
  p.gb = take(3 * static_cast<size_t>(p.q_c) * mat);
  p.g = take(map);
  p.total = (at + 255) / 256 * 256;
  return true;
}

}  // namespace
}  // namespace ow

extern "C" {

size_t ow_bwd_block_workspace(const OwPlan* plan, int32_t batch, int32_t rd, int32_t dtype, int32_t flags, int32_t drop,
                              int32_t scales) {
  ow::BwdPlan p{};
  return ow::bwd_plan(plan, batch, rd, dtype, flags, drop != 0, scales != 0, p) ? p.total : 0;
}

int ow_bwd_block(const void* grad, const void* x, const void* const* small, const int32_t* small_dtype, const void* b_u,
                 const void* b_v, const void* b_o, int32_t weight_dtype, const float* row_scale, const float* drop_scale,
                 const int32_t* token_index, const int32_t* channel_index, const OwPlan* plan, int32_t batch, int32_t rd,
                 int32_t dtype, int32_t flags, float eps, void* dx, float* grads, void* cast, int32_t cast_dtype,
                 void* workspace, size_t workspace_bytes, void* stream) {
  ow::BwdPlan p{};
  OW_CHECK_SUPPORTED(ow::bwd_plan(plan, batch, rd, dtype, flags, drop_scale != nullptr, row_scale != nullptr, p),
                     "no single-call backward for this shape or dtype");
  OW_CHECK_ARG(small && small_dtype && b_u && b_v && b_o && grads && token_index && channel_index,
               "tensor pointer is NULL");
  OW_CHECK_ARG(workspace && workspace_bytes >= p.total && ow::aligned16(workspace),
               "workspace holds %zu bytes; %zu needed (16-byte aligned)", workspace_bytes, p.total);
  OW_CHECK_ARG(!cast || cast_dtype == OW_DTYPE_BF16 || cast_dtype == OW_DTYPE_F16, "cast dtype %d", cast_dtype);
  uint8_t* ws = static_cast<uint8_t*>(workspace);
  auto f = [&](size_t o) { return reinterpret_cast<float*>(ws + o); };
  auto v = [&](size_t o) { return static_cast<void*>(ws + o); };
  const bool norm = flags & OW_FUSE_NORM, residual = flags & OW_FUSE_RESIDUAL;
  const int32_t c = plan->channels, d = p.d, q_c = p.q_c;
  const int64_t slots = p.slots, nb = static_cast<int64_t>(q_c) * d * rd;
#define OW_STEP(call)            \
  do {                           \
    if (int rc_ = (call)) return rc_; \
  } while (0)
  // norm weight (with the norm), gamma, A_u, A_v, A_o in fp32
  const int n_small = norm ? 5 : 4;
  const int64_t counts[5] = {c, c, 256, 256, 256};
  OW_STEP(ow_small_to_f32(small + (norm ? 0 : 1), small_dtype + (norm ? 0 : 1), counts + (norm ? 0 : 1), n_small,
                          f(p.small), stream));
  const float* nw = norm ? f(p.small) : nullptr;
  const float* gm = f(p.small) + (norm ? c : 0);
  const float *au = gm + c, *av = au + 256, *ao = av + 256;
  const void* delta = grad;  // upstream gradient of the delta branch
  if (drop_scale) {
    OW_STEP(ow_scale_samples(grad, drop_scale, v(p.delta), batch,
                             static_cast<int64_t>(plan->height) * plan->width * c, dtype, stream));
    delta = v(p.delta);
  }
  const float* rs = nullptr;
  if (norm) {
    rs = row_scale;
    if (!rs) {
      OW_STEP(ow_rms_scale(x, f(p.rscale), p.rows, c, eps, dtype, stream));
      rs = f(p.rscale);
    }
  }
  if (!p.routed)
    OW_STEP(ow_bwd_gather(x, delta, rs, token_index, channel_index, plan, batch, dtype, v(p.xt), v(p.dyt), stream));
  OW_STEP(ow_pack_bwd_weights(b_u, b_v, b_o, weight_dtype, nw, gm, channel_index, c, q_c, d, rd, dtype, v(p.wpk),
                              stream));
  if (p.fused64) {
    if (p.routed)
      OW_STEP(ow_bwd_fused_routed(x, delta, rs, token_index, plan, batch, au, av, ao, v(p.wpk), p.packed_bytes, v(p.pu),
                                  v(p.pv), v(p.dw), v(p.g), f(p.partial), p.n_part, rd, dtype, stream));
    else
      OW_STEP(ow_bwd_fused(v(p.xt), v(p.dyt), au, av, ao, v(p.wpk), p.packed_bytes, v(p.pu), v(p.pv), v(p.dw), v(p.dxt),
                           f(p.partial), p.n_part, slots, q_c, d, rd, dtype, stream));
  } else if (p.routed) {
    OW_STEP(ow_bwd_channel_routed(x, delta, rs, token_index, plan, batch, au, av, ao, v(p.wpk), p.packed_bytes, v(p.pu),
                                  v(p.pv), v(p.dw), v(p.z), v(p.du), v(p.dv), rd, dtype, stream));
    OW_STEP(ow_bwd_channel2_routed(x, delta, rs, v(p.z), v(p.du), v(p.dv), au, av, v(p.wpk), p.packed_bytes, token_index,
                                   plan, batch, v(p.g), f(p.partial), p.n_part, rd, dtype, stream));
  } else {
    OW_STEP(ow_bwd_channel(v(p.xt), v(p.dyt), au, av, ao, v(p.wpk), p.packed_bytes, v(p.pu), v(p.pv), v(p.dw), v(p.z),
                           v(p.du), v(p.dv), slots, q_c, d, rd, dtype, stream));
    OW_STEP(ow_bwd_channel2(v(p.xt), v(p.dyt), v(p.z), v(p.du), v(p.dv), au, av, v(p.wpk), p.packed_bytes, v(p.dxt),
                            f(p.partial), p.n_part, slots, q_c, d, rd, dtype, stream));
  }
  OW_STEP(ow_sum_rows(f(p.partial), p.n_part, 768, grads, stream));  // dA_u, dA_v, dA_o
  if (p.fused64)
    OW_STEP(ow_bwd_param_reduce64(v(p.pu), v(p.pv), v(p.dw), v(p.wpk), p.packed_bytes, f(p.red), p.n_red, slots, q_c, rd,
                                  dtype, stream));
  else
    OW_STEP(ow_bwd_param_reduce128(v(p.pu), v(p.pv), v(p.dw), v(p.z), v(p.du), v(p.dv), f(p.red), p.n_red, slots, q_c, rd,
                                   dtype, stream));
  OW_STEP(ow_sum_rows(f(p.red), p.n_red / q_c, 3 * nb, f(p.gb), stream));
  if (!p.routed) OW_STEP(ow_bwd_scatter(v(p.dxt), token_index, channel_index, plan, batch, dtype, v(p.g), stream));
  OW_STEP(ow_bwd_rmsnorm(x, v(p.g), rs, grad, dx, p.rows, c, residual ? 1 : 0, dtype, stream));
  float* gb = grads + 768;
  float* gc = gb + 3 * nb;
  OW_STEP(ow_bwd_params(b_u, b_v, b_o, weight_dtype, nw, gm, channel_index, c, q_c, d, rd, f(p.gb), f(p.gb) + nb,
                        f(p.gb) + 2 * nb, gb, gb + nb, gb + 2 * nb, gc, norm ? gc + c : nullptr, stream));
#undef OW_STEP
  if (cast) {
    const int64_t n = 768 + 3 * nb + (norm ? 2 : 1) * c;
    const dim3 grid(static_cast<unsigned>((n + 1023) / 1024));
    hipStream_t s = static_cast<hipStream_t>(stream);
    uint16_t* dst = static_cast<uint16_t*>(cast);
    if (cast_dtype == OW_DTYPE_BF16)
      hipLaunchKernelGGL(ow::cast_grads_kernel<ow::BF16>, grid, dim3(256), 0, s, grads, dst, n);
    else
      hipLaunchKernelGGL(ow::cast_grads_kernel<ow::F16>, grid, dim3(256), 0, s, grads, dst, n);
    if (int rc = ow::hip_status(hipGetLastError(), "cast_grads_kernel launch")) return rc;
  }
  ow::clear_error();
  return OW_OK;
}

}  // extern "C"
