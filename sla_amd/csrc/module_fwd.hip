// Forward of the whole module (mask builder, linear branch's states, attention with the linear branch in its epilogue) as
// one call.
//
// Stands in for SparseLinearAttention.forward of the reference (sparse_linear_attention/core.py:69-105).  On `stream`:
//     [16-bit copies of fp32 inputs] | mask builder | attention
// with the state build (k, v only) on the caller's second stream beside the mask builder where that pays.
#include "fwd_steps.h"
#include "side_events.h"

namespace sla {

// 16-bit copies of three fp32 tensors of n elements each, one after the other in `dst` (n a multiple of 8).
template <typename Tag>
__global__ __launch_bounds__(256) void cast3_kernel(const float* __restrict__ a, const float* __restrict__ b,
                                                    const float* __restrict__ c, uint16_t* __restrict__ dst, int64_t n) {
  const float* src = blockIdx.y == 0 ? a : blockIdx.y == 1 ? b : c;
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 8;
  if (i >= n) return;
  const f32x4_t x = *reinterpret_cast<const f32x4_t*>(src + i), y = *reinterpret_cast<const f32x4_t*>(src + i + 4);
  i32x4_t w;
  w[0] = (int)Elem<Tag>::pack2(x[0], x[1]);
  w[1] = (int)Elem<Tag>::pack2(x[2], x[3]);
  w[2] = (int)Elem<Tag>::pack2(y[0], y[1]);
  w[3] = (int)Elem<Tag>::pack2(y[2], y[3]);
  *reinterpret_cast<i32x4_t*>(dst + (int64_t)blockIdx.y * n + i) = w;
}

int64_t module_fwd_workspace_bytes(int in_dtype, int BH, int L, int D, int BLKQ, int BLKK) {
  return align_up(block_map_workspace_bytes(in_dtype, BH, L, D, BLKQ, BLKK), 256) + linear_parts_bytes(BH, L, D);
}

}  // namespace sla

using namespace sla;

extern "C" int sla_module_fwd(const void* q, const void* k, const void* v, const int64_t* qkv_strides, int in_dtype, void* cast,
                              const float* weight, const float* bias, void* out, const int64_t* out_strides, void* o_s,
                              float* lse, int8_t* sparse_map, void* lut, int lut_elem_bytes, void* states, int dtype, int fmap,
                              int B, int H, int L, int D, int BLKQ, int BLKK, int topk, float qk_scale, void* workspace,
                              int64_t workspace_bytes, void* stream, void* side_stream) {
  int rc = validate_attn_shape(dtype, B, H, L, D, BLKQ, BLKK, topk, lut_elem_bytes);
  if (rc) return rc;
  if ((rc = validate_linear(dtype, fmap, B, H, L, D))) return rc;
  SLA_REQUIRE(in_dtype == dtype || in_dtype == SLA_F32 || in_dtype == SLA_MASK_GIVEN, SLA_ERR_BAD_ARG,
              "in_dtype %d is neither fp32 nor the compute dtype", in_dtype);
  const bool casts = in_dtype == SLA_F32, mask_given = in_dtype == SLA_MASK_GIVEN;
  if (mask_given) in_dtype = dtype;
  SLA_REQUIRE(q && k && v && weight && bias && out && lse && (lut || topk == 0) && states && workspace && (cast || !casts),
              SLA_ERR_BAD_ARG, "null pointer");
  SLA_REQUIRE(((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)cast | (uintptr_t)weight | (uintptr_t)out | (uintptr_t)o_s |
               (uintptr_t)lut | (uintptr_t)states | (uintptr_t)workspace) % 16 == 0,
              SLA_ERR_BAD_ARG, "pointers must be 16-byte aligned");
  SLA_REQUIRE(!casts || !qkv_strides, SLA_ERR_BAD_ARG, "fp32 inputs are contiguous");
  const int BH = B * H;
  const int64_t need = module_fwd_workspace_bytes(in_dtype, BH, L, D, BLKQ, BLKK);
  SLA_REQUIRE(workspace_bytes >= need, SLA_ERR_WORKSPACE, "workspace of %lld bytes, need %lld", (long long)workspace_bytes,
              (long long)need);
  RowLayout lin, lout;
  if ((rc = make_layout(qkv_strides, B, H, L, D, 2, &lin))) return rc;
  if ((rc = make_layout(out_strides, B, H, L, D, 2, &lout))) return rc;
  hipStream_t st = (hipStream_t)stream, side = (hipStream_t)side_stream;
  char* const map_part = (char*)workspace;
  const int64_t map_bytes = align_up(block_map_workspace_bytes(in_dtype, BH, L, D, BLKQ, BLKK), 256);
  char* const parts = map_part + map_bytes;
  if (!mask_given) {                   // (the mask builder's own checks too, before the first launch)
    RowLayout unused;
    rc = block_map_check(q, k, qkv_strides, in_dtype, B, H, L, D, BLKQ, BLKK, topk, map_part, map_bytes, sparse_map,
                         sparse_map != nullptr, lut, lut_elem_bytes, &unused);
    if (rc) return rc;
  }

  const void *qc = q, *kc = k, *vc = v;
  if (casts) {
    const int64_t n = (int64_t)BH * L * D;
    const dim3 grid((unsigned)((n / 8 + 255) / 256), 3);
    if (dtype == SLA_BF16)
      hipLaunchKernelGGL((cast3_kernel<bf16_tag>), grid, dim3(256), 0, st, (const float*)q, (const float*)k, (const float*)v,
                         (uint16_t*)cast, n);
    else
      hipLaunchKernelGGL((cast3_kernel<f16_tag>), grid, dim3(256), 0, st, (const float*)q, (const float*)k, (const float*)v,
                         (uint16_t*)cast, n);
    qc = cast;
    kc = (uint16_t*)cast + n;
    vc = (uint16_t*)cast + 2 * n;
  }
  const auto state = [&](hipStream_t s) {
    return linear_state_run(kc, vc, lin, weight, dtype, fmap, BH, L, D, (char*)states, parts, s);
  };
  const auto mask = [&]() -> int {
    if (mask_given) return SLA_OK;
    return block_map_entry(q, k, qkv_strides, in_dtype, B, H, L, D, BLKQ, BLKK, topk, map_part, map_bytes, sparse_map,
                           sparse_map != nullptr, lut, lut_elem_bytes, st);
  };
  const auto attention = [&]() {
    return attn_linear_run(qc, kc, vc, lin, lut, lut_elem_bytes, (const char*)states, bias, o_s, out, lout, lse, dtype, fmap, BH,
                           L, D, BLKQ, topk, qk_scale, st);
  };
  if (!side || side == st || !side_stream_pays(B, H, L, D, topk)) {
    if ((rc = state(st))) return rc;
    if ((rc = mask())) return rc;
    return attention();
  }
  std::lock_guard<std::mutex> lock(side_events_mutex());
  SideEvents* ev;
  if ((rc = side_events_for_current_device(&ev))) return rc;
  SLA_HIP_OK(hipEventRecord(ev->fork, st));
  SLA_HIP_OK(hipStreamWaitEvent(side, ev->fork, 0));
  // (once the second stream waits on `stream`, no path leaves without `stream` waiting for it in turn)
  rc = state(side);
  const int rc_mask = mask();
  SLA_HIP_OK(hipEventRecord(ev->first, side));
  SLA_HIP_OK(hipStreamWaitEvent(st, ev->first, 0));
  if (rc) return rc;
  if (rc_mask) return rc_mask;
  return attention();
}
