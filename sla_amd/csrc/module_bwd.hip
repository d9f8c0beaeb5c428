// Backward of the whole module (block-sparse attention + linear branch + projection) as one call.
//
// Stands in for autograd through SparseLinearAttention.forward of the reference (sparse_linear_attention/core.py:88-100:
// _attention.backward, kernel.py:277-320, and the autograd graph of calc_linear / proj_l).  It launches the kernels of
// sla_linear_bwd and of sla_sparse_attn_bwd, on `stream`, in this order:
//     linear branch: dq and the sums over the rows | dS, dz, the heads' weight gradients, beside the lists of the map | linear
//     branch: dk, dv | delta, dQ, beside the work items of dK/dV and d_weight, d_bias | dK/dV
// The linear branch comes first and writes dq, dk, dv; the attention kernels, which have arithmetic to do meanwhile, read and
// add.  (The other way round the memory-bound kernels read them: 125 + 108 us for the two at B1 H12 L32760 D128, now 112 + 83.)
// Five launches where there were ten: B2 H4 L4096 D128 forward and backward 215 -> 195 us; the longest calls run against the
// power limit in the attention kernels, whatever the others take (40 heads x 75600: 26.0 ms either way).  More than five: from 40 slices
// of the sequence per head on their sums are added up first; where the general dQ kernel runs (fewer than 320 query blocks of 64
// rows, or 512 of 128), delta and the short jobs have a launch each, and the sums behind the general dK/dV kernel another; states
// that the caller does not have are built before everything else.
// The results equal the two separate calls, the linear one accumulating into the other's gradients, bit for bit.
#include "bwd_steps.h"

namespace sla {

static int module_bwd_run(const void* q, const void* k, const void* v, const int64_t* qkv_strides, const void* o_s,
                          const void* d_out, const int64_t* do_strides, const float* lse, const int8_t* sparse_map,
                          const void* lut, int lut_elem_bytes, const float* weight, const float* bias, const void* states,
                          void* dq, void* dk, void* dv, float* d_weight, float* d_bias, int dtype, int fmap, int B, int H, int L,
                          int D, int BLKQ, int BLKK, int topk, float qk_scale, int flags, void* sparse_workspace,
                          int64_t sparse_workspace_bytes, void* linear_workspace, int64_t linear_workspace_bytes, void* stream) {
  SLA_REQUIRE((flags & ~SLA_BWD_STATES_READY) == 0, SLA_ERR_BAD_ARG, "unknown flag bits in %d", flags);
  SLA_REQUIRE((qkv_strides == nullptr) == (do_strides == nullptr), SLA_ERR_BAD_ARG, "pass both stride arrays or neither");
  ColLists lists;
  HeadSums heads;
  const auto sparse = [&](int steps) {
    return attn_bwd_steps(q, k, v, qkv_strides, o_s, d_out, do_strides, lse, sparse_map, lut, lut_elem_bytes, dq, dk, dv, dtype,
                          B, H, L, D, BLKQ, BLKK, topk, qk_scale, sparse_workspace, sparse_workspace_bytes, stream, steps, &heads,
                          steps ? nullptr : &lists);
  };
  const auto linear = [&](int steps) {
    return linear_bwd_steps(q, k, v, qkv_strides, weight, bias, d_out, do_strides, dq, dk, dv, d_weight, d_bias, dtype, fmap, B,
                            H, L, D, flags, states, linear_workspace, linear_workspace_bytes, stream, steps, &lists,
                            steps ? nullptr : &heads);
  };
  int rc;
  // every argument of both calls is checked before the first kernel of either is launched
  if ((rc = sparse(0))) return rc;
  if ((rc = linear(0))) return rc;
  if ((rc = linear(LB_STATES | LB_QUERY | LB_REDUCE | LB_KEYS))) return rc;
  return sparse(SB_DQ | SB_DKDV | SB_ADD);
}

}  // namespace sla

using namespace sla;

extern "C" int sla_module_bwd(const void* q, const void* k, const void* v, const int64_t* qkv_strides, const void* o_s,
                              const void* d_out, const int64_t* do_strides, const float* lse, const int8_t* sparse_map,
                              const void* lut, int lut_elem_bytes, const float* weight, const float* bias, void* dq, void* dk,
                              void* dv, float* d_weight, float* d_bias, int dtype, int fmap, int B, int H, int L, int D,
                              int BLKQ, int BLKK, int topk, float qk_scale, int flags, void* sparse_workspace,
                              int64_t sparse_workspace_bytes, void* linear_workspace, int64_t linear_workspace_bytes,
                              void* stream, void* side_stream) {
  return module_bwd_run(q, k, v, qkv_strides, o_s, d_out, do_strides, lse, sparse_map, lut, lut_elem_bytes, weight, bias, nullptr,
                        dq, dk, dv, d_weight, d_bias, dtype, fmap, B, H, L, D, BLKQ, BLKK, topk, qk_scale, flags,
                        sparse_workspace, sparse_workspace_bytes, linear_workspace, linear_workspace_bytes, stream);
}

extern "C" int sla_module_bwd_states(const void* q, const void* k, const void* v, const int64_t* qkv_strides, const void* o_s,
                                     const void* d_out, const int64_t* do_strides, const float* lse, const int8_t* sparse_map,
                                     const void* lut, int lut_elem_bytes, const float* weight, const float* bias,
                                     const void* states, void* dq, void* dk, void* dv, float* d_weight, float* d_bias, int dtype,
                                     int fmap, int B, int H, int L, int D, int BLKQ, int BLKK, int topk, float qk_scale,
                                     void* sparse_workspace, int64_t sparse_workspace_bytes, void* linear_workspace,
                                     int64_t linear_workspace_bytes, void* stream, void* side_stream) {
  SLA_REQUIRE(states, SLA_ERR_BAD_ARG, "null states");
  return module_bwd_run(q, k, v, qkv_strides, o_s, d_out, do_strides, lse, sparse_map, lut, lut_elem_bytes, weight, bias, states,
                        dq, dk, dv, d_weight, d_bias, dtype, fmap, B, H, L, D, BLKQ, BLKK, topk, qk_scale, 0,
                        sparse_workspace, sparse_workspace_bytes, linear_workspace, linear_workspace_bytes, stream);
}
