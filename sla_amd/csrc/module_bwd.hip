// Backward of the whole module (block-sparse attention + linear branch + projection) as one call.
//
// Stands in for autograd through SparseLinearAttention.forward of the reference (sparse_linear_attention/core.py:88-100:
// _attention.backward, kernel.py:277-320, and the autograd graph of calc_linear / proj_l).  It launches the kernels of
// sla_sparse_attn_bwd and sla_linear_bwd (with SLA_BWD_ACCUMULATE: the linear branch adds into dq, dk, dv), in this order
// on `stream`:
//     delta, dQ | linear branch: dq and the sums over the rows | dK/dV | linear branch: dk, dv
// and, when the caller passes a second stream, the short kernels on it beside the long ones:
//     the per-key-block lists of the map (needed by dK/dV only)            beside delta and dQ
//     dS, dz, d_weight, d_bias from the sums (needed by dk, dv of the linear branch)   beside dK/dV
// `stream` waits for everything put on `side_stream` before the call returns, so the caller orders later work by
// `stream` alone.  The results equal the two separate calls bit for bit.
#include "bwd_steps.h"
#include "side_events.h"

namespace sla {

static int module_bwd_run(const void* q, const void* k, const void* v, const int64_t* qkv_strides, const void* o_s,
                          const void* d_out, const int64_t* do_strides, const float* lse, const int8_t* sparse_map,
                          const void* lut, int lut_elem_bytes, const float* weight, const float* bias, const void* states,
                          void* dq, void* dk, void* dv, float* d_weight, float* d_bias, int dtype, int fmap, int B, int H, int L,
                          int D, int BLKQ, int BLKK, int topk, float qk_scale, int flags, void* sparse_workspace,
                          int64_t sparse_workspace_bytes, void* linear_workspace, int64_t linear_workspace_bytes, void* stream,
                          void* side_stream) {
  SLA_REQUIRE((flags & ~SLA_BWD_STATES_READY) == 0, SLA_ERR_BAD_ARG, "unknown flag bits in %d", flags);
  SLA_REQUIRE((qkv_strides == nullptr) == (do_strides == nullptr), SLA_ERR_BAD_ARG, "pass both stride arrays or neither");
  const int lflags = flags | SLA_BWD_ACCUMULATE;
  hipStream_t st = (hipStream_t)stream, side = (hipStream_t)side_stream;
  const auto sparse = [&](hipStream_t s, int steps) {
    return attn_bwd_steps(q, k, v, qkv_strides, o_s, d_out, do_strides, lse, sparse_map, lut, lut_elem_bytes, dq, dk, dv, dtype,
                          B, H, L, D, BLKQ, BLKK, topk, qk_scale, sparse_workspace, sparse_workspace_bytes, s, steps);
  };
  const auto linear = [&](hipStream_t s, int steps) {
    return linear_bwd_steps(q, k, v, qkv_strides, weight, bias, d_out, do_strides, dq, dk, dv, d_weight, d_bias, dtype, fmap, B,
                            H, L, D, lflags, states, linear_workspace, linear_workspace_bytes, s, steps);
  };
  int rc;
  // every argument of both calls is checked before the first kernel of either is launched
  if ((rc = sparse(st, 0))) return rc;
  if ((rc = linear(st, 0))) return rc;
  if (!side || side == st || !side_stream_pays(B, H, L, D, topk)) {
    // one stream: the same order, the short kernels in between
    if ((rc = sparse(st, SB_ALL))) return rc;
    return linear(st, LB_ALL);
  }
  std::lock_guard<std::mutex> lock(side_events_mutex());
  SideEvents* ev;
  if ((rc = side_events_for_current_device(&ev))) return rc;
  // Once the second stream has been made to wait on `stream`, no path leaves this call without `stream` waiting for
  // the second one in turn: the caller orders later work (and the reuse of the workspaces) by `stream` alone, and a
  // capture in progress must not be left forked.
  const auto forked = [&]() -> int {
    int r;
    // side: lists of the map.  main: delta, dQ, then the query side of the linear branch
    if ((r = sparse(side, SB_LISTS))) return r;
    SLA_HIP_OK(hipEventRecord(ev->first, side));
    if ((r = sparse(st, SB_DQ))) return r;
    if ((r = linear(st, LB_STATES | LB_QUERY))) return r;
    SLA_HIP_OK(hipEventRecord(ev->second, st));
    // side: the small products of the linear branch.  main: dK/dV, then the key side of the linear branch
    SLA_HIP_OK(hipStreamWaitEvent(side, ev->second, 0));
    if ((r = linear(side, LB_REDUCE | LB_BESIDE))) return r;
    SLA_HIP_OK(hipEventRecord(ev->third, side));
    SLA_HIP_OK(hipStreamWaitEvent(st, ev->first, 0));
    if ((r = sparse(st, SB_DKDV))) return r;
    SLA_HIP_OK(hipStreamWaitEvent(st, ev->third, 0));
    return linear(st, LB_KEYS);
  };
  SLA_HIP_OK(hipEventRecord(ev->fork, st));
  SLA_HIP_OK(hipStreamWaitEvent(side, ev->fork, 0));
  rc = forked();
  if (rc) {
    // join whatever the second stream was given before the failure (its last event may never have been recorded)
    if (hipEventRecord(ev->third, side) == hipSuccess) (void)hipStreamWaitEvent(st, ev->third, 0);
  }
  return rc;
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
                        sparse_workspace, sparse_workspace_bytes, linear_workspace, linear_workspace_bytes, stream, side_stream);
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
                        sparse_workspace, sparse_workspace_bytes, linear_workspace, linear_workspace_bytes, stream, side_stream);
}
