// Backward of the linear-attention branch + projection for gfx950.
//
// Stands in for torch autograd through sparse_linear_attention/core.py:90-99 of the reference.
// With a = phi(q), c = phi(k), S = c^T v, z = sum c, n = a S, den = 1e-5 + a.z, y = n/den,
// out = y W^T + b and G = d(out):
//   db = sum G ; dW = G^T y ; dy = G W ; dn = dy/den ; dden = -sum_d(dy*y)/den
//   da = dn S^T + dden z ; dS = a^T dn ; dz = sum_l dden a
//   dc = v dS^T + dz ; dv = c dS ; dq = phi'(q) da ; dk = phi'(k) dc
//
// Kernels (linear_bwd_stream.h, linear_state.h):
//   state build (shared with the forward) : S and z again from k, v
//   stream : q and G once: dq, and per slice of the sequence the partial sums M^T, dz, db
//   presum : many slices of few heads added up first
//   finish : those sums added up -> dS (16 bit, both orientations), dz, per-head dW, db
//   heads  : the heads' dW and db added up
//   keys   : k and v once: dk, dv (a whole module's backward with few key blocks: in the attention's dK/dV kernel instead)
// The complement-mode branch forms dW and db from row-wise temporaries, with the state kernel and the reduction below.
#include "bwd_steps.h"
#include "linear_bwd_stream.h"

namespace sla {

// ---- weight gradients apart ------------------------------------------------------------------
// grid (cdiv(D*D,256), BH): a head's dW^T, db from its slices' partial sums, in ascending order.
__global__ __launch_bounds__(256) void linear_bwd_reduce_kernel(const float* __restrict__ dw_part, const float* __restrict__ db_part,
                                                                float* __restrict__ dw_head, float* __restrict__ db_head,
                                                                int nsplit, int D) {
  const int DD = D * D;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int bh = blockIdx.y;
  if (i < DD) {
    const float* p = dw_part + (size_t)bh * nsplit * DD + i;
    float s = 0.f;
#pragma unroll 16
    for (int sp = 0; sp < nsplit; ++sp) s += p[(size_t)sp * DD];
    dw_head[(size_t)bh * DD + i] = s;
  }
  if (i < D) {
    const float* p = db_part + (size_t)bh * nsplit * D + i;
    float s = 0.f;
#pragma unroll 16
    for (int sp = 0; sp < nsplit; ++sp) s += p[(size_t)sp * D];
    db_head[(size_t)bh * D + i] = s;
  }
}

// ---- host ---------------------------------------------------------------------------------
struct LinBwdWs {
  LinWs fwd;
  LinSplit sp;   // slices of the stream and keys kernels (128 rows per step)
  size_t m_part, dz_part, db_part, ds, dst, dz, dw_head, db_head, total;
};
// (own_states = false: the forward's states lie elsewhere, the workspace holds none)
static LinBwdWs lin_bwd_ws(int BH, int L, int D, bool own_states) {
  LinBwdWs w;
  w.fwd = lin_ws(BH, L, D);
  w.sp = lin_split(BH, L, D == 128 ? 256 : 512, LBS_TR);       // (one workgroup per compute unit at head dim 128, two at 64)
  const int64_t np = (int64_t)BH * w.sp.nsplit;
  size_t off = own_states ? w.fwd.total : 0;
  w.m_part = off;  off += align_up(np * D * D * 4, 256);
  w.dz_part = off; off += align_up(np * D * 4, 256);
  w.db_part = off; off += align_up(np * D * 4, 256);
  w.ds = off;      off += align_up((int64_t)BH * D * D * 2, 256);
  w.dst = off;     off += align_up((int64_t)BH * D * D * 2, 256);
  w.dz = off;      off += align_up((int64_t)BH * D * 4, 256);
  w.dw_head = off; off += align_up((int64_t)BH * D * D * 4, 256);
  w.db_head = off; off += align_up((int64_t)BH * D * 4, 256);
  w.total = off;
  return w;
}
int64_t linear_bwd_workspace_bytes(int BH, int L, int D) { return (int64_t)lin_bwd_ws(BH, L, D, true).total; }
int64_t linear_bwd_states_apart_bytes(int BH, int L, int D) { return (int64_t)lin_bwd_ws(BH, L, D, false).total; }

template <typename Tag, int D>
static int linear_bwd_impl(const void* q, const void* k, const void* v, const float* weight, const void* d_out, void* dq,
                           void* dk, void* dv, const RowLayout& lin, const RowLayout& ldo, float* d_weight, float* d_bias,
                           int fmap, int BH, int L, int flags, const char* states, char* ws, hipStream_t st, int steps,
                           const ColLists& lists, HeadSums* heads, LinearKeys* keys) {
  const LinBwdWs w = lin_bwd_ws(BH, L, D, !states);
  const HeadSums hs = {(const float*)(ws + w.dw_head), (const float*)(ws + w.db_head), d_weight, d_bias, BH, D, D * D / 256};
  if (heads) *heads = hs;
  if (keys) *keys = LinearKeys{(const uint16_t*)(ws + w.ds), (const uint16_t*)(ws + w.dst), (const float*)(ws + w.dz), fmap};
  if (steps == 0) return SLA_OK;        // (arguments checked, nothing asked for)
  const int accumulate = flags & SLA_BWD_ACCUMULATE;
  if ((steps & LB_STATES) && !states && !(flags & SLA_BWD_STATES_READY)) {
    // everything the forward's state build leaves: transposed state, z, and (fold) the folded state
    launch_state_build<Tag, D>(k, v, lin, weight, fmap, BH, L, ws, ws + w.fwd.states_end, w.fwd, st);
  }
  if (!states) states = ws;
  const uint16_t* kvt = (const uint16_t*)(states + w.fwd.kvt);
  const uint16_t* z = (const uint16_t*)(states + w.fwd.z);
  float* m_part = (float*)(ws + w.m_part);
  if (steps & LB_QUERY) {
#define SLA_LBS_LAUNCH(FM, ACC)                                                                                            \
  hipLaunchKernelGGL((linear_bwd_stream_kernel<Tag, D, FM, ACC>), dim3(w.sp.nsplit, BH), dim3(512), 0, st, (const uint16_t*)q, \
                     (const uint16_t*)d_out, (const uint16_t*)(states + w.fwd.kvw), z, (uint16_t*)dq, lin, ldo, m_part,      \
                     (float*)(ws + w.dz_part), (float*)(ws + w.db_part), L, w.sp.rows_per_split)
#define SLA_LB_FMAPS(LAUNCH)                                          \
  if (accumulate) {                                                   \
    if (fmap == SLA_FMAP_ELU) LAUNCH(SLA_FMAP_ELU, true);             \
    else if (fmap == SLA_FMAP_RELU) LAUNCH(SLA_FMAP_RELU, true);      \
    else LAUNCH(SLA_FMAP_SOFTMAX, true);                              \
  } else {                                                            \
    if (fmap == SLA_FMAP_ELU) LAUNCH(SLA_FMAP_ELU, false);            \
    else if (fmap == SLA_FMAP_RELU) LAUNCH(SLA_FMAP_RELU, false);     \
    else LAUNCH(SLA_FMAP_SOFTMAX, false);                             \
  }
    SLA_LB_FMAPS(SLA_LBS_LAUNCH)
#undef SLA_LBS_LAUNCH
  }
  // (the line of the forward's states)
  const bool presum = w.sp.nsplit >= PRESUM_MIN_SLICES;
  if ((steps & LB_REDUCE) && presum)
    hipLaunchKernelGGL((linear_state_presum_kernel<D>), dim3(D * D / 256 + 2, BH), dim3(512), 0, st, m_part, (float*)(ws + w.dz_part),
                       (float*)(ws + w.db_part), w.sp.nsplit);
  if (steps & LB_REDUCE)
    hipLaunchKernelGGL((linear_bwd_finish_kernel<Tag, D>), dim3(xcd_grid(lists.wgs) + xcd_grid((int64_t)BH * (D / 8))), dim3(512),
                       0, st, (const float*)m_part, (const float*)(ws + w.dz_part), (const float*)(ws + w.db_part), weight, kvt,
                       (uint16_t*)(ws + w.ds), (uint16_t*)(ws + w.dst), (float*)(ws + w.dz), (float*)(ws + w.dw_head),
                       (float*)(ws + w.db_head), w.sp.nsplit, presum ? 1 : w.sp.nsplit, BH * (D / 8), xcd_grid(lists.wgs), lists);
  if (steps & LB_HEADS) launch_head_sums(hs, st);
  if (steps & LB_KEYS) {
#define SLA_LBK_LAUNCH(FM, ACC)                                                                                          \
  hipLaunchKernelGGL((linear_bwd_keys_kernel<Tag, D, FM, ACC>), dim3(w.sp.nsplit, BH), dim3(512), 0, st, (const uint16_t*)k, \
                     (const uint16_t*)v, (const uint16_t*)(ws + w.ds), (const uint16_t*)(ws + w.dst),                      \
                     (const float*)(ws + w.dz), (uint16_t*)dk, (uint16_t*)dv, lin, L, w.sp.rows_per_split)
    SLA_LB_FMAPS(SLA_LBK_LAUNCH)
#undef SLA_LBK_LAUNCH
#undef SLA_LB_FMAPS
  }
  return check_launch("linear_bwd");
}

// dW and db alone, from d(out) and the row-wise y a rows kernel has left (used by the backward of the complement-mode linear
// branch, whose state gradients are per query block and formed elsewhere): dW^T = y^T d(out) and db = sum d(out) are the state
// kernel's sums with d(out) and y in the place of k and v.  Returns the sum over the heads for a later launch to take along.
// `ws` is a region of weight_grads_workspace_bytes() bytes.
// Bound by memory.  12 heads x 16380 x 128: 34 us and their reduction 9, where a kernel that formed the states' gradients
// beside them, which this branch has per query block already, took 59 and its reduction 22.
struct WeightGradWs {
  LinSplit st;
  size_t dw_part, db_part, dw_head, db_head, total;
};
static WeightGradWs weight_grad_ws(int BH, int L, int D) {
  WeightGradWs w;
  const int min_rows = L >= 4096 ? 256 : cdiv(L, 16);             // (as in lin_ws)
  w.st = lin_split(BH, L, 512, D == 64 ? StateTile<64, false>::TR : StateTile<128, false>::TR, min_rows);
  const int64_t np = (int64_t)BH * w.st.nsplit;
  size_t off = 0;
  w.dw_part = off; off += align_up(np * D * D * 4, 256);
  w.db_part = off; off += align_up(np * D * 4, 256);
  w.dw_head = off; off += align_up((int64_t)BH * D * D * 4, 256);
  w.db_head = off; off += align_up((int64_t)BH * D * 4, 256);
  w.total = off;
  return w;
}
int64_t weight_grads_workspace_bytes(int BH, int L, int D) { return (int64_t)weight_grad_ws(BH, L, D).total; }

template <typename Tag, int D>
static HeadSums weight_grads_impl(const void* gout, const void* y, int BH, int L, char* ws, float* d_weight, float* d_bias,
                                  hipStream_t st) {
  const WeightGradWs w = weight_grad_ws(BH, L, D);
  float *const dw_head = (float*)(ws + w.dw_head), *const db_head = (float*)(ws + w.db_head);
  hipLaunchKernelGGL((linear_state_partial_kernel<Tag, D, false, false, false, true>), dim3(w.st.nsplit, BH),
                     dim3(StateTile<D, false>::NTH), 0, st, (const uint16_t*)gout, (const uint16_t*)y, contiguous_layout(BH, L, D),
                     (void*)(ws + w.dw_part), (float*)(ws + w.db_part), L, w.st.rows_per_split, 0);
  hipLaunchKernelGGL(linear_bwd_reduce_kernel, dim3(cdiv(D * D, 256), BH), dim3(256), 0, st, (const float*)(ws + w.dw_part),
                     (const float*)(ws + w.db_part), dw_head, db_head, w.st.nsplit, D);
  return HeadSums{dw_head, db_head, d_weight, d_bias, BH, D, D * D / 256};
}
HeadSums launch_weight_grads(int dtype, int D, const void* gout, const void* y, int BH, int L, char* ws, float* d_weight,
                             float* d_bias, hipStream_t st) {
  if (dtype == SLA_BF16) {
    if (D == 128) return weight_grads_impl<bf16_tag, 128>(gout, y, BH, L, ws, d_weight, d_bias, st);
    return weight_grads_impl<bf16_tag, 64>(gout, y, BH, L, ws, d_weight, d_bias, st);
  }
  if (D == 128) return weight_grads_impl<f16_tag, 128>(gout, y, BH, L, ws, d_weight, d_bias, st);
  return weight_grads_impl<f16_tag, 64>(gout, y, BH, L, ws, d_weight, d_bias, st);
}

int linear_bwd_steps(const void* q, const void* k, const void* v, const int64_t* qkv_strides, const float* weight,
                     const float* bias, const void* d_out, const int64_t* do_strides, void* dq, void* dk, void* dv,
                     float* d_weight, float* d_bias, int dtype, int fmap, int B, int H, int L, int D, int flags,
                     const void* states, void* workspace, int64_t workspace_bytes, void* stream, int steps, const ColLists* lists,
                     HeadSums* heads, LinearKeys* keys) {
  int rc = validate_linear(dtype, fmap, B, H, L, D);
  if (rc) return rc;
  SLA_REQUIRE((flags & ~(SLA_BWD_ACCUMULATE | SLA_BWD_STATES_READY)) == 0, SLA_ERR_BAD_ARG, "unknown flag bits in %d", flags);
  (void)bias;  // the bias does not enter any gradient
  SLA_REQUIRE(q && k && v && weight && d_out && dq && dk && dv && d_weight && d_bias && workspace, SLA_ERR_BAD_ARG,
              "null pointer");
  SLA_REQUIRE(((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)d_out | (uintptr_t)dq | (uintptr_t)dk | (uintptr_t)dv |
               (uintptr_t)weight | (uintptr_t)states | (uintptr_t)workspace) % 16 == 0,
              SLA_ERR_BAD_ARG, "pointers must be 16-byte aligned");
  const int BH = B * H;
  const int64_t need = (int64_t)lin_bwd_ws(BH, L, D, !states).total;
  SLA_REQUIRE(workspace_bytes >= need, SLA_ERR_WORKSPACE, "workspace of %lld bytes, need %lld", (long long)workspace_bytes,
              (long long)need);
  RowLayout lin, ldo;
  rc = make_layout(qkv_strides, B, H, L, D, 2, &lin);
  if (rc) return rc;
  rc = make_layout(do_strides, B, H, L, D, 2, &ldo);
  if (rc) return rc;
  hipStream_t st = (hipStream_t)stream;
  char* ws = (char*)workspace;
#define SLA_LINB_CASE(TAG, DD) \
  return linear_bwd_impl<TAG, DD>(q, k, v, weight, d_out, dq, dk, dv, lin, ldo, d_weight, d_bias, fmap, BH, L, flags, (const char*)states, ws, st, \
                                  steps, lists ? *lists : ColLists{}, heads, keys)
  if (dtype == SLA_BF16) {
    if (D == 128) SLA_LINB_CASE(bf16_tag, 128);
    SLA_LINB_CASE(bf16_tag, 64);
  }
  if (D == 128) SLA_LINB_CASE(f16_tag, 128);
  SLA_LINB_CASE(f16_tag, 64);
#undef SLA_LINB_CASE
}

}  // namespace sla

using namespace sla;

extern "C" int sla_linear_bwd(const void* q, const void* k, const void* v, const float* weight, const float* bias,
                              const void* d_out, void* dq, void* dk, void* dv, float* d_weight, float* d_bias, int dtype,
                              int fmap, int B, int H, int L, int D, int flags, void* workspace,
                              int64_t workspace_bytes, void* stream) {
  return linear_bwd_steps(q, k, v, nullptr, weight, bias, d_out, nullptr, dq, dk, dv, d_weight, d_bias, dtype, fmap, B, H, L,
                          D, flags, nullptr, workspace, workspace_bytes, stream, LB_ALL);
}

extern "C" int sla_linear_bwd_strided(const void* q, const void* k, const void* v, const int64_t* qkv_strides,
                                      const float* weight, const float* bias, const void* d_out, const int64_t* do_strides,
                                      void* dq, void* dk, void* dv, float* d_weight, float* d_bias, int dtype, int fmap,
                                      int B, int H, int L, int D, int flags, void* workspace, int64_t workspace_bytes,
                                      void* stream) {
  SLA_REQUIRE(qkv_strides && do_strides, SLA_ERR_BAD_ARG, "null strides");
  return linear_bwd_steps(q, k, v, qkv_strides, weight, bias, d_out, do_strides, dq, dk, dv, d_weight, d_bias, dtype, fmap, B,
                          H, L, D, flags, nullptr, workspace, workspace_bytes, stream, LB_ALL);
}
