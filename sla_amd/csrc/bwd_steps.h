// The two backward calls of the module cut into steps, so that one caller can order the kernels of both and let the short
// ones ride in launches of the long ones (module_bwd.hip); each call on its own runs every step.
#pragma once
#include "bwd_lists.h"
#include "common.h"

namespace sla {

// block-sparse attention backward
constexpr int SB_LISTS = 1;   // per-key-block lists of the map (needs the map only); or the caller runs the job `lists` receives
constexpr int SB_DQ = 2;      // delta and dQ, the work items of dK / dV (needs the lists), and the caller's sum over the heads
constexpr int SB_DKDV = 4;    // dK / dV over the lists (needs SB_DQ)
constexpr int SB_ALL = 7;
constexpr int SB_ADD = 8;     // dq, dk, dv already hold another branch's gradients: add to them
int attn_bwd_steps(const void* q, const void* k, const void* v, const int64_t* qkv_strides, const void* o, const void* d_o,
                   const int64_t* do_strides, const float* lse, const int8_t* sparse_map, const void* lut, int lut_elem_bytes,
                   void* dq, void* dk, void* dv, int dtype, int B, int H, int L, int D, int BLKQ, int BLKK, int topk,
                   float qk_scale, void* workspace, int64_t workspace_bytes, void* stream, int steps,
                   const HeadSums* heads = nullptr, ColLists* lists = nullptr);

// linear branch backward
constexpr int LB_STATES = 1;  // the forward's per-head states again (skipped with SLA_BWD_STATES_READY)
constexpr int LB_QUERY = 2;   // dq and the sums over the rows (needs LB_STATES)
constexpr int LB_REDUCE = 4;  // dS, dz and the heads' weight gradients from those sums; `lists` rides along
constexpr int LB_HEADS = 8;   // d_weight, d_bias; or the caller runs the job `heads` receives (needs LB_REDUCE)
constexpr int LB_KEYS = 16;   // dk, dv (needs LB_REDUCE)
constexpr int LB_ALL = 31;
int linear_bwd_steps(const void* q, const void* k, const void* v, const int64_t* qkv_strides, const float* weight,
                     const float* bias, const void* d_out, const int64_t* do_strides, void* dq, void* dk, void* dv,
                     float* d_weight, float* d_bias, int dtype, int fmap, int B, int H, int L, int D, int flags,
                     const void* states, void* workspace, int64_t workspace_bytes, void* stream, int steps,
                     const ColLists* lists = nullptr, HeadSums* heads = nullptr);
// (states: the forward's finished states where they lie, or null: they are built, or with SLA_BWD_STATES_READY found, at the
//  start of the workspace.  With states given the workspace needs linear_bwd_states_apart_bytes() only.)
int64_t linear_bwd_states_apart_bytes(int BH, int L, int D);
int64_t sparse_bwd_workspace_bytes(int BH, int L, int D, int BLKQ, int BLKK, int topk);
void launch_head_sums(const HeadSums& heads, hipStream_t st);

}  // namespace sla
