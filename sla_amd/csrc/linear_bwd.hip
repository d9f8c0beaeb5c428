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
//   finish : those sums added up -> dS (16 bit, both orientations), dz, per-head dW, db
//   heads  : the heads' dW and db added up
//   keys   : k and v once: dk, dv
// The complement-mode branch forms dW and db with the states / reduce kernels below, from row-wise temporaries.
#include "bwd_steps.h"
#include "linear_bwd_stream.h"

namespace sla {

// ---- states -------------------------------------------------------------------------------
// grid (nsplit, BH).  dS^T partial [d2][d1] per (bh, split); dW^T partial [d][e] per (bh, split).
template <typename Tag, int D>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void linear_bwd_states_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ dn, const uint16_t* __restrict__ gout,
    const uint16_t* __restrict__ y, const float* __restrict__ dden, const RowLayout lin, const RowLayout ldo,
    float* __restrict__ ds_part, float* __restrict__ dw_part, float* __restrict__ dz_part, float* __restrict__ db_part, int L,
    int rows_per_split, int fmap) {
  using E = Elem<Tag>;
  constexpr int TR = 64;
  constexpr int STR = D + 16;
  constexpr int CPR = D / 8;
  constexpr int RPP = 256 / CPR;
  constexpr int NP = TR / RPP;
  constexpr int DT = D / 32;
  constexpr int WPT = (DT * DT) / 4;

  __shared__ __attribute__((aligned(16))) uint16_t sA[TR * STR];
  __shared__ __attribute__((aligned(16))) uint16_t sDN[TR * STR];
  __shared__ __attribute__((aligned(16))) uint16_t sG[TR * STR];
  __shared__ __attribute__((aligned(16))) uint16_t sY[TR * STR];
  // the cross-thread sums of dz / db at the very end reuse the first two tiles (two workgroups per
  // compute unit need the LDS footprint below 80 KB)
  static_assert(2 * TR * STR * 2 >= 2 * RPP * D * 4, "reduction scratch does not fit the tiles it reuses");
  float (*sRed)[RPP][D] = reinterpret_cast<float (*)[RPP][D]>(sA);

  const int split = blockIdx.x, bh = blockIdx.y, nsplit = gridDim.x;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int g = lane >> 5;
  const int row_begin = split * rows_per_split;
  const int row_end = min(L, row_begin + rows_per_split);
  const size_t head_off = (size_t)bh * L * D;
  const int lrow = tid / CPR, lcol = (tid % CPR) * 8;

  f32x16_t sacc[WPT], wacc[WPT];
#pragma unroll
  for (int t = 0; t < WPT; ++t)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      sacc[t][i] = 0.f;
      wacc[t][i] = 0.f;
    }
  float zacc[8], bacc[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    zacc[e] = 0.f;
    bacc[e] = 0.f;
  }
  const int tr_row = (lane & 15) >> 2;
  const int tr_col = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);

  // (no register prefetch of the next tile: the second workgroup on the compute unit covers the latency,
  //  and the registers it would take are what lets that second workgroup fit)
  i16x8_t rq[NP], rdn[NP], rg[NP], ry[NP];
  float rdd[NP];
  auto fetch = [&](int r0) {
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const int grow = r0 + lrow + p * RPP;
      rq[p] = i16x8_t{0, 0, 0, 0, 0, 0, 0, 0};
      rdn[p] = rq[p];
      rg[p] = rq[p];
      ry[p] = rq[p];
      rdd[p] = 0.f;
      if (grow < row_end) {
        const size_t off = head_off + (size_t)grow * D + lcol;          // dn, y: contiguous temporaries
        rq[p] = *reinterpret_cast<const i16x8_t*>(q + lin.head(bh) + (size_t)grow * (size_t)lin.sl + lcol);
        rdn[p] = *reinterpret_cast<const i16x8_t*>(dn + off);
        rg[p] = *reinterpret_cast<const i16x8_t*>(gout + ldo.head(bh) + (size_t)grow * (size_t)ldo.sl + lcol);
        ry[p] = *reinterpret_cast<const i16x8_t*>(y + off);
        rdd[p] = dden[(size_t)bh * L + grow];
      }
    }
  };
  for (int r0 = row_begin; r0 < row_end; r0 += TR) {
    fetch(r0);
    __syncthreads();
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const int row = lrow + p * RPP;
      const int grow = r0 + row;
      const bool ok = grow < row_end;
      const i16x8_t xq = rq[p], xdn = rdn[p], xg = rg[p], xy = ry[p];
      const float dd = rdd[p];
      float f[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) f[e] = E::to_float((uint16_t)xq[e]);
      if (fmap == SLA_FMAP_SOFTMAX) {
        float mx = f[0];
#pragma unroll
        for (int e = 1; e < 8; ++e) mx = fmaxf(mx, f[e]);
#pragma unroll
        for (int s = 1; s < CPR; s <<= 1) mx = fmaxf(mx, __shfl_xor(mx, s));
        float sum = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          f[e] = __expf(f[e] - mx);
          sum += f[e];
        }
#pragma unroll
        for (int s = 1; s < CPR; s <<= 1) sum += __shfl_xor(sum, s);
        const float inv = 1.0f / sum;
#pragma unroll
        for (int e = 0; e < 8; ++e) f[e] = round16<Tag>(f[e] * inv);
      } else if (fmap == SLA_FMAP_RELU) {
#pragma unroll
        for (int e = 0; e < 8; ++e) f[e] = fmap_pointwise<Tag>(SLA_FMAP_RELU, f[e]);
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) f[e] = fmap_pointwise<Tag>(SLA_FMAP_ELU, f[e]);
      }
      i16x8_t fa;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        if (!ok) f[e] = 0.f;
        zacc[e] += dd * f[e];
        bacc[e] += E::to_float((uint16_t)xg[e]);
        fa[e] = (short)E::from_float(f[e]);
      }
      *reinterpret_cast<i16x8_t*>(&sA[row * STR + lcol]) = fa;
      *reinterpret_cast<i16x8_t*>(&sDN[row * STR + lcol]) = xdn;
      *reinterpret_cast<i16x8_t*>(&sG[row * STR + lcol]) = xg;
      *reinterpret_cast<i16x8_t*>(&sY[row * STR + lcol]) = xy;
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < TR / 16; ++c) {
      const int l0 = 16 * c + 8 * g + tr_row;
#pragma unroll
      for (int t = 0; t < WPT; ++t) {
        const int tile = wave * WPT + t;
        const int mt = tile / DT, nt = tile % DT;
        const uint16_t* pa = &sA[l0 * STR + 32 * mt + tr_col];
        const uint16_t* pb = &sDN[l0 * STR + 32 * nt + tr_col];
        sacc[t] = E::mfma32(concat4(lds_read_tr16(pa), lds_read_tr16(pa + 4 * STR)),
                            concat4(lds_read_tr16(pb), lds_read_tr16(pb + 4 * STR)), sacc[t]);
        const uint16_t* pg = &sG[l0 * STR + 32 * mt + tr_col];
        const uint16_t* py = &sY[l0 * STR + 32 * nt + tr_col];
        wacc[t] = E::mfma32(concat4(lds_read_tr16(pg), lds_read_tr16(pg + 4 * STR)),
                            concat4(lds_read_tr16(py), lds_read_tr16(py + 4 * STR)), wacc[t]);
      }
    }
  }
  // accumulator: rows = first operand's index (d1 / e), column = second operand's index (d2 / d);
  // stored with the column as the slow axis: part[col][row]
  const size_t pidx = (size_t)bh * nsplit + split;
  float* so = ds_part + pidx * D * D;
  float* wo = dw_part + pidx * D * D;
#pragma unroll
  for (int t = 0; t < WPT; ++t) {
    const int tile = wave * WPT + t;
    const int mt = tile / DT, nt = tile % DT;
    const int col = 32 * nt + (lane & 31);
#pragma unroll
    for (int i4 = 0; i4 < 4; ++i4) {
      const f32x4_t a = {sacc[t][4 * i4], sacc[t][4 * i4 + 1], sacc[t][4 * i4 + 2], sacc[t][4 * i4 + 3]};
      const f32x4_t b = {wacc[t][4 * i4], wacc[t][4 * i4 + 1], wacc[t][4 * i4 + 2], wacc[t][4 * i4 + 3]};
      *reinterpret_cast<f32x4_t*>(so + (size_t)col * D + 32 * mt + 8 * i4 + 4 * g) = a;
      *reinterpret_cast<f32x4_t*>(wo + (size_t)col * D + 32 * mt + 8 * i4 + 4 * g) = b;
    }
  }
  __syncthreads();
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    sRed[0][lrow][lcol + e] = zacc[e];
    sRed[1][lrow][lcol + e] = bacc[e];
  }
  __syncthreads();
  if (tid < D) {
    float s0 = 0.f, s1 = 0.f;
#pragma unroll
    for (int rr = 0; rr < RPP; ++rr) {
      s0 += sRed[0][rr][tid];
      s1 += sRed[1][rr][tid];
    }
    dz_part[pidx * D + tid] = s0;
    db_part[pidx * D + tid] = s1;
  }
}

// ---- reduce -------------------------------------------------------------------------------
// Stage 1, grid (cdiv(D*D,256), BH): per head, add the split partials in ascending order:
//   dS (16 bit, both orientations), dz, and this head's dW^T / db (fp32).
// Stage 2 (head_sums_body): add the per-head dW^T / db in ascending head order.
template <typename Tag>
__global__ __launch_bounds__(256) void linear_bwd_reduce_kernel(const float* __restrict__ ds_part,
                                                                const float* __restrict__ dw_part,
                                                                const float* __restrict__ dz_part,
                                                                const float* __restrict__ db_part, uint16_t* __restrict__ ds,
                                                                uint16_t* __restrict__ dst, float* __restrict__ dz,
                                                                float* __restrict__ dw_head, float* __restrict__ db_head,
                                                                int nsplit, int D) {
  using E = Elem<Tag>;
  const int DD = D * D;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int bh = blockIdx.y;
  if (i < DD) {
    const float* p = ds_part + (size_t)bh * nsplit * DD + i;
    const float* pw = dw_part + (size_t)bh * nsplit * DD + i;
    float s = 0.f, sw = 0.f;
#pragma unroll 8
    for (int sp = 0; sp < nsplit; ++sp) {
      s += p[(size_t)sp * DD];
      sw += pw[(size_t)sp * DD];
    }
    const int d2 = i / D, d1 = i % D;   // partial layout [d2][d1]
    const uint16_t h = E::from_float(s);
    dst[(size_t)bh * DD + i] = h;                 // dS^T [d2][d1]
    ds[(size_t)bh * DD + d1 * D + d2] = h;        // dS   [d1][d2]
    dw_head[(size_t)bh * DD + i] = sw;            // dW^T [d][e] of this head
  }
  if (i < D) {
    const float* p = dz_part + (size_t)bh * nsplit * D + i;
    const float* pb = db_part + (size_t)bh * nsplit * D + i;
    float s = 0.f, sb = 0.f;
    for (int sp = 0; sp < nsplit; ++sp) {
      s += p[(size_t)sp * D];
      sb += pb[(size_t)sp * D];
    }
    dz[(size_t)bh * D + i] = s;
    db_head[(size_t)bh * D + i] = sb;
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
                           const ColLists& lists, HeadSums* heads) {
  const LinBwdWs w = lin_bwd_ws(BH, L, D, !states);
  const HeadSums hs = {(const float*)(ws + w.dw_head), (const float*)(ws + w.db_head), d_weight, d_bias, BH, D, D * D / 256};
  if (heads) *heads = hs;
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
  if (steps & LB_REDUCE)
    hipLaunchKernelGGL((linear_bwd_finish_kernel<Tag, D>), dim3(xcd_grid(lists.wgs) + xcd_grid((int64_t)BH * (D / 8))), dim3(512),
                       0, st, (const float*)m_part, (const float*)(ws + w.dz_part), (const float*)(ws + w.db_part), weight, kvt,
                       (uint16_t*)(ws + w.ds), (uint16_t*)(ws + w.dst), (float*)(ws + w.dz), (float*)(ws + w.dw_head),
                       (float*)(ws + w.db_head), w.sp.nsplit, BH * (D / 8), xcd_grid(lists.wgs), lists);
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

// dW and db alone, from the row-wise temporaries a rows kernel has left (used by the backward of the complement-mode
// linear branch, whose state gradients are per query block and formed elsewhere): the states kernel, its reduction and
// the sum over the heads.  `ws` is a region of weight_grads_workspace_bytes() bytes.
struct WeightGradWs {
  LinSplit st;
  size_t ds_part, dw_part, dz_part, db_part, ds, dst, dz, dw_head, db_head, total;
};
static WeightGradWs weight_grad_ws(int BH, int L, int D) {
  WeightGradWs w;
  w.st = lin_split(BH, L, 512);
  const int64_t np = (int64_t)BH * w.st.nsplit;
  size_t off = 0;
  w.ds_part = off; off += align_up(np * D * D * 4, 256);
  w.dw_part = off; off += align_up(np * D * D * 4, 256);
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
int64_t weight_grads_workspace_bytes(int BH, int L, int D) { return (int64_t)weight_grad_ws(BH, L, D).total; }

template <typename Tag, int D>
static void weight_grads_impl(const void* q, const void* dn, const void* gout, const void* y, const float* dden, int BH, int L,
                              int fmap, char* ws, float* d_weight, float* d_bias, hipStream_t st) {
  const WeightGradWs w = weight_grad_ws(BH, L, D);
  const RowLayout lay = contiguous_layout(BH, L, D);
  hipLaunchKernelGGL((linear_bwd_states_kernel<Tag, D>), dim3(w.st.nsplit, BH), dim3(256), 0, st, (const uint16_t*)q,
                     (const uint16_t*)dn, (const uint16_t*)gout, (const uint16_t*)y, dden, lay, lay, (float*)(ws + w.ds_part),
                     (float*)(ws + w.dw_part), (float*)(ws + w.dz_part), (float*)(ws + w.db_part), L, w.st.rows_per_split, fmap);
  hipLaunchKernelGGL((linear_bwd_reduce_kernel<Tag>), dim3(cdiv(D * D, 256), BH), dim3(256), 0, st,
                     (const float*)(ws + w.ds_part), (const float*)(ws + w.dw_part), (const float*)(ws + w.dz_part),
                     (const float*)(ws + w.db_part), (uint16_t*)(ws + w.ds), (uint16_t*)(ws + w.dst), (float*)(ws + w.dz),
                     (float*)(ws + w.dw_head), (float*)(ws + w.db_head), w.st.nsplit, D);
  launch_head_sums(HeadSums{(const float*)(ws + w.dw_head), (const float*)(ws + w.db_head), d_weight, d_bias, BH, D, D * D / 256},
                   st);
}
void launch_weight_grads(int dtype, int D, const void* q, const void* dn, const void* gout, const void* y, const float* dden,
                         int BH, int L, int fmap, char* ws, float* d_weight, float* d_bias, hipStream_t st) {
  if (dtype == SLA_BF16) {
    if (D == 128) weight_grads_impl<bf16_tag, 128>(q, dn, gout, y, dden, BH, L, fmap, ws, d_weight, d_bias, st);
    else weight_grads_impl<bf16_tag, 64>(q, dn, gout, y, dden, BH, L, fmap, ws, d_weight, d_bias, st);
  } else {
    if (D == 128) weight_grads_impl<f16_tag, 128>(q, dn, gout, y, dden, BH, L, fmap, ws, d_weight, d_bias, st);
    else weight_grads_impl<f16_tag, 64>(q, dn, gout, y, dden, BH, L, fmap, ws, d_weight, d_bias, st);
  }
}

int linear_bwd_steps(const void* q, const void* k, const void* v, const int64_t* qkv_strides, const float* weight,
                     const float* bias, const void* d_out, const int64_t* do_strides, void* dq, void* dk, void* dv,
                     float* d_weight, float* d_bias, int dtype, int fmap, int B, int H, int L, int D, int flags,
                     const void* states, void* workspace, int64_t workspace_bytes, void* stream, int steps, const ColLists* lists,
                     HeadSums* heads) {
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
                                  steps, lists ? *lists : ColLists{}, heads)
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
