// Forward of the whole module (mask builder, linear branch's states, attention with the linear branch in its epilogue) as
// one call.
//
// Stands in for SparseLinearAttention.forward of the reference (sparse_linear_attention/core.py:69-105).  On `stream`, launches
// that need nothing of each other in one:
//     block means of q, chunk sums of k [fp32 inputs: and the 16-bit copies] | slices' partial states, column mean of k |
//     states finished, block means of k | scores and selection | attention
// (five launches; in eight of their own, and seven with 16-bit inputs, everything before the attention took 34 us for 2 heads x
// 1024 x 64 in fp32, 57 for 8 x 4096 x 128: now 25 and 43.  A sixth adds up the slices' states from 40 slices per head on; scores and
// selection are two where a row's scores go through memory.)
// From 64 MiB per tensor on the state build (k, v only) runs on the caller's second stream beside the mask builder instead.
#include "block_pool.h"
#include "fwd_steps.h"
#include "linear_state.h"
#include "side_events.h"

namespace sla {

// First pass over q and k (pool_pair_body); grid (., heads, 2).  Cast: fp32 inputs, whose 16-bit copies leave on the way (n
// elements each, one after the other in `cast`); blockIdx.z == 2 copies v.
template <typename IO, int W, typename Cast>
__global__ __launch_bounds__(256) void prefix_pool_kernel(const typename IO::raw* __restrict__ q, const typename IO::raw* __restrict__ k,
                                                          const typename IO::raw* __restrict__ v, const RowLayout lay,
                                                          const MapParts m, int BLKQ, int L, int D, uint16_t* __restrict__ cast,
                                                          int64_t n) {
  if (!__is_same(Cast, NoCast) && blockIdx.z == 2) {
    if constexpr (!__is_same(Cast, NoCast)) {
      const int64_t stride = (int64_t)gridDim.x * gridDim.y * 256 * 8;
      for (int64_t i = (((int64_t)blockIdx.y * gridDim.x + blockIdx.x) * 256 + threadIdx.x) * 8; i < n; i += stride) {
        const f32x4_t x = *reinterpret_cast<const f32x4_t*>(v + i), y = *reinterpret_cast<const f32x4_t*>(v + i + 4);
        i32x4_t w;
        w[0] = (int)Elem<Cast>::pack2(x[0], x[1]);
        w[1] = (int)Elem<Cast>::pack2(x[2], x[3]);
        w[2] = (int)Elem<Cast>::pack2(y[0], y[1]);
        w[3] = (int)Elem<Cast>::pack2(y[2], y[3]);
        *reinterpret_cast<i32x4_t*>(cast + 2 * n + i) = w;
      }
    }
    return;
  }
  pool_pair_body<IO, W, Cast>(k, m.chunk_sums, m.nchunk, q, lay, (typename IO::raw*)m.pq, BLKQ, m.M, L, D, m.tiled, blockIdx.x,
                              blockIdx.y, blockIdx.z, cast, n);
}

// The slices' partial states and, in the workgroups from `state_wgs` on, the column mean of k; one head's slices are adjacent.  (The
// means' workgroups, D / 16 short ones per head, ahead of the slices: from 320 of them on a slice per compute unit no longer
// starts everywhere at once.  Forward, ahead / behind: 48 heads x 4096 x 128 158 / 149 us, 72 x 2500 x 128 153 / 140, 100 x 2500 x 64 101.4
// / 96.1; up to 288 of them equal.)
template <typename Tag, int D, typename IO>
__global__ __launch_bounds__((StateTile<D, false>::NTH)) __attribute__((amdgpu_waves_per_eu(4, 4))) void prefix_state_kernel(
    const uint16_t* __restrict__ k, const uint16_t* __restrict__ v, const RowLayout lay, float* __restrict__ kv_part,
    float* __restrict__ z_part, int L, int rows_per_split, int nsplit, int fmap, const MapParts m, int state_wgs) {
  static_assert(COLMEAN_MAX_GROUPS * COLMEAN_SLAB * 4 <= StateTile<D, false>::LDS, "the column mean's sums fit the tiles");
  __shared__ __attribute__((aligned(16))) char smem[StateTile<D, false>::LDS];
  const int wg = blockIdx.x, mean = wg - state_wgs;
  if (mean >= 0) {
    colmean_body<IO, StateTile<D, false>::NTH>(m.chunk_sums, (typename IO::raw*)m.colmean, m.nchunk, (m.nchunk + KMEAN_GROUP - 1) / KMEAN_GROUP, D, L,
                     mean % (D / COLMEAN_SLAB), mean / (D / COLMEAN_SLAB), reinterpret_cast<float*>(smem));
    return;
  }
  const int bh = wg / nsplit;
  state_partial_body<Tag, D, false, false, false>(k, v, lay, kv_part, z_part, L, rows_per_split, fmap, nullptr, nullptr,
                                                  wg - bh * nsplit, bh, nsplit, smem);
}

// The states finished and, in the workgroups from `first_pool` on (`per_head` for each head), the block means of k.
template <typename Tag, int D, typename IO, int W>
__global__ __launch_bounds__(512) void prefix_finish_kernel(const StateFinish job, int first_pool, const typename IO::raw* __restrict__ k,
                                                            const RowLayout lay, const MapParts m, int L, int per_head) {
  __shared__ __attribute__((aligned(16))) char smem[state_finish_lds<D>()];
  const int wg = blockIdx.x;
  if (wg < first_pool) {
    const int logical = xcd_remap(wg, first_pool, job.total);
    if (logical >= 0) state_finish_body<Tag, D>(job, logical, smem);
    return;
  }
  const int bh = (wg - first_pool) / per_head;
  pool_body<IO, 2, W, 512>(k, lay, (const typename IO::raw*)m.colmean, m.pk, L, D, 64, m.N, m.tiled, wg - first_pool - bh * per_head, bh);
}

template <typename IO, typename Cast>
static void launch_prefix_pool(const void* q, const void* k, const void* v, const RowLayout& lay, const MapParts& m, int in_dtype,
                               int BLKQ, int BH, int L, int D, void* cast, hipStream_t st) {
  typedef typename IO::raw raw;
  const int64_t n = (int64_t)BH * L * D;
  const int z = __is_same(Cast, NoCast) ? 2 : 3;
#define SLA_POOL_CASE(W)                                                                                                      \
  hipLaunchKernelGGL((prefix_pool_kernel<IO, W, Cast>), dim3(cdiv(max(m.nchunk, m.M), 256 / (D / (W))), BH, z), dim3(256), 0, st, \
                     (const raw*)q, (const raw*)k, (const raw*)v, lay, m, BLKQ, L, D, (uint16_t*)cast, n)
  if (narrow_pools(in_dtype, BH, L, D)) SLA_POOL_CASE(IO::VEC / 4);
  else SLA_POOL_CASE(IO::VEC);
#undef SLA_POOL_CASE
}

// partial states | column mean; states finished | block means of k
template <typename IO, typename Tag, int D>
static void launch_prefix_rest(const void* k, const RowLayout& lin, const void* kc, const void* vc, const RowLayout& lay, const MapParts& m,
                               int in_dtype, const float* weight, int fmap, int BH, int L, char* states, char* parts, hipStream_t st) {
  typedef typename IO::raw raw;
  const LinWs w = lin_ws(BH, L, D);
  const int state_wgs = BH * w.nsplit;
  hipLaunchKernelGGL((prefix_state_kernel<Tag, D, IO>), dim3(state_wgs + BH * (D / COLMEAN_SLAB)), dim3(StateTile<D, false>::NTH), 0, st, (const uint16_t*)kc,
                     (const uint16_t*)vc, lay, (float*)(parts + (w.kv_part - w.states_end)),
                     (float*)(parts + (w.z_part - w.states_end)), L, w.rows_per_split, w.nsplit, fmap, m, state_wgs);
  launch_state_presum<D>(BH, parts, w, st);
  const StateFinish job = state_finish_job<D>(weight, BH, states, parts, w);
#define SLA_FINISH_CASE(W)                                                                                                   \
  {                                                                                                                          \
    const int per_head = cdiv(m.N, 512 / (D / (W)));                                                                         \
    hipLaunchKernelGGL((prefix_finish_kernel<Tag, D, IO, W>), dim3(xcd_grid(job.total) + BH * per_head), dim3(512), 0, st, job, \
                       xcd_grid(job.total), (const raw*)k, lin, m, L, per_head);                                             \
  }
  if (narrow_pools(in_dtype, BH, L, D)) SLA_FINISH_CASE(IO::VEC / 4)
  else SLA_FINISH_CASE(IO::VEC)
#undef SLA_FINISH_CASE
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
  SLA_REQUIRE(in_dtype == dtype || in_dtype == SLA_F32 || in_dtype == SLA_F32_BOTH || in_dtype == SLA_MASK_GIVEN, SLA_ERR_BAD_ARG,
              "in_dtype %d is neither fp32 nor the compute dtype", in_dtype);
  const int out32 = in_dtype == SLA_F32_BOTH;
  if (out32) in_dtype = SLA_F32;
  const bool casts = in_dtype == SLA_F32, mask_given = in_dtype == SLA_MASK_GIVEN;
  if (mask_given) in_dtype = dtype;
  SLA_REQUIRE(q && k && v && weight && bias && out && lse && (lut || topk == 0) && states && workspace && (cast || !casts),
              SLA_ERR_BAD_ARG, "null pointer");
  SLA_REQUIRE(((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)cast | (uintptr_t)weight | (uintptr_t)out | (uintptr_t)o_s |
               (uintptr_t)lut | (uintptr_t)states | (uintptr_t)workspace) % 16 == 0,
              SLA_ERR_BAD_ARG, "pointers must be 16-byte aligned");
  SLA_REQUIRE(!casts || !qkv_strides, SLA_ERR_BAD_ARG, "fp32 inputs are contiguous");
  SLA_REQUIRE(!out32 || !out_strides, SLA_ERR_BAD_ARG, "an fp32 output is contiguous");
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
  MapParts m{};
  RowLayout lmap = lin;                // (q and k as the mask builder reads them: the inputs themselves)
  if (!mask_given) m = block_map_parts(in_dtype, BH, L, D, BLKQ, BLKK, map_part, map_bytes);
  if (casts) {
    const int64_t n = (int64_t)BH * L * D;
    if (dtype == SLA_BF16) launch_prefix_pool<IoF32, bf16_tag>(q, k, v, lmap, m, in_dtype, BLKQ, BH, L, D, cast, st);
    else launch_prefix_pool<IoF32, f16_tag>(q, k, v, lmap, m, in_dtype, BLKQ, BH, L, D, cast, st);
    qc = cast;
    kc = (uint16_t*)cast + n;
    vc = (uint16_t*)cast + 2 * n;
  }
  const int lut64 = lut_elem_bytes == 8;
  const auto attention = [&]() {
    return attn_linear_run(qc, kc, vc, lin, lut, lut_elem_bytes, (const char*)states, bias, o_s, out, lout, lse, dtype, fmap, BH,
                           L, D, BLKQ, topk, qk_scale, st, out32);
  };
  const bool two = side && side != st && side_stream_pays_fwd(B, H, L, D);
  if (!two) {
    if (mask_given) {
      if ((rc = linear_state_run(kc, vc, lin, weight, dtype, fmap, BH, L, D, (char*)states, parts, st))) return rc;
      return attention();
    }
    if (in_dtype == SLA_BF16) launch_prefix_pool<IoBf16, NoCast>(q, k, v, lmap, m, in_dtype, BLKQ, BH, L, D, nullptr, st);
    else if (in_dtype == SLA_F16) launch_prefix_pool<IoF16, NoCast>(q, k, v, lmap, m, in_dtype, BLKQ, BH, L, D, nullptr, st);
#define SLA_REST_CASE(IO, TAG)                                                                                                  \
  if (D == 128)                                                                                                                 \
    launch_prefix_rest<IO, TAG, 128>(k, lmap, kc, vc, lin, m, in_dtype, weight, fmap, BH, L, (char*)states, parts, st);         \
  else                                                                                                                          \
    launch_prefix_rest<IO, TAG, 64>(k, lmap, kc, vc, lin, m, in_dtype, weight, fmap, BH, L, (char*)states, parts, st)
    if (casts && dtype == SLA_BF16) {
      SLA_REST_CASE(IoF32, bf16_tag);
    } else if (casts) {
      SLA_REST_CASE(IoF32, f16_tag);
    } else if (dtype == SLA_BF16) {
      SLA_REST_CASE(IoBf16, bf16_tag);
    } else {
      SLA_REST_CASE(IoF16, f16_tag);
    }
#undef SLA_REST_CASE
    block_map_select(in_dtype, m, BH, D, topk, sparse_map, lut, lut64, st);
    return attention();
  }
  std::lock_guard<std::mutex> lock(side_events_mutex());
  SideEvents* ev;
  if ((rc = side_events_for_current_device(&ev))) return rc;
  SLA_HIP_OK(hipEventRecord(ev->fork, st));
  SLA_HIP_OK(hipStreamWaitEvent(side, ev->fork, 0));
  // (once the second stream waits on `stream`, no path leaves without `stream` waiting for it in turn)
  rc = linear_state_run(kc, vc, lin, weight, dtype, fmap, BH, L, D, (char*)states, parts, side);
  const int rc_mask = mask_given ? (int)SLA_OK
                                 : block_map_run(q, k, lmap, in_dtype, m, BH, L, D, BLKQ, BLKK, topk, sparse_map, lut, lut64, !casts, st);
  SLA_HIP_OK(hipEventRecord(ev->join, side));
  SLA_HIP_OK(hipStreamWaitEvent(st, ev->join, 0));
  if (rc) return rc;
  if (rc_mask) return rc_mask;
  return attention();
}
