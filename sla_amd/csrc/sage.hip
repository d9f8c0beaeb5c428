// SageSLA quantised forward for gfx950: INT8 QK^T and FP8 (e4m3) PV on the matrix cores.
//
// Stands in for the third-party calls of SageSLA/core.py:102-144 of the reference
// (spas_sage_attn get_vanilla_qk_quant, block_map_lut_triton, transpose_pad_permute_cuda,
// scale_fuse_quant_cuda, qk_int8_sv_f8_*): that extension is not part of the reference tree,
// so the scheme below follows its published description, not its code:
//   q_int8 = rint(q / sq), sq = max|q| / 127 over each block of BLKQ rows;
//   k_int8 = rint((k - mean_L k) / sk), sk per block of BLKK rows;
//   v_fp8  = e4m3(v / sv), sv[d] = max_L |v[:, d]| / v_range (448 by default; the reference's call passes 2.25);
//   S = (q_int8 . k_int8) * sq * sk * scale ; P = softmax numerators over the selected blocks ;
//   O = (e4m3(c P) . v_fp8) * sv / sum(e4m3(c P)), c = 112 with P <= 4 (reference maximum lagging by <= 2).
// The look-up table of the bf16 path is used as is (no delta encoding is needed here).
#include <type_traits>
#include "block_map.h"
#include "block_select.h"
#include "common.h"
#include "linear_state.h"
#include "sage_steps.h"

namespace sla {

int64_t k_colmean_scratch_floats(int BH, int L, int D);
int64_t linear_fwd_workspace_bytes(int BH, int L, int D);
void launch_k_colmean(const void* k, const RowLayout& lay, int dtype, int BH, int L, int D, float* scratch, void* colmean,
                      hipStream_t st);
void launch_map_from_pooled(int dtype, const void* pq, const void* pk, void* score, int BH, int M, int N, int D, int topk,
                            int8_t* sparse_map, void* lut, int lut64, hipStream_t st);

// ---- INT8 block quantisation ----------------------------------------------------------------
// One workgroup per (block, bh).  SUB_MEAN: subtract the column mean of the head (`colmean`: its D means) first.
// POOL: also write the block mean the mask builder needs (of x, or of x - colmean rounded to 16 bit, as
// get_block_map pools it: utils.py:55-58 of the reference), summed row by row in fp32 and divided once,
// exactly as the pooling kernel of the mask builder does, so the block is read from memory once for both.
template <int D, int BLK, bool POOL>
constexpr int quant_int8_lds() { return 16 + (POOL ? BLK * (D + 8) * 2 : 0); }       // bytes
// (tid: this thread among the 256 of the block; a workgroup may hold several blocks, of which some are not `active`)
template <typename Tag, int D, int BLK, bool SUB_MEAN, bool POOL>
static __device__ __forceinline__ void quant_int8_body(const uint16_t* __restrict__ x, const RowLayout lay,
                                                       const uint16_t* __restrict__ colmean, int8_t* __restrict__ xq,
                                                       float* __restrict__ scale, uint16_t* __restrict__ pooled, int L,
                                                       int nblk, int tiled, int blk, int bh, int tid, bool active, char* smem) {
  using E = Elem<Tag>;
  constexpr int CPR = D / 8;
  constexpr int RPP = 256 / CPR;
  constexpr int NP = BLK / RPP;
  constexpr int TSTR = D + 8;
  float* const sred = reinterpret_cast<float*>(smem);
  uint16_t* const tile = reinterpret_cast<uint16_t*>(smem + 16);
  if (!active) blk = nblk;                 // (every row of it lies past the end)
  const int lrow = tid / CPR, lcol = (tid % CPR) * 8;
  float cm[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) cm[e] = 0.f;
  if (SUB_MEAN) {
    const i16x8_t m = *reinterpret_cast<const i16x8_t*>(colmean + lcol);
#pragma unroll
    for (int e = 0; e < 8; ++e) cm[e] = E::to_float((uint16_t)m[e]);
  }
  // every row of the block is asked for before the first is used (rows past L lie outside the descriptor and read as
  // zero): one memory latency per block instead of one per row group
  const __amdgpu_buffer_rsrc_t xb = make_rsrc(x + lay.head(bh), lay.head_range_bytes(L, D));
  i16x8_t raw[NP];
#pragma unroll
  for (int p = 0; p < NP; ++p)
    raw[p] = buf_load_b128(xb, (uint32_t)(blk * BLK + lrow + p * RPP) * (uint32_t)(lay.sl * 2) + (uint32_t)lcol * 2u);
  float val[NP][8];
  float amax = 0.f;
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const int grow = blk * BLK + lrow + p * RPP;
    i16x8_t v = raw[p];
    const bool ok = grow < L;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      val[p][e] = ok ? E::to_float((uint16_t)v[e]) - cm[e] : 0.f;
      amax = fmaxf(amax, fabsf(val[p][e]));
    }
    if (POOL) {
      if (SUB_MEAN) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = (short)E::from_float(val[p][e]);
      }
      *reinterpret_cast<i16x8_t*>(&tile[(lrow + p * RPP) * TSTR + lcol]) = v;
    }
  }
#pragma unroll
  for (int s = 1; s < 64; s <<= 1) amax = fmaxf(amax, __shfl_xor(amax, s));
  if ((tid & 63) == 0) sred[tid >> 6] = amax;
  __syncthreads();
  if (!active) return;
  amax = fmaxf(fmaxf(sred[0], sred[1]), fmaxf(sred[2], sred[3]));
  const float sc = fmaxf(amax, 1e-30f) / 127.0f;
  if (tid == 0) scale[(size_t)bh * nblk + blk] = sc;
  const float inv_sc = 1.0f / sc;
  if (POOL && tid < D) {   // one column per thread (the barrier above also covers the tile)
    const int nrows = min(BLK, L - blk * BLK);
    float acc = 0.f;
    // rows are read sixteen at a time (all reads of a batch in flight together), then added in row order
    constexpr int BATCH = 16;
    int r = 0;
    for (; r + BATCH <= nrows; r += BATCH) {
      uint16_t t[BATCH];
#pragma unroll
      for (int i = 0; i < BATCH; ++i) t[i] = tile[(r + i) * TSTR + tid];
#pragma unroll
      for (int i = 0; i < BATCH; ++i) acc = acc + E::to_float(t[i]);
    }
    for (; r < nrows; ++r) acc = acc + E::to_float(tile[r * TSTR + tid]);
    pooled[tiled ? tiled_head(bh, nblk, D) + tiled_pos(blk, tid, D) : ((size_t)bh * nblk + blk) * D + tid] =
        E::from_float(acc / (float)nrows);
  }
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const int grow = blk * BLK + lrow + p * RPP;
    if (grow >= L) continue;
    i32x2_t w;
    int8_t* b = reinterpret_cast<int8_t*>(&w);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      // round(val / sc) through the reciprocal: the product is within two units in the last place of the quotient
      // (< 3e-5 for |quotient| <= 127), so both round to the same integer unless the product lies that close to a
      // half-integer; those few elements take the division itself.
      const float t = val[p][e] * inv_sc;
      float r = rintf(t);
      if (fabsf(t - r) > 0.4999f) r = rintf(val[p][e] / sc);
      r = fminf(fmaxf(r, -127.f), 127.f);
      b[e] = (int8_t)(int)r;
    }
    *reinterpret_cast<i32x2_t*>(xq + ((size_t)bh * L + grow) * D + lcol) = w;
  }
}

template <typename Tag, int D, int BLK, bool SUB_MEAN, bool POOL>
__global__ __launch_bounds__(256) void quant_int8_kernel(const uint16_t* __restrict__ x, const RowLayout lay,
                                                         const uint16_t* __restrict__ colmean, int8_t* __restrict__ xq,
                                                         float* __restrict__ scale, uint16_t* __restrict__ pooled, int L,
                                                         int nblk, int tiled) {
  __shared__ __attribute__((aligned(16))) char smem[quant_int8_lds<D, BLK, POOL>()];
  quant_int8_body<Tag, D, BLK, SUB_MEAN, POOL>(x, lay, SUB_MEAN ? colmean + (size_t)blockIdx.y * D : nullptr, xq, scale, pooled, L, nblk, tiled, blockIdx.x, blockIdx.y,
                                               threadIdx.x, true, smem);
}

// ---- FP8 per-channel quantisation of V ------------------------------------------------------
// pass 1: per (chunk of 256 rows, bh) column abs-max -> partial; pass 2: reduce partials;
// pass 3: v_fp8 = e4m3(v / scale).
template <typename Tag, int D>
__global__ __launch_bounds__(256) void v_amax_partial_kernel(const uint16_t* __restrict__ v, const RowLayout lay,
                                                             float* __restrict__ part, int L, int rows_per_chunk) {
  using E = Elem<Tag>;
  constexpr int CPR = D / 8;
  constexpr int RPP = 256 / CPR;
  __shared__ float sm[RPP][D];
  const int chunk = blockIdx.x, bh = blockIdx.y, nchunk = gridDim.x;
  const int tid = threadIdx.x;
  const int lrow = tid / CPR, lcol = (tid % CPR) * 8;
  const int r_end = min(L, (chunk + 1) * rows_per_chunk);
  float am[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) am[e] = 0.f;
  for (int row = chunk * rows_per_chunk + lrow; row < r_end; row += RPP) {
    const i16x8_t x = *reinterpret_cast<const i16x8_t*>(v + lay.head(bh) + (size_t)row * (size_t)lay.sl + lcol);
#pragma unroll
    for (int e = 0; e < 8; ++e) am[e] = fmaxf(am[e], fabsf(E::to_float((uint16_t)x[e])));
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) sm[lrow][lcol + e] = am[e];
  __syncthreads();
  if (tid < D) {
    float a = 0.f;
#pragma unroll
    for (int r = 0; r < RPP; ++r) a = fmaxf(a, sm[r][tid]);
    part[((size_t)bh * nchunk + chunk) * D + tid] = a;
  }
}

// D / 16 workgroups of 256 threads per head: thread (cg, c) = (tid / 16, tid % 16) takes the maximum of column 16 bx + c
// over chunks cg, cg + 16, ...; the 16 partial maxima per column meet in LDS.
static __device__ __forceinline__ void v_scale_body(const float* __restrict__ part, float* __restrict__ v_scale, int nchunk, int D,
                                                    float v_range, int bx, int bh, float* sm) {
  const int tid = threadIdx.x;
  const int d = bx * 16 + (tid & 15), cg = tid >> 4;
  float a = 0.f;
  for (int c = cg; c < nchunk; c += 16) a = fmaxf(a, part[((size_t)bh * nchunk + c) * D + d]);
  sm[tid] = a;
  __syncthreads();
  if (tid < 16) {
    for (int j = 1; j < 16; ++j) a = fmaxf(a, sm[j * 16 + tid]);
    v_scale[(size_t)bh * D + d] = fmaxf(a, 1e-30f) / v_range;
  }
}
__global__ __launch_bounds__(256) void v_scale_kernel(const float* __restrict__ part, float* __restrict__ v_scale, int nchunk,
                                                     int D, float v_range) {
  __shared__ float sm[256];
  v_scale_body(part, v_scale, nchunk, D, v_range, blockIdx.x, blockIdx.y, sm);
}

static __device__ __forceinline__ uint32_t cvt4_fp8(float a, float b, float c, float d) {
  int w = __builtin_amdgcn_cvt_pk_fp8_f32(a, b, __float_as_int(a), false);      // (the upper half is written next: any value will do)
  w = __builtin_amdgcn_cvt_pk_fp8_f32(c, d, w, true);
  return (uint32_t)w;
}

template <typename Tag, int D>
__global__ __launch_bounds__(256) void v_quant_fp8_kernel(const uint16_t* __restrict__ v, const RowLayout lay,
                                                          const float* __restrict__ v_scale, uint8_t* __restrict__ v8, int L) {
  using E = Elem<Tag>;
  constexpr int CPR = D / 8;
  constexpr int RPP = 256 / CPR;
  const int bh = blockIdx.y;
  const int row = blockIdx.x * RPP + threadIdx.x / CPR;
  const int lcol = (threadIdx.x % CPR) * 8;
  if (row >= L) return;
  const i16x8_t x = *reinterpret_cast<const i16x8_t*>(v + lay.head(bh) + (size_t)row * (size_t)lay.sl + lcol);
  float f[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) f[e] = E::to_float((uint16_t)x[e]) / v_scale[(size_t)bh * D + lcol + e];
  i32x2_t w;
  w[0] = (int)cvt4_fp8(f[0], f[1], f[2], f[3]);
  w[1] = (int)cvt4_fp8(f[4], f[5], f[6], f[7]);
  *reinterpret_cast<i32x2_t*>(v8 + ((size_t)bh * L + row) * D + lcol) = w;
}

// ---- quantised block-sparse attention ----------------------------------------------------------
typedef __attribute__((address_space(3))) i32x2_t lds_i32x2_t;
typedef __attribute__((address_space(3))) i32x4_t lds_i32x4_t;

// One workgroup per query block of BLKQ rows, one wave per 32 queries, two waves per SIMD at head dim 128, three at 64.
// S^T = K8 Q8^T with v_mfma_i32_32x32x32_i8 (exact), dequantised by sq*sk*scale*log2(e) inside the exponent's
// FMA.  Both 32-key halves of a tile are exponentiated against one reference maximum and packed to e4m3: the
// 32 probabilities a lane then holds are, as they stand, its B operand of ONE v_mfma_f32_32x32x64_f8f6f4 per
// 32 output channels (O^T += V8^T P^T, contraction over all 64 keys of the tile); V^T fragments come from the
// row-major V tile with the transposing 8-bit LDS read, whose row addresses follow the accumulator's key order.
// The reference maximum only moves when a tile's maximum exceeds it by more than TAU = 2 (log2 units), so
// probabilities are at most 4; they are scaled by 112 = 448/4 to use the e4m3 range.
// K/V tiles go from memory straight into LDS (buffer loads with the LDS bit), in rings of three tiles each, swizzled; a tile is
// requested two steps before it is read, and there is one barrier per tile.  No registers hold tiles on their way, and the
// scores of two neighbouring tiles share three blocks of sixteen registers instead of four: head dim 64 then fits three waves
// per SIMD (with its query fragments in LDS), and the scheduling room takes nothing to scratch at 128.  Tiles through registers,
// a step ahead, into rows padded by 16 bytes, against this: 40 heads x 32760 x 128, 51 of 512 key blocks, 1616 -> 1500 us
// (sequence too long for an XCD's L2); 16 heads x 5003 x 64, 15 of 79, 640 workgroups, 40.6 -> 34.6 us, of which the third
// wave per SIMD is 6: they are one round now.
// LINEAR: the linear branch of the same rows, projection, bias and sum in the epilogue (bit for bit what the attention and
// linear_out_kernel behind it leave): the per-head state (32 KB) is read straight from L2 in operand order, as in the 16-bit
// kernel's epilogue, so that no barrier holds the other workgroup of the compute unit.  It costs this kernel 55 us at 40 heads x
// 32760 x 128, softmax map, where the launch of its own, bound by memory (o_s written and read again), took 203.  q's rows are
// loaded behind the last product: beside it they cost spills (1.66 ms for 1.62).
struct SageLinear {
  const uint16_t *q, *kvwt, *z;
  const float* bias;
  RowLayout lq, lout;
  int fmap;
};
template <int N>
using Slot = std::integral_constant<int, N>;

template <typename OutTag, int D, int BLKQ, bool LINEAR>
__global__ __launch_bounds__(BLKQ * 2) __attribute__((amdgpu_waves_per_eu(D == 64 ? 3 : 2, D == 64 ? 3 : 2))) void sage_fwd_kernel(
    const int8_t* __restrict__ q8, const float* __restrict__ q_scale, const int8_t* __restrict__ k8,
    const float* __restrict__ k_scale, const uint8_t* __restrict__ v8, const float* __restrict__ v_scale,
    const void* __restrict__ lut, int lut64, uint16_t* __restrict__ o, int L, int Mblk, int Nblk, int topk,
    float scale_log2e, int total, const SageLinear lin) {
  using EO = Elem<OutTag>;
  constexpr int BLKK = 64;
  constexpr int NT = BLKQ * 2;
  constexpr int QC = D / 32;                // 32-wide int8 contraction chunks
  constexpr int DT = D / 32;                // 32-row tiles of O^T
  constexpr int TILE = BLKK * D;            // bytes of a tile of K or of V
  constexpr int RPR = 1024 / D;             // rows of a tile that one request moves
  constexpr int CPR = D / 16;               // 16-byte pieces per row
  constexpr int NR = TILE / 1024 / (NT / 64);      // requests per wave and tile
  constexpr int NS = 3;                     // tiles of either matrix in LDS
  static_assert(NT == 256 && NR >= 1, "four waves share a tile's requests");
  constexpr float TAU = 2.0f;
  // probabilities are scaled by 112 = 448 / 2^TAU, applied as an offset of the exponent
  constexpr float LOG2_P_SCALE = 6.807354922057604f;

  constexpr bool Q_LDS = D == 64;           // the query fragments wait in LDS, each lane's own
  constexpr int RINGS = 2 * NS * TILE;      // K and V of tile i: slot i % NS of either ring
  __shared__ __attribute__((aligned(1024))) uint8_t smem[RINGS + (Q_LDS ? NT * QC * 16 : 0)];
  uint8_t* const sK = smem;
  uint8_t* const sV = smem + NS * TILE;

  const int logical = xcd_remap(blockIdx.x, gridDim.x, total);
  if (logical < 0) return;
  const int bh = logical / Mblk;
  const int mb = logical - bh * Mblk;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int lane = tid & 63, g = lane >> 5, r = lane & 31;

  const size_t head_off = first_lane64((size_t)bh * L * D);
  const uint32_t head_bytes = (uint32_t)L * D;
  const __amdgpu_buffer_rsrc_t qh = make_rsrc(q8 + head_off, head_bytes);
  const __amdgpu_buffer_rsrc_t kh = make_rsrc(k8 + head_off, head_bytes);
  const __amdgpu_buffer_rsrc_t vh = make_rsrc(v8 + head_off, head_bytes);
  int qrow = mb * BLKQ + wave * 32 + r;
  i32x4_t qf[QC];
#pragma unroll
  for (int c = 0; c < QC; ++c)
    qf[c] = __builtin_bit_cast(i32x4_t, buf_load_b128(qh, (uint32_t)qrow * D + 32 * c + 16 * g));   // rows past L: 0
  const float qs = q_scale[(size_t)bh * Mblk + mb] * scale_log2e;
  const float* ksc = k_scale + (size_t)bh * Nblk;

  const size_t lut_row = ((size_t)bh * Mblk + mb) * topk;
  // 64 entries of the list at a time in the wave's lanes, with the tiles' dequantisation factors (as scalar loads, two per
  // tile, they share their counter with the LDS reads: 1 % of the kernel).
  int list_nb = 0;
  float list_sc = 0.f;
  auto entry = [&](int i, float& sc) -> int {                  // (i ascending by one)
    if ((i & 63) == 0) {
      const int at = min(i + lane, topk - 1);
      list_nb = lut64 ? (int)reinterpret_cast<const long long*>(lut)[lut_row + at] : reinterpret_cast<const int*>(lut)[lut_row + at];
      // an all-zero block has scale 1e-30/127; the floor keeps -inf * sc = -inf (never NaN) for masked rows
      list_sc = fmaxf(qs * ksc[list_nb], 1e-37f);
    }
    sc = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(list_sc), i & 63));
    return __builtin_amdgcn_readlane(list_nb, i & 63);
  };
  // The 16-byte pieces of a row are exchanged: piece p of row r lies in slot p ^ swz(r).  16 adjacent rows of one piece (a
  // row-wise read) then hit 16 different slots of the 256 bytes LDS serves at a time, and so do the eight rows of 32 bytes
  // of a transposing read (keys 0..3 and 8..11, or 4..7 and 12..15).
  const auto swz = [](int row) __attribute__((always_inline)) {
    return D == 128 ? ((row >> 2) & 1) | (row & 2) | ((row >> 1) & 4) : (row >> 2) & 3;
  };
  // A request moves RPR rows, 64 lanes x 16 bytes; this wave's are NR wave + 0 .. NR - 1 of a tile.
  uint32_t req_off[NR];
#pragma unroll
  for (int j = 0; j < NR; ++j) {
    const int row = (NR * wave + j) * RPR + lane / CPR;
    req_off[j] = (uint32_t)row * D + (uint32_t)((lane % CPR) ^ swz(row)) * 16;
  }
  const uint32_t req_lds = __builtin_amdgcn_readfirstlane((uint32_t)(size_t)smem + (uint32_t)(NR * wave) * 1024);
  // (rows past L touch neither memory nor LDS; between a scalar write of M0 and the load that reads it the hardware wants a wait state)
  auto request = [&](int which, int row0, int slot) __attribute__((always_inline)) {      // 0 K, 1 V
    const uint32_t at = (uint32_t)row0 * D;
#pragma unroll
    for (int j = 0; j < NR; ++j)
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(
                       req_lds + (uint32_t)((which * NS + slot) * TILE + j * 1024)),
                   "v"(req_off[j] + at), "s"(which ? vh : kh)
                   : "memory");
  };
  const int row_none = (L + 63) & ~63;     // past every head
  // (rows of the ragged last block are never written: what LDS holds in their place has to be finite, as their probabilities are 0)
  if (L % BLKK) {
#pragma unroll
    for (int i = 0; i < NS * TILE / 16 / NT; ++i) reinterpret_cast<i32x4_t*>(sV)[i * NT + tid] = i32x4_t{0, 0, 0, 0};
    lds_barrier();
  }

  f32x16_t oacc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) oacc[dt][i] = 0.f;
  float m_used = -INFINITY;   // reference maximum (log2 units)
  // Row sums of the e4m3 probabilities come from the matrix core as well: an A operand of ones makes every
  // row of this accumulator the sum over all 64 keys of a tile, so each lane holds l of its query column
  // (numerator and denominator then see the same rounded probabilities, and no vector-ALU adds are spent).
  f32x16_t lacc;
#pragma unroll
  for (int i = 0; i < 16; ++i) lacc[i] = 0.f;
  const i32x8_t ones = {0x22222222, 0x22222222, 0x22222222, 0x22222222, 0, 0, 0, 0};   // e2m1 1.0, 32 of them in four registers

  // transposed 8-bit read: lane i of a 16-lane group passes the address of (row i/2, 8 bytes at
  // column 8*(i%2)) and receives column i of the 8x16 tile.  Row i/2 is mapped to the key that
  // accumulator slot i/2 of the probabilities holds: keys 4g+{0..3} and 8+4g+{0..3} of a 16-key chunk.
  const int li = lane & 15;
  const int slot = li >> 1;
  const int tr_key = 8 * (slot >> 2) + 4 * g + (slot & 3);
  // a lane's places in a tile: row-wise, row r, piece 2 c + g (32 rows on, the same piece); transposed, row tr_key, 8 bytes of
  // piece 2 dt + (lane / 16) % 2 (16 rows on, the same piece)
  uint32_t q_at = (uint32_t)(size_t)smem + RINGS + wave * (QC * 1024) + lane * 16;
  if constexpr (Q_LDS) {
#pragma unroll
    for (int c = 0; c < QC; ++c) *(lds_i32x4_t*)(size_t)(q_at + (uint32_t)(c * 1024)) = qf[c];
    asm volatile("" : "+v"(q_at)::"memory");
  }
  uint32_t kp[QC], vp[DT];
#pragma unroll
  for (int c = 0; c < QC; ++c) {
    kp[c] = (uint32_t)(size_t)sK + r * D + ((2 * c + g) ^ swz(r)) * 16;
    asm volatile("" : "+v"(kp[c]));
  }
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) {
    vp[dt] = (uint32_t)(size_t)sV + tr_key * D + ((2 * dt + ((lane >> 4) & 1)) ^ swz(tr_key)) * 16 + 8 * (li & 1);
    asm volatile("" : "+v"(vp[dt]));
  }

  // The integer products start from the bit pattern of the float 1.5 * 2^23 instead of from zero: the integer
  // MAGIC + s, read as a float, IS the float 12582912 + s (|s| <= 128 * 127^2 < 2^22 stays inside the binade whose
  // unit in the last place is 1), so the scores reach the exponent's multiply-add without an int -> float
  // conversion per element; 12582912 * sc joins the constant that multiply-add subtracts.
  constexpr int MAGIC = 0x4B400000;
  constexpr float MAGIC_F = 12582912.0f;
  i32x16_t magic;
#pragma unroll
  for (int i = 0; i < 16; ++i) magic[i] = MAGIC;
  asm volatile("" : "+v"(magic));           // (kept, not formed again for every tile)
  // S^T of one 32-key half of a tile: MAGIC + raw int32 products
  auto scores = [&](int kslot, int t, i32x16_t& acc) __attribute__((always_inline)) {
#pragma unroll
    for (int c = 0; c < QC; ++c) {
      const i32x4_t a = *(lds_i32x4_t*)(size_t)(kp[c] + (uint32_t)(kslot * TILE + 32 * t * D));
      const i32x4_t b = Q_LDS ? *(lds_i32x4_t*)(size_t)(q_at + (uint32_t)(c * 1024)) : qf[c];
      acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, c == 0 ? magic : acc, 0, 0, 0);
    }
  };
  // ragged last key block (kv_valid existing key rows): missing rows take no part
  // (the lane's number formed again where it is rarely wanted, instead of kept through the loop)
  const auto lane_again = [&]() __attribute__((always_inline)) {
    int ones32 = -1;
    asm volatile("" : "+s"(ones32));
    return (int)__builtin_amdgcn_mbcnt_hi(ones32, __builtin_amdgcn_mbcnt_lo(ones32, 0));
  };
  auto mask = [&](i32x16_t& acc, int t, int kv_valid) __attribute__((always_inline)) {
    const int lim = kv_valid - (lane_again() >> 5) * 4;      // key index of register i is 32t + 8(i/4) + i%4 + 4g
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      int s = 32 * t + 8 * (i >> 2) + (i & 3) >= lim ? (int)0xff800000u : acc[i];      // -inf
      asm volatile("" : "+v"(s));         // (in place)
      acc[i] = s;
    }
  };
  // raw maximum of this lane's 32 scores (sc > 0, so the maximum commutes with the scaling)
  auto maximum = [&](const i32x16_t& acc0, const i32x16_t& acc1) __attribute__((always_inline)) {
    float mx = __int_as_float(acc0[0]);                                                // = 12582912 + score
#pragma unroll
    for (int i = 0; i < 16; ++i) mx = fmaxf(mx, __int_as_float(acc0[i]));
#pragma unroll
    for (int i = 0; i < 16; ++i) mx = fmaxf(mx, __int_as_float(acc1[i]));
    return mx - MAGIC_F;                   // (exact: both are integers below 2^24)
  };
  // rare: moves the reference and rescales what is accumulated
  auto raise_reference = [&](float mx, float sc) __attribute__((always_inline)) {
    if (__any(mx * sc > m_used + TAU)) {
      float m_new = fmaxf(mx, __shfl_xor(mx, 32)) * sc;
      m_new = fmaxf(m_used, m_new);
      const float f = fast_exp2(m_used - m_new);     // 0 on the first tile
      m_used = m_new;
#pragma unroll
      for (int i = 0; i < 16; ++i) lacc[i] *= f;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) oacc[dt][i] *= f;
    }
  };
  // softmax numerators of half t of a tile (scores acc, dequantisation factor sc), packed to e4m3 in the B-operand order of the
  // 64-key product: 112 p = exp2(s*sc - (m_used - log2 112)); -inf scores give exactly 0
  auto probabilities = [&](const i32x16_t& acc, int t, float sc, float m_off, i32x8_t& pb) __attribute__((always_inline)) {
#pragma unroll
    for (int i4 = 0; i4 < 4; ++i4) {
      float pv[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) pv[j] = fast_exp2(__builtin_fmaf(__int_as_float(acc[4 * i4 + j]), sc, -m_off));
      pb[4 * t + i4] = (int)cvt4_fp8(pv[0], pv[1], pv[2], pv[3]);
    }
  };
  const auto offset = [&](float sc) __attribute__((always_inline)) { return __builtin_fmaf(MAGIC_F, sc, m_used - LOG2_P_SCALE); };
  // l += sum_keys P ; O^T += V8^T P^T: one 64-key product per 32 output channels
  auto accumulate = [&](int vslot, const i32x8_t& pb) __attribute__((always_inline)) {
    // formats 0 = e4m3, 4 = e2m1, block scales 2^0
    lacc = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(ones, pb, lacc, 4, 0, 0, 0x7f7f7f7f, 0, 0x7f7f7f7f);
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      i32x8_t a;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int c2 = 0; c2 < 2; ++c2) {
          const i32x2_t x = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_i32x2_t*)(size_t)(vp[dt] + (uint32_t)(vslot * TILE + (32 * t + 16 * c2) * D)));
          a[4 * t + 2 * c2] = x[0];
          a[4 * t + 2 * c2 + 1] = x[1];
        }
      oacc[dt] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a, pb, oacc[dt], 0, 0, 0, 0x7f7f7f7f, 0, 0x7f7f7f7f);
    }
  };

  // Software pipeline over the selected tiles: step i issues the int8 products of tile i beside the exponentials of tile i-1,
  // then the fp8 products of tile i-1 beside the maxima of tile i; between the two only the rare branches.  Bound by the vector
  // ALU (63 % of the cycles at 40 heads x 32760 x 128, the matrix cores 40; at a tile a step ahead 60 and 35).
  int key0 = 0, key1 = 0;                   // first keys of this step's tile and of the next
  float sc = 0.f, sc1 = 0.f, sc_prev = 0.f, mx_prev = 0.f;
  // the scores of a tile's halves: those of the tile before (p0, p1) are used up half by half, the second of this tile takes p0's place
  i32x16_t acc_a, acc_b, acc_c;
  auto step = [&](int it, auto slot, i32x16_t& acc, i32x16_t& p0, const i32x16_t& p1, auto first) __attribute__((always_inline)) {
    constexpr int S = decltype(slot)::value;
    // (both slots were used up in the step before; past the list's end a request moves nothing, so that the count below holds)
    int key2 = row_none;
    float sc2 = 0.f;
    if (it + 2 < topk) key2 = entry(it + 2, sc2) * BLKK;
    request(0, key2, (S + 2) % NS);
    request(1, key1, (S + 1) % NS);
    i32x8_t pb;
    if constexpr (first) {
      scores(S, 0, acc);
      scores(S, 1, p0);
    } else {
      raise_reference(mx_prev, sc_prev);
      const float m_off = offset(sc_prev);
      __builtin_amdgcn_sched_barrier(0);
      scores(S, 0, acc);
      probabilities(p0, 0, sc_prev, m_off, pb);
      if (D == 64) __builtin_amdgcn_sched_barrier(0);
      scores(S, 1, p0);
      probabilities(p1, 1, sc_prev, m_off, pb);
      if constexpr (D == 128) {
        // (the first fragments' way from LDS is covered by exponentials, the other ones are read a half ahead)
        __builtin_amdgcn_sched_group_barrier(0x100, QC, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, 12, 0);
#pragma unroll
        for (int c = 0; c < 2 * QC; ++c) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          if (c < QC) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x002, 9, 0);
        }
      }
      asm volatile("" :: "v"(pb));          // (formed here, not where the products below read them)
      __builtin_amdgcn_sched_barrier(0);
    }
    if (L - key0 < BLKK) {
      mask(acc, 0, L - key0);
      mask(p0, 1, L - key0);
    }
    if constexpr (!first) {
      __builtin_amdgcn_sched_barrier(0);
      accumulate((S + 2) % NS, pb);
    }
    mx_prev = maximum(acc, p0);
    sc_prev = sc;
    sc = sc1;
    sc1 = sc2;
    key0 = key1;
    key1 = key2;
    // the next step's tiles visible (only the requests above may still be out), this step's consumed
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(2 * NR) : "memory");
  };
  int it = 0;
  if (topk > 0) {
    key0 = entry(0, sc) * BLKK;
    request(0, key0, 0);
    key1 = row_none;
    if (topk > 1) key1 = entry(1, sc1) * BLKK;
    request(1, key0, 0);
    request(0, key1, 1);
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(2 * NR) : "memory");
    step(0, Slot<0>{}, acc_a, acc_b, acc_c, std::true_type{});
    for (it = 1; it + 2 < topk; it += 3) {
      step(it, Slot<1>{}, acc_c, acc_a, acc_b, std::false_type{});
      step(it + 1, Slot<2>{}, acc_b, acc_c, acc_a, std::false_type{});
      step(it + 2, Slot<0>{}, acc_a, acc_b, acc_c, std::false_type{});
    }
  }
  const auto last = [&](const i32x16_t& p0, const i32x16_t& p1, auto slot) __attribute__((always_inline)) {
    i32x8_t pb;
    raise_reference(mx_prev, sc_prev);
    const float m_off = offset(sc_prev);
    probabilities(p0, 0, sc_prev, m_off, pb);
    probabilities(p1, 1, sc_prev, m_off, pb);
    accumulate(decltype(slot)::value, pb);
  };
  constexpr int DC = D / 16;
  i16x8_t xq[DC];                          // q as it is: this lane holds d = 16c + 8g + j of its row
  const auto fetch_q = [&]() __attribute__((always_inline)) {
    if constexpr (LINEAR) {
      const uint16_t* p = lin.q + lin.lq.head(bh) + (size_t)min(qrow, L - 1) * (size_t)lin.lq.sl + 8 * g;
#pragma unroll
      for (int c = 0; c < DC; ++c) xq[c] = *reinterpret_cast<const i16x8_t*>(p + 16 * c);
    }
  };
  // up to two steps are left; the last tile's probabilities and products
  if (it < topk) {
    step(it, Slot<1>{}, acc_c, acc_a, acc_b, std::false_type{});
    if (it + 1 < topk) {
      step(it + 1, Slot<2>{}, acc_b, acc_c, acc_a, std::false_type{});
      last(acc_b, acc_c, Slot<2>{});
    } else {
      last(acc_c, acc_a, Slot<1>{});
    }
  } else if (topk > 0) {
    last(acc_a, acc_b, Slot<0>{});
  }
  lane = lane_again();
  g = lane >> 5;
  r = lane & 31;
  qrow = mb * BLKQ + wave * 32 + r;
  fetch_q();
  const float inv = 1.0f / lacc[0];        // P_SCALE cancels: numerator and l carry the same factor
  // The rounded rows go through LDS (every wave is done with the tiles) and leave as whole rows in streaming stores:
  // they are not read again here, and what does not stay behind as modified lines in L2 need not be written back when
  // the kernel ends.
  __syncthreads();
  {
    constexpr int SSTR = TileRows<D>::SSTR;
    static_assert(4 * 32 * SSTR * 2 <= (int)sizeof(smem), "staging tiles of four waves");
    uint16_t* const stage = reinterpret_cast<uint16_t*>(smem) + wave * (32 * SSTR);
    const float* vs = v_scale + (size_t)bh * D;
    const int row0 = mb * BLKQ + wave * 32;
    // the attention's values of registers 4 i4 .. of tile dt, in 16 bit
    const auto attention = [&](int dt, int i4) __attribute__((always_inline)) -> i32x2_t {
      const f32x4_t sv = *reinterpret_cast<const f32x4_t*>(vs + 32 * dt + 8 * i4 + 4 * g);
      i32x2_t w;
      w[0] = (int)EO::pack2(oacc[dt][4 * i4 + 0] * inv * sv[0], oacc[dt][4 * i4 + 1] * inv * sv[1]);
      w[1] = (int)EO::pack2(oacc[dt][4 * i4 + 2] * inv * sv[2], oacc[dt][4 * i4 + 3] * inv * sv[3]);
      return w;
    };
    if constexpr (!LINEAR) {
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int i4 = 0; i4 < 4; ++i4)
          *reinterpret_cast<i32x2_t*>(&stage[r * SSTR + 32 * dt + 8 * i4 + 4 * g]) = attention(dt, i4);
    } else {
      const uint16_t* const state = lin.kvwt + (size_t)bh * D * D;
      const uint16_t* const z = lin.z + (size_t)bh * D;
      i16x8_t zc[DC];
#pragma unroll
      for (int c = 0; c < DC; ++c) zc[c] = *reinterpret_cast<const i16x8_t*>(z + 16 * c + 8 * g);
      i16x8_t fq[DC];
      float den = phi_pack_den<OutTag, DC>(lin.fmap, xq, fq, [&](int c, int j) { return EO::to_float((uint16_t)zc[c][j]); });
      den += __shfl_xor(den, 32);
      den = round16<OutTag>(1e-5f + round16<OutTag>(den));
      const float inv_den = 1.0f / den;
#pragma unroll
      for (int et = 0; et < DT; ++et) {
        i16x8_t a[DC];
#pragma unroll
        for (int c = 0; c < DC; ++c) a[c] = *reinterpret_cast<const i16x8_t*>(state + (size_t)(32 * et + r) * D + 16 * c + 8 * g);
        f32x16_t acc;
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[i] = 0.f;
#pragma unroll
        for (int c = 0; c < DC; ++c) acc = EO::mfma32(a[c], fq[c], acc);
#pragma unroll
        for (int i4 = 0; i4 < 4; ++i4) {
          const int e0 = 32 * et + 8 * i4 + 4 * g;
          const i32x2_t o_s = attention(et, i4);
          i32x2_t w;
#pragma unroll
          for (int h = 0; h < 2; ++h) {    // (both summands in 16 bit, one rounded sum, as tensors)
            const uint32_t x = (uint32_t)o_s[h];
            float l[2];
#pragma unroll
            for (int j = 0; j < 2; ++j)
              l[j] = round16<OutTag>(pin_f32(__builtin_fmaf(acc[4 * i4 + 2 * h + j], inv_den, round16<OutTag>(lin.bias[e0 + 2 * h + j]))));
            w[h] = (int)EO::pack2(EO::to_float((uint16_t)(x & 0xffff)) + l[0], EO::to_float((uint16_t)(x >> 16)) + l[1]);
          }
          *reinterpret_cast<i32x2_t*>(&stage[r * SSTR + e0]) = w;
        }
      }
    }
    wave_lds_fence();
    TileRows<D> t;
    t.unpark(stage, lane);
    const size_t pitch = LINEAR ? (size_t)lin.lout.sl : (size_t)D;
    t.store_streaming(o + (LINEAR ? lin.lout.head(bh) : head_off) + (size_t)row0 * pitch, L - row0, lane, pitch);
  }
}

// ---- host -------------------------------------------------------------------------------------
struct SageWs {
  int nchunk_v, rows_per_chunk_v;
  size_t chunk_sums, colmean, v_part, total;
};
static SageWs sage_ws(int BH, int L, int D) {
  SageWs w;
  w.rows_per_chunk_v = 256;
  w.nchunk_v = cdiv(L, w.rows_per_chunk_v);
  size_t off = 0;
  w.chunk_sums = off; off += align_up(k_colmean_scratch_floats(BH, L, D) * 4, 256);
  w.colmean = off;    off += align_up((int64_t)BH * D * 2, 256);
  w.v_part = off;     off += align_up((int64_t)BH * w.nchunk_v * D * 4, 256);
  w.total = off;
  return w;
}
int64_t sage_quant_workspace_bytes(int BH, int L, int D) { return (int64_t)sage_ws(BH, L, D).total; }

// workspace of the one-call preparation: the quantisers' workspace, then block means and scores
struct SagePrepWs {
  size_t pq, pk, score, total;
};
static SagePrepWs sage_prep_ws(int BH, int L, int D) {
  const int64_t M = cdiv(L, 128), N = cdiv(L, 64);
  SagePrepWs w;
  size_t off = sage_ws(BH, L, D).total;
  w.pq = off;    off += align_up((int64_t)BH * align_up(M, 32) * D * 2, 256);      // (whole tiles of 32)
  w.pk = off;    off += align_up((int64_t)BH * align_up(N, 32) * D * 2, 256);
  w.score = off; off += scores_in_memory((int)N, D) ? align_up((int64_t)BH * M * N * 2, 256) : 0;
  w.total = off;
  return w;
}
int64_t sage_prepare_workspace_bytes(int BH, int L, int D) { return (int64_t)sage_prep_ws(BH, L, D).total; }

static int validate_sage(int dtype, int B, int H, int L, int D, int BLKQ, int BLKK) {
  SLA_REQUIRE(B > 0 && H > 0 && L > 0, SLA_ERR_BAD_ARG, "non-positive size (B=%d H=%d L=%d)", B, H, L);
  SLA_REQUIRE((int64_t)B * H <= 65535, SLA_ERR_UNSUPPORTED, "B*H exceeds 65535");
  SLA_REQUIRE(dtype == SLA_BF16 || dtype == SLA_F16, SLA_ERR_UNSUPPORTED, "SageSLA takes bf16 or f16, got dtype %d", dtype);
  SLA_REQUIRE(D == 64 || D == 128, SLA_ERR_UNSUPPORTED, "headdim should be in [64, 128], got %d", D);
  SLA_REQUIRE(BLKQ == 128 && BLKK == 64, SLA_ERR_UNSUPPORTED, "SageSLA only supports BLKQ=128 and BLKK=64, got %d/%d", BLKQ,
              BLKK);
  return SLA_OK;
}

// range of the e4m3 values v is quantised to: the format's largest finite value (448) or less
int validate_v_range(float v_range) {
  SLA_REQUIRE(v_range > 0.f && v_range <= 448.f, SLA_ERR_BAD_ARG, "v_range=%g outside (0, 448]", (double)v_range);
  return SLA_OK;
}

template <typename Tag, int D>
static int quant_qk_impl(const void* q, const void* k, int dtype, int BH, int L, int8_t* q8, float* qs, int8_t* k8,
                         float* ks, char* ws, hipStream_t st) {
  const SageWs w = sage_ws(BH, L, D);
  const int M = cdiv(L, 128), N = cdiv(L, 64);
  const RowLayout lay = contiguous_layout(BH, L, D);
  launch_k_colmean(k, lay, dtype, BH, L, D, (float*)(ws + w.chunk_sums), ws + w.colmean, st);
  hipLaunchKernelGGL((quant_int8_kernel<Tag, D, 128, false, false>), dim3(M, BH), dim3(256), 0, st, (const uint16_t*)q, lay,
                     nullptr, q8, qs, nullptr, L, M, 0);
  hipLaunchKernelGGL((quant_int8_kernel<Tag, D, 64, true, false>), dim3(N, BH), dim3(256), 0, st, (const uint16_t*)k, lay,
                     (const uint16_t*)(ws + w.colmean), k8, ks, nullptr, L, N, 0);
  return check_launch("sage_quant_qk");
}

// Mask, INT8 q/k and FP8 v in one pass structure: the column mean of k is formed once (the mask builder
// and the quantiser both subtract it) and the quantisers emit the block means the scores are made of, so
// q is read once and k twice instead of q twice and k four times.
template <typename Tag, int D>
static int quant_v_impl(const void* v, const RowLayout& lay, int BH, int L, uint8_t* v8, float* vs, float v_range, char* ws,
                        hipStream_t st);

// (lay: where the rows of q, k, v lie; the quantised outputs are always contiguous (B, H, L, D))
template <typename Tag, int D>
static int prepare_impl(const void* q, const void* k, const void* v, const RowLayout& lay, int dtype, int BH, int L, int topk,
                        int8_t* sparse_map,
                        void* lut, int lut64, int8_t* q8, float* qs, int8_t* k8, float* ks, uint8_t* v8, float* vs, float v_range,
                        char* ws, hipStream_t st) {
  const SageWs w = sage_ws(BH, L, D);
  const SagePrepWs p = sage_prep_ws(BH, L, D);
  const int M = cdiv(L, 128), N = cdiv(L, 64);
  uint16_t* pq = (uint16_t*)(ws + p.pq);
  uint16_t* pk = (uint16_t*)(ws + p.pk);
  const int tiled = score_takes_tiled(dtype, D);
  launch_k_colmean(k, lay, dtype, BH, L, D, (float*)(ws + w.chunk_sums), ws + w.colmean, st);
  hipLaunchKernelGGL((quant_int8_kernel<Tag, D, 128, false, true>), dim3(M, BH), dim3(256), 0, st, (const uint16_t*)q, lay,
                     nullptr, q8, qs, pq, L, M, tiled);
  hipLaunchKernelGGL((quant_int8_kernel<Tag, D, 64, true, true>), dim3(N, BH), dim3(256), 0, st, (const uint16_t*)k, lay,
                     (const uint16_t*)(ws + w.colmean), k8, ks, pk, L, N, tiled);
  launch_map_from_pooled(dtype, pq, pk, ws + p.score, BH, M, N, D, topk, sparse_map, lut, lut64, st);
  int rc = check_launch("sage_prepare");
  if (rc || !v) return rc;
  return quant_v_impl<Tag, D>(v, lay, BH, L, v8, vs, v_range, ws, st);
}

template <typename Tag, int D>
static int quant_v_impl(const void* v, const RowLayout& lay, int BH, int L, uint8_t* v8, float* vs, float v_range, char* ws,
                        hipStream_t st) {
  const SageWs w = sage_ws(BH, L, D);
  float* part = (float*)(ws + w.v_part);
  hipLaunchKernelGGL((v_amax_partial_kernel<Tag, D>), dim3(w.nchunk_v, BH), dim3(256), 0, st, (const uint16_t*)v, lay, part, L,
                     w.rows_per_chunk_v);
  hipLaunchKernelGGL(v_scale_kernel, dim3(D / 16, BH), dim3(256), 0, st, part, vs, w.nchunk_v, D, v_range);
  constexpr int RPP = 256 / (D / 8);
  hipLaunchKernelGGL((v_quant_fp8_kernel<Tag, D>), dim3(cdiv(L, RPP), BH), dim3(256), 0, st, (const uint16_t*)v, lay, vs, v8,
                     L);
  return check_launch("sage_quant_v");
}

int quant_v_from_partial_amax(const void* v, const RowLayout& lay, int dtype, int BH, int L, int D, const float* part,
                              int nparts, uint8_t* v8, float* vs, float v_range, hipStream_t st) {
  hipLaunchKernelGGL(v_scale_kernel, dim3(D / 16, BH), dim3(256), 0, st, part, vs, nparts, D, v_range);
#define SAGE_VQ_CASE(TAG, DD)                                                                                         \
  hipLaunchKernelGGL((v_quant_fp8_kernel<TAG, DD>), dim3(cdiv(L, 256 / (DD / 8)), BH), dim3(256), 0, st, (const uint16_t*)v, \
                     lay, vs, v8, L)
  if (dtype == SLA_BF16) {
    if (D == 128) SAGE_VQ_CASE(bf16_tag, 128);
    else SAGE_VQ_CASE(bf16_tag, 64);
  } else {
    if (D == 128) SAGE_VQ_CASE(f16_tag, 128);
    else SAGE_VQ_CASE(f16_tag, 64);
  }
#undef SAGE_VQ_CASE
  return check_launch("linear_state_quant_v");
}

}  // namespace sla

using namespace sla;

extern "C" int sage_quant_qk(const void* q, const void* k, int dtype, int B, int H, int L, int D, int BLKQ, int BLKK,
                             int8_t* q_int8, float* q_scale, int8_t* k_int8, float* k_scale, void* workspace,
                             int64_t workspace_bytes, void* stream) {
  int rc = validate_sage(dtype, B, H, L, D, BLKQ, BLKK);
  if (rc) return rc;
  SLA_REQUIRE(q && k && q_int8 && q_scale && k_int8 && k_scale && workspace, SLA_ERR_BAD_ARG, "null pointer");
  SLA_REQUIRE(((uintptr_t)q | (uintptr_t)k | (uintptr_t)q_int8 | (uintptr_t)k_int8 | (uintptr_t)workspace) % 16 == 0,
              SLA_ERR_BAD_ARG, "pointers must be 16-byte aligned");
  const int BH = B * H;
  SLA_REQUIRE(workspace_bytes >= sage_quant_workspace_bytes(BH, L, D), SLA_ERR_WORKSPACE, "workspace too small");
  hipStream_t st = (hipStream_t)stream;
  char* ws = (char*)workspace;
  if (dtype == SLA_BF16) {
    if (D == 128) return quant_qk_impl<bf16_tag, 128>(q, k, dtype, BH, L, q_int8, q_scale, k_int8, k_scale, ws, st);
    return quant_qk_impl<bf16_tag, 64>(q, k, dtype, BH, L, q_int8, q_scale, k_int8, k_scale, ws, st);
  }
  if (D == 128) return quant_qk_impl<f16_tag, 128>(q, k, dtype, BH, L, q_int8, q_scale, k_int8, k_scale, ws, st);
  return quant_qk_impl<f16_tag, 64>(q, k, dtype, BH, L, q_int8, q_scale, k_int8, k_scale, ws, st);
}

// Everything prepare_entry asks of its arguments, for a caller that launches something else before it.
static int prepare_check(const void* q, const void* k, const void* v, const int64_t* qkv_strides, int dtype, int B, int H, int L,
                         int D, int BLKQ, int BLKK, int topk, const int8_t* sparse_map, const void* lut, int lut_elem_bytes,
                         const int8_t* q_int8, const float* q_scale, const int8_t* k_int8, const float* k_scale,
                         const uint8_t* v_fp8, const float* v_scale, float v_range, const void* workspace,
                         int64_t workspace_bytes, bool want_map, RowLayout* lay) {
  int rc = validate_sage(dtype, B, H, L, D, BLKQ, BLKK);
  if (rc) return rc;
  rc = validate_v_range(v_range);
  if (rc) return rc;
  rc = make_layout(qkv_strides, B, H, L, D, 2, lay);
  if (rc) return rc;
  const int N = cdiv(L, 64);
  SLA_REQUIRE(topk >= 0 && topk <= N, SLA_ERR_BAD_ARG, "topk=%d outside [0, %d]", topk, N);
  SLA_REQUIRE(N <= 4096, SLA_ERR_UNSUPPORTED, "more than 4096 key blocks (%d)", N);
  SLA_REQUIRE(lut_elem_bytes == 4 || lut_elem_bytes == 8, SLA_ERR_BAD_ARG, "lut_elem_bytes must be 4 or 8, got %d",
              lut_elem_bytes);
  // (v, v_fp8 and v_scale may all three be NULL: the caller then quantises v itself with sage_quant_v, e.g. on another
  //  stream)
  SLA_REQUIRE(q && k && (sparse_map || !want_map) && (lut || topk == 0) && q_int8 && q_scale && k_int8 && k_scale && workspace &&
                  ((v && v_fp8 && v_scale) || (!v && !v_fp8 && !v_scale)),
              SLA_ERR_BAD_ARG, "null pointer");
  SLA_REQUIRE(((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)lut | (uintptr_t)q_int8 | (uintptr_t)k_int8 |
               (uintptr_t)v_fp8 | (uintptr_t)workspace) % 16 == 0,
              SLA_ERR_BAD_ARG, "pointers must be 16-byte aligned");
  const int BH = B * H;
  SLA_REQUIRE(workspace_bytes >= sage_prepare_workspace_bytes(BH, L, D), SLA_ERR_WORKSPACE, "workspace of %lld bytes, need %lld",
              (long long)workspace_bytes, (long long)sage_prepare_workspace_bytes(BH, L, D));
  return SLA_OK;
}

static int prepare_entry(const void* q, const void* k, const void* v, const int64_t* qkv_strides, int dtype, int B, int H, int L,
                         int D, int BLKQ, int BLKK, int topk, int8_t* sparse_map, void* lut, int lut_elem_bytes, int8_t* q_int8,
                         float* q_scale, int8_t* k_int8, float* k_scale, uint8_t* v_fp8, float* v_scale, float v_range,
                         void* workspace, int64_t workspace_bytes, void* stream) {
  RowLayout lay;
  const int rc = prepare_check(q, k, v, qkv_strides, dtype, B, H, L, D, BLKQ, BLKK, topk, sparse_map, lut, lut_elem_bytes, q_int8,
                               q_scale, k_int8, k_scale, v_fp8, v_scale, v_range, workspace, workspace_bytes, true, &lay);
  if (rc) return rc;
  const int BH = B * H;
  hipStream_t st = (hipStream_t)stream;
  char* ws = (char*)workspace;
  const int lut64 = lut_elem_bytes == 8;
#define SLA_PREP_CASE(TAG, DD) \
  return prepare_impl<TAG, DD>(q, k, v, lay, dtype, BH, L, topk, sparse_map, lut, lut64, q_int8, q_scale, k_int8, k_scale, \
                               v_fp8, v_scale, v_range, ws, st)
  if (dtype == SLA_BF16) {
    if (D == 128) SLA_PREP_CASE(bf16_tag, 128);
    SLA_PREP_CASE(bf16_tag, 64);
  }
  if (D == 128) SLA_PREP_CASE(f16_tag, 128);
  SLA_PREP_CASE(f16_tag, 64);
#undef SLA_PREP_CASE
}

extern "C" int sage_prepare(const void* q, const void* k, const void* v, int dtype, int B, int H, int L, int D, int BLKQ,
                            int BLKK, int topk, int8_t* sparse_map, void* lut, int lut_elem_bytes, int8_t* q_int8,
                            float* q_scale, int8_t* k_int8, float* k_scale, uint8_t* v_fp8, float* v_scale, float v_range,
                            void* workspace, int64_t workspace_bytes, void* stream) {
  return prepare_entry(q, k, v, nullptr, dtype, B, H, L, D, BLKQ, BLKK, topk, sparse_map, lut, lut_elem_bytes, q_int8, q_scale,
                       k_int8, k_scale, v_fp8, v_scale, v_range, workspace, workspace_bytes, stream);
}

extern "C" int sage_prepare_strided(const void* q, const void* k, const void* v, const int64_t* qkv_strides, int dtype, int B,
                                    int H, int L, int D, int BLKQ, int BLKK, int topk, int8_t* sparse_map, void* lut,
                                    int lut_elem_bytes, int8_t* q_int8, float* q_scale, int8_t* k_int8, float* k_scale,
                                    uint8_t* v_fp8, float* v_scale, float v_range, void* workspace,
                                    int64_t workspace_bytes, void* stream) {
  SLA_REQUIRE(qkv_strides, SLA_ERR_BAD_ARG, "null strides");
  return prepare_entry(q, k, v, qkv_strides, dtype, B, H, L, D, BLKQ, BLKK, topk, sparse_map, lut, lut_elem_bytes, q_int8,
                       q_scale, k_int8, k_scale, v_fp8, v_scale, v_range, workspace, workspace_bytes, stream);
}

static int quant_v_entry(const void* v, const int64_t* v_strides, int dtype, int B, int H, int L, int D, uint8_t* v_fp8,
                         float* v_scale, float v_range, void* workspace, int64_t workspace_bytes, void* stream) {
  int rc = validate_sage(dtype, B, H, L, D, 128, 64);
  if (rc) return rc;
  rc = validate_v_range(v_range);
  if (rc) return rc;
  RowLayout lay;
  rc = make_layout(v_strides, B, H, L, D, 2, &lay);
  if (rc) return rc;
  SLA_REQUIRE(v && v_fp8 && v_scale && workspace, SLA_ERR_BAD_ARG, "null pointer");
  SLA_REQUIRE(((uintptr_t)v | (uintptr_t)v_fp8 | (uintptr_t)workspace) % 16 == 0, SLA_ERR_BAD_ARG,
              "pointers must be 16-byte aligned");
  const int BH = B * H;
  SLA_REQUIRE(workspace_bytes >= sage_quant_workspace_bytes(BH, L, D), SLA_ERR_WORKSPACE, "workspace too small");
  hipStream_t st = (hipStream_t)stream;
  char* ws = (char*)workspace;
  if (dtype == SLA_BF16) {
    if (D == 128) return quant_v_impl<bf16_tag, 128>(v, lay, BH, L, v_fp8, v_scale, v_range, ws, st);
    return quant_v_impl<bf16_tag, 64>(v, lay, BH, L, v_fp8, v_scale, v_range, ws, st);
  }
  if (D == 128) return quant_v_impl<f16_tag, 128>(v, lay, BH, L, v_fp8, v_scale, v_range, ws, st);
  return quant_v_impl<f16_tag, 64>(v, lay, BH, L, v_fp8, v_scale, v_range, ws, st);
}

extern "C" int sage_quant_v(const void* v, int dtype, int B, int H, int L, int D, uint8_t* v_fp8, float* v_scale,
                            float v_range, void* workspace, int64_t workspace_bytes, void* stream) {
  return quant_v_entry(v, nullptr, dtype, B, H, L, D, v_fp8, v_scale, v_range, workspace, workspace_bytes, stream);
}

extern "C" int sage_quant_v_strided(const void* v, const int64_t* v_strides, int dtype, int B, int H, int L, int D,
                                    uint8_t* v_fp8, float* v_scale, float v_range, void* workspace,
                                    int64_t workspace_bytes, void* stream) {
  SLA_REQUIRE(v_strides, SLA_ERR_BAD_ARG, "null strides");
  return quant_v_entry(v, v_strides, dtype, B, H, L, D, v_fp8, v_scale, v_range, workspace, workspace_bytes, stream);
}

namespace sla {
// (lin null: the attention alone, contiguous rows)
static int sage_attention_run(const int8_t* q8, const float* qs, const int8_t* k8, const float* ks, const uint8_t* v8, const float* vs,
                              const void* lut, int lut64, void* o, int dtype, int BH, int L, int D, int topk, float qk_scale,
                              const SageLinear* lin, hipStream_t st) {
  const int Mblk = cdiv(L, 128), Nblk = cdiv(L, 64), total = BH * Mblk;
  const float c = qk_scale * 1.4426950408889634f;
#define SAGE_CASE(TAG, DD)                                                                                                  \
  if (lin)                                                                                                                  \
    hipLaunchKernelGGL((sage_fwd_kernel<TAG, DD, 128, true>), dim3(xcd_grid(total)), dim3(256), 0, st, q8, qs, k8, ks, v8, vs, \
                       lut, lut64, (uint16_t*)o, L, Mblk, Nblk, topk, c, total, *lin);                                      \
  else                                                                                                                      \
    hipLaunchKernelGGL((sage_fwd_kernel<TAG, DD, 128, false>), dim3(xcd_grid(total)), dim3(256), 0, st, q8, qs, k8, ks, v8, vs, \
                       lut, lut64, (uint16_t*)o, L, Mblk, Nblk, topk, c, total, SageLinear{})
  if (dtype == SLA_BF16) {
    if (D == 128) { SAGE_CASE(bf16_tag, 128); }
    else { SAGE_CASE(bf16_tag, 64); }
  } else {
    if (D == 128) { SAGE_CASE(f16_tag, 128); }
    else { SAGE_CASE(f16_tag, 64); }
  }
#undef SAGE_CASE
  return check_launch("sage_sparse_attn_fwd");
}
}  // namespace sla

extern "C" int sage_sparse_attn_fwd(const int8_t* q_int8, const float* q_scale, const int8_t* k_int8,
                                    const float* k_scale, const uint8_t* v_fp8, const float* v_scale, const void* lut,
                                    int lut_elem_bytes, void* o, int out_dtype, int B, int H, int L, int D, int BLKQ,
                                    int BLKK, int topk, float qk_scale, void* stream) {
  int rc = validate_sage(out_dtype, B, H, L, D, BLKQ, BLKK);
  if (rc) return rc;
  const int Nblk = cdiv(L, BLKK);
  SLA_REQUIRE(topk >= 0 && topk <= Nblk, SLA_ERR_BAD_ARG, "topk=%d outside [0, %d]", topk, Nblk);
  SLA_REQUIRE(lut_elem_bytes == 4 || lut_elem_bytes == 8, SLA_ERR_BAD_ARG, "lut_elem_bytes must be 4 or 8");
  SLA_REQUIRE(q_int8 && q_scale && k_int8 && k_scale && v_fp8 && v_scale && o && (lut || topk == 0), SLA_ERR_BAD_ARG,
              "null pointer");
  SLA_REQUIRE(((uintptr_t)q_int8 | (uintptr_t)k_int8 | (uintptr_t)v_fp8 | (uintptr_t)o | (uintptr_t)v_scale) % 16 == 0,
              SLA_ERR_BAD_ARG, "pointers must be 16-byte aligned");
  return sage_attention_run(q_int8, q_scale, k_int8, k_scale, v_fp8, v_scale, lut, lut_elem_bytes == 8, o, out_dtype, B * H, L, D,
                            topk, qk_scale, nullptr, (hipStream_t)stream);
}

// ---- the preparation of small inputs in three launches -----------------------------------------------------------------
// The same work as sage_prepare and sla_linear_state_quant_v_fwd, launches that need nothing of each other in one:
//   q quantised (with its block means), chunk sums of k | slices' partial states (with the maxima of |v|), k quantised (with its block
//   means), by workgroups that form its column mean themselves (at most 512 chunk sums, from L2, for two key blocks) | states
//   finished, v quantised, scores and selection
// Each is hidden by what it rides with.  Eleven launches of 2 to 12 us were what a call on 16 heads x 5003 x 64 consisted of besides its
// attention; its kernels in us with the column mean beside the partial states, k beside v and the selection behind: 10.8 + 11.9 + 4.6,
// here 16.3 + 7.7.
//
// Large inputs are bound by their passes over memory: there the chunk sums of k come with the states, which saves one of k, q is
// quantised beside them (at a slice per compute unit they leave room for it), and k and v by a launch that holds little else:
//   slices' partial states with chunk sums of k and maxima of v, q quantised | column mean, scales of v | k and v quantised | states
//   finished, scores and selection (where rows are too long for that in one launch: three)
// LARGE_BYTES: small / large in us, 8 heads x 6000 x 128 (11.7 MiB) 98.0 / 100.5, 12 x 4000 x 128 (11.7 MiB) 66.7 / 68.3, 16 x 6400 x 64
// (12.5 MiB) 66.2 / 67.5, 4 x 13000 x 128 (12.7 MiB) 91.8 / 86.4, 12 x 4400 x 128 (12.9 MiB) 71.7 / 69.8, 16 x 7000 x 64 (13.7 MiB) 74.3
// / 72.5, 12 x 5400 x 128 (15.8 MiB) 92.9 / 87.8; 32 x 3000 x 64 (11.7 MiB) 61.6 / 59.5.  Rows of more than 512 key blocks, which small
// inputs would select from in launches of their own, at any size: 1 head x 40000 x 128 145.3 / 137.6, 1 x 75600 x 64 207 / 203.
// The separate calls, states and v on a second stream, against this: 12 heads x 6500 x 128 113 / 104, 24 x 6500 x 64 96 / 80, 16 x 8000
// x 128 136 / 122, 12 x 16000 x 128 227 / 209, 24 x 16000 x 128 412 / 406, 40 x 20000 x 64 525 / 518, 40 x 32760 x 128 1921 / 1887.
namespace sla {

constexpr int64_t LARGE_BYTES = 25ll << 19;          // of one of q, k, v

template <typename Tag>
struct IoOf;
template <>
struct IoOf<bf16_tag> {
  typedef IoBf16 type;
};
template <>
struct IoOf<f16_tag> {
  typedef IoF16 type;
};

template <typename Tag, int D>
__global__ __launch_bounds__(256) void sage_first_kernel(const uint16_t* __restrict__ q, const uint16_t* __restrict__ k,
                                                         const RowLayout lay, int8_t* __restrict__ q8, float* __restrict__ qs,
                                                         uint16_t* __restrict__ pq, int M, int tiled, float* __restrict__ chunk_sums,
                                                         int nchunk, int L, int quant_wgs, int per_head) {
  __shared__ __attribute__((aligned(16))) char smem[quant_int8_lds<D, 128, true>()];
  const int wg = blockIdx.x;
  if (wg < quant_wgs) {
    quant_int8_body<Tag, D, 128, false, true>(q, lay, nullptr, q8, qs, pq, L, M, tiled, wg % M, wg / M, threadIdx.x, true, smem);
  } else {
    const int i = wg - quant_wgs, bh = i / per_head;
    pool_body<typename IoOf<Tag>::type, 0, 2, 256>(k, lay, nullptr, chunk_sums, L, D, KMEAN_CHUNK, nchunk, 0, i - bh * per_head, bh);
  }
}

// 512 * 8 values of v in FP8, by workgroup `wg` of a head's `v_wgs`, whose scales it forms from the slices' maxima itself (the first
// one of a head leaves them for the attention).  s_scale: D words of LDS.
template <typename Tag, int D>
static __device__ __forceinline__ void sage_quant_v_body(const uint16_t* __restrict__ v, const RowLayout& lay,
                                                         const float* __restrict__ vmax_part, int nsplit, uint8_t* __restrict__ v8,
                                                         float* __restrict__ vs, float v_range, int L, int v_wgs, int wg,
                                                         float* s_scale) {
  using E = Elem<Tag>;
  constexpr int CPR = D / 8, RPP = 512 / CPR;
  const int bh = wg / v_wgs, part = wg - bh * v_wgs, tid = threadIdx.x;
  if (tid < D) {
    const float* p = vmax_part + (size_t)bh * nsplit * D + tid;
    float a = 0.f;
    // (sixteen loads in flight and for the rest eight or sixteen, past the last slice its maxima again.  With the rest one by one the
    //  kernel took 30.3 us with 15 slices of 12 heads x 5400 x 128 and 19.8 with 17; shared among all threads, with a barrier more, the
    //  call at 16 heads x 6001 x 64, 16 slices, 70.3 us where it is 69.2)
    const auto batch = [&](int c, auto loads) __attribute__((always_inline)) {
      constexpr int N = decltype(loads)::value;
      float x[N];
#pragma unroll
      for (int i = 0; i < N; ++i) x[i] = p[(size_t)min(c + i, nsplit - 1) * D];
#pragma unroll
      for (int i = 0; i < N; ++i) a = fmaxf(a, x[i]);
    };
    int c = 0;
    for (; c + 8 < nsplit; c += 16) batch(c, std::integral_constant<int, 16>{});
    if (c < nsplit) batch(c, std::integral_constant<int, 8>{});
    a = fmaxf(a, 1e-30f) / v_range;
    s_scale[tid] = a;
    if (part == 0) vs[(size_t)bh * D + tid] = a;
  }
  const int row = part * RPP + tid / CPR, lcol = (tid % CPR) * 8;
  i16x8_t x = {0, 0, 0, 0, 0, 0, 0, 0};
  if (row < L) x = *reinterpret_cast<const i16x8_t*>(v + lay.head(bh) + (size_t)row * (size_t)lay.sl + lcol);
  lds_barrier();
  if (row >= L) return;
  float f[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) f[e] = E::to_float((uint16_t)x[e]) / s_scale[lcol + e];
  i32x2_t w;
  w[0] = (int)cvt4_fp8(f[0], f[1], f[2], f[3]);
  w[1] = (int)cvt4_fp8(f[4], f[5], f[6], f[7]);
  *reinterpret_cast<i32x2_t*>(v8 + ((size_t)bh * L + row) * D + lcol) = w;
}

template <typename Tag, int D>
__global__ __launch_bounds__((StateTile<D, false>::NTH)) __attribute__((amdgpu_waves_per_eu(4, 4))) void sage_state_k_kernel(
    const uint16_t* __restrict__ k, const uint16_t* __restrict__ v, const RowLayout lay, float* __restrict__ kv_part,
    float* __restrict__ z_part, float* __restrict__ vmax_part, int L, int rows_per_split, int nsplit, int fmap,
    const float* __restrict__ chunk_sums, int nchunk, int state_wgs, int per_head, int8_t* __restrict__ k8, float* __restrict__ ks,
    uint16_t* __restrict__ pk, int N, int tiled) {
  constexpr int QLDS = (quant_int8_lds<D, 64, true>() + 15) / 16 * 16;
  static_assert(2 * QLDS + 2 * D <= StateTile<D, false>::LDS && COLMEAN_LDS_GROUPS * D * 4 <= 2 * QLDS, "two blocks and the mean fit the tiles");
  __shared__ __attribute__((aligned(16))) char smem[StateTile<D, false>::LDS];
  const int wg = blockIdx.x;
  if (wg >= state_wgs) {
    const int bh = (wg - state_wgs) / per_head, half = threadIdx.x >> 8, blk = 2 * (wg - state_wgs - bh * per_head) + half;
    uint16_t* const mean = reinterpret_cast<uint16_t*>(smem + 2 * QLDS);
    colmean_all_body<typename IoOf<Tag>::type, D, 512>(chunk_sums, nchunk, L, bh, reinterpret_cast<float*>(smem), mean);
    quant_int8_body<Tag, D, 64, true, true>(k, lay, mean, k8, ks, pk, L, N, tiled, blk, bh, threadIdx.x & 255, blk < N, smem + half * QLDS);
    return;
  }
  const int bh = wg / nsplit;
  state_partial_body<Tag, D, false, false, true>(k, v, lay, kv_part, z_part, L, rows_per_split, fmap, nullptr, vmax_part,
                                                 wg - bh * nsplit, bh, nsplit, smem);
}
template <typename Tag, int D, int MAX_N>
__global__ __launch_bounds__(512) void sage_finish_select_kernel(const StateFinish job, int finish_wgs, const uint16_t* __restrict__ pq,
                                                                 const uint16_t* __restrict__ pk, void* __restrict__ lut, int M, int N,
                                                                 int T, int select_wgs, const uint16_t* __restrict__ v, const RowLayout lay,
                                                                 const float* __restrict__ vmax_part, uint8_t* __restrict__ v8,
                                                                 float* __restrict__ vs, float v_range, int L, int v_wgs) {
  typedef typename IoOf<Tag>::type IO;
  constexpr int SLDS = SelectLds<IO, D, MAX_N>::BYTES;
  __shared__ __attribute__((aligned(16))) char smem[state_finish_lds<D>() > SLDS ? state_finish_lds<D>() : SLDS];
  int wg = blockIdx.x;
  if (wg < finish_wgs) {
    const int logical = xcd_remap(wg, finish_wgs, job.total);
    if (logical >= 0) state_finish_body<Tag, D>(job, logical, smem);
    return;
  }
  wg -= finish_wgs;
  if (wg < select_wgs) {
    const int per_head = (M + 15) >> 4, bh = wg / per_head;
    select_body<IO, D, true, MAX_N>(pq, pk, nullptr, lut, 0, M, N, T, wg - bh * per_head, bh, smem);
    return;
  }
  sage_quant_v_body<Tag, D>(v, lay, vmax_part, job.nsplit, v8, vs, v_range, L, v_wgs, wg - select_wgs, reinterpret_cast<float*>(smem));
}

template <typename Tag, int D>
static void launch_small_preparation(const void* q, const void* k, const void* v, const RowLayout& lay, int dtype, const float* weight,
                                     int fmap, int BH, int L, int topk, void* lut, int8_t* q8, float* qs, int8_t* k8, float* ks,
                                     uint8_t* v8, float* vs, float v_range, char* prep, char* linear, hipStream_t st) {
  const SageWs w = sage_ws(BH, L, D);
  const SagePrepWs p = sage_prep_ws(BH, L, D);
  const LinWs lw = lin_ws(BH, L, D);
  const int M = cdiv(L, 128), N = cdiv(L, 64), tiled = score_takes_tiled(dtype, D);
  float* const chunk_sums = (float*)(prep + w.chunk_sums);
  uint16_t *const pq = (uint16_t*)(prep + p.pq), *const pk = (uint16_t*)(prep + p.pk);
  const int per_head = cdiv(N, 256 / (D / 2));               // (chunks of KMEAN_CHUNK = 64 rows)
  hipLaunchKernelGGL((sage_first_kernel<Tag, D>), dim3(BH * M + BH * per_head), dim3(256), 0, st, (const uint16_t*)q,
                     (const uint16_t*)k, lay, q8, qs, pq, M, tiled, chunk_sums, N, L, BH * M, per_head);
  const int state_wgs = BH * lw.nsplit, v_wgs = cdiv(L, 512 / (D / 8));
  const int k_per_head = cdiv(N, 2);
  hipLaunchKernelGGL((sage_state_k_kernel<Tag, D>), dim3(state_wgs + BH * k_per_head), dim3(StateTile<D, false>::NTH), 0, st,
                     (const uint16_t*)k, (const uint16_t*)v, lay, (float*)(linear + lw.kv_part), (float*)(linear + lw.z_part),
                     (float*)(linear + lw.vmax_part), L, lw.rows_per_split, lw.nsplit, fmap, (const float*)chunk_sums, N, state_wgs,
                     k_per_head, k8, ks, pk, N, tiled);
  launch_state_presum<D>(BH, linear + lw.states_end, lw, st);
  const StateFinish job = state_finish_job<D>(weight, BH, linear, linear + lw.states_end, lw);
  const int finish_wgs = xcd_grid(job.total), select_wgs = BH * cdiv(M, 16);
#define SAGE_FINISH_CASE(MAX_N)                                                                                               \
  hipLaunchKernelGGL((sage_finish_select_kernel<Tag, D, MAX_N>), dim3(finish_wgs + select_wgs + BH * v_wgs), dim3(512), 0, st, job, \
                     finish_wgs, (const uint16_t*)pq, (const uint16_t*)pk, lut, M, N, topk, select_wgs, (const uint16_t*)v, lay,   \
                     (const float*)(linear + lw.vmax_part), v8, vs, v_range, L, v_wgs)
  if (N > SELECT_ONE_N) SAGE_FINISH_CASE(SELECT_LONG_N);
  else if (N > SELECT_FUSED_N) SAGE_FINISH_CASE(SELECT_ONE_N);
  else SAGE_FINISH_CASE(SELECT_FUSED_N);
#undef SAGE_FINISH_CASE
}

// ---- and of large ones
// grid (2 D / 16, heads): column mean of k, scales of v
template <typename Tag, int D>
__global__ __launch_bounds__(256) void sage_means_kernel(const float* __restrict__ chunk_sums, uint16_t* __restrict__ colmean, int nchunk,
                                                         int L, const float* __restrict__ vmax_part, float* __restrict__ vs, int nsplit,
                                                         float v_range) {
  __shared__ float gs[COLMEAN_MAX_GROUPS * COLMEAN_SLAB];
  constexpr int SLABS = D / COLMEAN_SLAB;
  if (blockIdx.x < SLABS)
    colmean_body<typename IoOf<Tag>::type, 256>(chunk_sums, colmean, nchunk, (nchunk + KMEAN_GROUP - 1) / KMEAN_GROUP, D, L, blockIdx.x,
                                                blockIdx.y, gs);
  else
    v_scale_body(vmax_part, vs, nsplit, D, v_range, blockIdx.x - SLABS, blockIdx.y, gs);
}

// the slices' partial states with the chunk sums of k and the maxima of v; from `state_wgs` on two query blocks per workgroup
template <typename Tag, int D>
__global__ __launch_bounds__((StateTile<D, false>::NTH)) __attribute__((amdgpu_waves_per_eu(4, 4))) void sage_large_first_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ k, const uint16_t* __restrict__ v, const RowLayout lay,
    float* __restrict__ kv_part, float* __restrict__ z_part, float* __restrict__ vmax_part, int L, int rows_per_split, int nsplit, int fmap,
    float* __restrict__ chunk_sums, int nchunk, int state_wgs, int8_t* __restrict__ q8, float* __restrict__ qs, uint16_t* __restrict__ pq,
    int M, int tiled) {
  constexpr int QLDS = (quant_int8_lds<D, 128, true>() + 15) / 16 * 16, SLDS = StateTile<D, false>::LDS_KSUM;
  __shared__ __attribute__((aligned(16))) char smem[2 * QLDS > SLDS ? 2 * QLDS : SLDS];
  const int wg = blockIdx.x;
  if (wg >= state_wgs) {
    const int per_head = (M + 1) / 2, i = wg - state_wgs, bh = i / per_head, half = threadIdx.x >> 8, blk = 2 * (i - bh * per_head) + half;
    quant_int8_body<Tag, D, 128, false, true>(q, lay, nullptr, q8, qs, pq, L, M, tiled, blk, bh, threadIdx.x & 255, blk < M, smem + half * QLDS);
    return;
  }
  const int bh = wg / nsplit;
  state_partial_body<Tag, D, false, false, true, false, true>(k, v, lay, kv_part, z_part, L, rows_per_split, fmap, nullptr, vmax_part,
                                                              wg - bh * nsplit, bh, nsplit, smem, chunk_sums, nchunk);
}

// k, a block per workgroup, then v, 4 * 256 * 8 values
constexpr int V_ROWS = 4;                  // rows per thread
template <typename Tag, int D>
__global__ __launch_bounds__(256) void sage_quant_kv_kernel(const uint16_t* __restrict__ k, const uint16_t* __restrict__ v, const RowLayout lay,
                                                            const uint16_t* __restrict__ colmean, int8_t* __restrict__ k8,
                                                            float* __restrict__ ks, uint16_t* __restrict__ pk, int N, int tiled,
                                                            const float* __restrict__ vs, uint8_t* __restrict__ v8, int L, int k_wgs,
                                                            int v_per_head) {
  using E = Elem<Tag>;
  __shared__ __attribute__((aligned(16))) char smem[quant_int8_lds<D, 64, true>()];
  int wg = blockIdx.x;
  if (wg < k_wgs) {
    const int bh = wg / N;
    quant_int8_body<Tag, D, 64, true, true>(k, lay, colmean + (size_t)bh * D, k8, ks, pk, L, N, tiled, wg - bh * N, bh, threadIdx.x, true, smem);
    return;
  }
  wg -= k_wgs;
  constexpr int CPR = D / 8, RPP = 256 / CPR;
  const int bh = wg / v_per_head, row0 = (wg - bh * v_per_head) * V_ROWS * RPP + threadIdx.x / CPR, lcol = (threadIdx.x % CPR) * 8;
  const uint16_t* const p = v + lay.head(bh) + lcol;
  i16x8_t x[V_ROWS];
#pragma unroll
  for (int i = 0; i < V_ROWS; ++i) x[i] = *reinterpret_cast<const i16x8_t*>(p + (size_t)min(row0 + i * RPP, L - 1) * (size_t)lay.sl);
  float s[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) s[e] = vs[(size_t)bh * D + lcol + e];
#pragma unroll
  for (int i = 0; i < V_ROWS; ++i) {
    const int row = row0 + i * RPP;
    if (row >= L) return;
    float f[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) f[e] = E::to_float((uint16_t)x[i][e]) / s[e];
    i32x2_t w;
    w[0] = (int)cvt4_fp8(f[0], f[1], f[2], f[3]);
    w[1] = (int)cvt4_fp8(f[4], f[5], f[6], f[7]);
    *reinterpret_cast<i32x2_t*>(v8 + ((size_t)bh * L + row) * D + lcol) = w;
  }
}

template <typename Tag, int D>
static void launch_large_preparation(const void* q, const void* k, const void* v, const RowLayout& lay, int dtype, const float* weight,
                                     int fmap, int BH, int L, int topk, void* lut, int8_t* q8, float* qs, int8_t* k8, float* ks,
                                     uint8_t* v8, float* vs, float v_range, char* prep, char* linear, hipStream_t st) {
  const SageWs w = sage_ws(BH, L, D);
  const SagePrepWs p = sage_prep_ws(BH, L, D);
  const LinWs lw = lin_ws(BH, L, D);
  const int M = cdiv(L, 128), N = cdiv(L, 64), tiled = score_takes_tiled(dtype, D);
  float* const chunk_sums = (float*)(prep + w.chunk_sums);
  uint16_t *const colmean = (uint16_t*)(prep + w.colmean), *const pq = (uint16_t*)(prep + p.pq), *const pk = (uint16_t*)(prep + p.pk);
  float* const vmax_part = (float*)(linear + lw.vmax_part);
  const int state_wgs = BH * lw.nsplit;
  hipLaunchKernelGGL((sage_large_first_kernel<Tag, D>), dim3(state_wgs + BH * cdiv(M, 2)), dim3(StateTile<D, false>::NTH), 0, st,
                     (const uint16_t*)q, (const uint16_t*)k, (const uint16_t*)v, lay, (float*)(linear + lw.kv_part),
                     (float*)(linear + lw.z_part), vmax_part, L, lw.rows_per_split, lw.nsplit, fmap, chunk_sums, N, state_wgs, q8, qs, pq, M,
                     tiled);
  hipLaunchKernelGGL((sage_means_kernel<Tag, D>), dim3(2 * D / COLMEAN_SLAB, BH), dim3(256), 0, st, (const float*)chunk_sums, colmean, N, L,
                     (const float*)vmax_part, vs, lw.nsplit, v_range);
  const int k_wgs = BH * N, v_per_head = cdiv(L, V_ROWS * 256 / (D / 8));
  hipLaunchKernelGGL((sage_quant_kv_kernel<Tag, D>), dim3(k_wgs + BH * v_per_head), dim3(256), 0, st, (const uint16_t*)k, (const uint16_t*)v,
                     lay, (const uint16_t*)colmean, k8, ks, pk, N, tiled, (const float*)vs, v8, L, k_wgs, v_per_head);
  launch_state_presum<D>(BH, linear + lw.states_end, lw, st);
  const StateFinish job = state_finish_job<D>(weight, BH, linear, linear + lw.states_end, lw);
  const int finish_wgs = xcd_grid(job.total), select_wgs = BH * cdiv(M, 16);
  if (select_fits(N, D, 2)) {
#define SAGE_FINISH_CASE(MAX_N)                                                                                               \
  hipLaunchKernelGGL((sage_finish_select_kernel<Tag, D, MAX_N>), dim3(finish_wgs + select_wgs), dim3(512), 0, st, job, finish_wgs, \
                     (const uint16_t*)pq, (const uint16_t*)pk, lut, M, N, topk, select_wgs, (const uint16_t*)v, lay,          \
                     (const float*)vmax_part, v8, vs, v_range, L, 0)
    if (N > SELECT_ONE_N) SAGE_FINISH_CASE(SELECT_LONG_N);
    else if (N > SELECT_FUSED_N) SAGE_FINISH_CASE(SELECT_ONE_N);
    else SAGE_FINISH_CASE(SELECT_FUSED_N);
#undef SAGE_FINISH_CASE
    return;
  }
  hipLaunchKernelGGL((linear_state_finish_kernel<Tag, D>), dim3(finish_wgs), dim3(512), 0, st, job);
  launch_map_from_pooled(dtype, pq, pk, prep + p.score, BH, M, N, D, topk, nullptr, lut, 0, st);
}

}  // namespace sla

// ---- the whole quantised forward in one call -----------------------------------------------------------------------
namespace sla {
struct SageModuleWs {
  int64_t prep_bytes, linear_bytes;
  size_t prep, linear, q8, k8, v8, qs, ks, vs, lut, total;
};
static SageModuleWs sage_module_ws(int B, int H, int L, int D, int topk) {
  const int64_t BH = (int64_t)B * H, M = cdiv(L, 128), N = cdiv(L, 64), elems = BH * L * D;
  SageModuleWs w;
  w.prep_bytes = sage_prepare_workspace_bytes((int)BH, L, D);
  w.linear_bytes = linear_fwd_workspace_bytes((int)BH, L, D);
  size_t off = 0;
  w.prep = off;   off += align_up(w.prep_bytes, 256);
  w.linear = off; off += align_up(w.linear_bytes, 256);
  w.q8 = off;     off += align_up(elems, 256);
  w.k8 = off;     off += align_up(elems, 256);
  w.v8 = off;     off += align_up(elems, 256);
  w.qs = off;     off += align_up(BH * M * 4, 256);
  w.ks = off;     off += align_up(BH * N * 4, 256);
  w.vs = off;     off += align_up(BH * D * 4, 256);
  w.lut = off;    off += align_up(BH * M * topk * 4, 256);
  w.total = off;
  return w;
}
int64_t sage_module_workspace_bytes(int B, int H, int L, int D, int topk) {
  return (int64_t)sage_module_ws(B, H, L, D, topk).total;
}
}  // namespace sla

extern "C" int sage_module_fwd(const void* q, const void* k, const void* v, const int64_t* qkv_strides, const float* weight,
                               const float* bias, void* out, const int64_t* out_strides, int dtype, int fmap, int B, int H, int L,
                               int D, int topk, float qk_scale, float v_range, void* workspace, int64_t workspace_bytes,
                               void* stream, void* /*side_stream*/) {
  int rc = validate_sage(dtype, B, H, L, D, 128, 64);
  if (rc) return rc;
  SLA_REQUIRE((qkv_strides == nullptr) == (out_strides == nullptr), SLA_ERR_BAD_ARG, "pass both stride arrays or neither");
  SLA_REQUIRE(topk >= 0 && topk <= cdiv(L, 64), SLA_ERR_BAD_ARG, "topk=%d outside [0, %d]", topk, cdiv(L, 64));
  SLA_REQUIRE(fmap == SLA_FMAP_ELU || fmap == SLA_FMAP_RELU || fmap == SLA_FMAP_SOFTMAX, SLA_ERR_BAD_ARG,
              "unknown feature map %d", fmap);
  SLA_REQUIRE(q && k && v && weight && bias && out && workspace, SLA_ERR_BAD_ARG, "null pointer");
  SLA_REQUIRE(((uintptr_t)k | (uintptr_t)v | (uintptr_t)workspace | (uintptr_t)weight | (uintptr_t)out) % 16 == 0,
              SLA_ERR_BAD_ARG, "pointers must be 16-byte aligned");
  const SageModuleWs w = sage_module_ws(B, H, L, D, topk);
  SLA_REQUIRE(workspace_bytes >= (int64_t)w.total, SLA_ERR_WORKSPACE, "workspace of %lld bytes, need %lld",
              (long long)workspace_bytes, (long long)w.total);
  RowLayout lay, lout;
  if ((rc = make_layout(out_strides, B, H, L, D, 2, &lout))) return rc;
  char* ws = (char*)workspace;
  hipStream_t st = (hipStream_t)stream;
  int8_t *q8 = (int8_t*)(ws + w.q8), *k8 = (int8_t*)(ws + w.k8);
  uint8_t* v8 = (uint8_t*)(ws + w.v8);
  float *qs = (float*)(ws + w.qs), *ks = (float*)(ws + w.ks), *vs = (float*)(ws + w.vs);
  void* lut = ws + w.lut;
  // (what the later steps would find wrong, before the first launch)
  rc = prepare_check(q, k, nullptr, qkv_strides, dtype, B, H, L, D, 128, 64, topk, nullptr, lut, 4, q8, qs, k8, ks, nullptr,
                     nullptr, v_range, ws + w.prep, w.prep_bytes, false, &lay);
  if (rc) return rc;
  RowLayout lq;
  if ((rc = make_layout(qkv_strides, B, H, L, D, 2, &lq))) return rc;
  const auto attention = [&]() -> int {
    const LinWs lw = lin_ws(B * H, L, D);
    const char* states = ws + w.linear;
    const SageLinear lin{(const uint16_t*)q, (const uint16_t*)(states + lw.kvwt), (const uint16_t*)(states + lw.z), bias, lq, lout, fmap};
    return sage_attention_run(q8, qs, k8, ks, v8, vs, lut, 0, out, dtype, B * H, L, D, topk, qk_scale, &lin, st);
  };
  const bool large = (int64_t)B * H * L * D * 2 > LARGE_BYTES || !select_fits(cdiv(L, 64), D, 2);
#define SAGE_PREPARE(TAG, DD)                                                                                                \
  (large ? launch_large_preparation<TAG, DD> : launch_small_preparation<TAG, DD>)(q, k, v, lq, dtype, weight, fmap, B * H, L, topk, lut, \
                                                                                  q8, qs, k8, ks, v8, vs, v_range, ws + w.prep,      \
                                                                                  ws + w.linear, st)
  if (dtype == SLA_BF16) {
    if (D == 128) SAGE_PREPARE(bf16_tag, 128);
    else SAGE_PREPARE(bf16_tag, 64);
  } else {
    if (D == 128) SAGE_PREPARE(f16_tag, 128);
    else SAGE_PREPARE(f16_tag, 64);
  }
#undef SAGE_PREPARE
  if ((rc = check_launch("sage_module_fwd"))) return rc;
  return attention();
}
