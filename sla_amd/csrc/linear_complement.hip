// Linear branch over the NON-selected key blocks ("complement" mode), projection and final sum, for gfx950.
//
// The mounted reference computes the linear branch over all keys (sparse_linear_attention/core.py:92-96);
// the variant in which query block i only sees the key blocks it did not select for the sparse branch has no
// code there.  Definition used here (per head, S_i = look-up row of query block i, block size BLKK = 64):
//   h_j = phi(K_j)^T V_j (D x D),  z_j = sum_rows phi(K_j)            per key block j
//   H_i = sum_j h_j - sum_{j in S_i} h_j,   z_i likewise              per query block i
//   o_l = phi(Q_i) H_i / (1e-5 + phi(Q_i) . z_i);  out = residual + o_l W^T + b
// Rounding: phi, h_j, H_i, z_i, o_l are rounded to the 16-bit dtype where the global path rounds its
// counterparts; a state is one fp32 accumulation over the blocks that take part, in ascending order (H_i is formed as the sum over
// the j outside S_i, nothing is subtracted).
//
// Kernels:
//   block states : linear_state_partial_kernel with one 64-row slice per workgroup, 16-bit h_j^T, fp32 z_j
//   weights      : one row of bits per query block, set for the key blocks its look-up row does not name
//   states       : H_i, z_i = weights times block states, per query block (H_i rounded); the backward reads them again
//   out          : N^T = H_i^T phi(Q)^T, OUT^T = W Y^T for the rows of a query block in the transposed
//                  formulation of the global output kernel.
// At 12 heads of 16380 rows, head dim 128, 12 of 256 blocks selected, with the states formed inside the kernels of the rows (a
// workgroup per query or key block, the whole state in 64 fp32 registers per thread, two waves per SIMD): out 236 us,
// rows 171 us, kv 171 us.  With the states in a kernel of their own: out 56 us, rows 97 us, kv 75 us.
#include "bwd_lists.h"
#include "linear_state.h"

namespace sla {

int validate_attn_shape(int dtype, int B, int H, int L, int D, int BLKQ, int BLKK, int topk, int lut_elem_bytes);
int64_t weight_grads_workspace_bytes(int BH, int L, int D);
HeadSums launch_weight_grads(int dtype, int D, const void* gout, const void* y, int BH, int L, char* ws, float* d_weight,
                             float* d_bias, hipStream_t st);

// Weights of the states: one bit per row and block state, 1 where the state takes part; zero from the table's end on.
// all[head][row] says that the row leaves every block out.  A lane of the matrix instruction holds one row and eight of sixteen
// columns; a word is what it needs of 64 columns, the even ones' bits in the lower half and the odd ones' in the upper, so that
// a shift and a mask leave the operand's pairs with the pattern of 2.0 (one bit in either 16-bit format, and in fp32) where the
// bit is set.  Words of a head: [32 rows][64 columns][lane].
constexpr int WEIGHT_STEP = 64;
static inline int64_t weight_words(int nrows, int nblk) { return (int64_t)cdiv(nrows, 32) * cdiv(nblk, WEIGHT_STEP) * 64; }
static __device__ __forceinline__ int weight_bit(int c) { return (c >> 2 & 12) + (c >> 1 & 3) + 16 * (c & 1); }

// Rows of a look-up table (query blocks): the blocks the row does not name.  grid (nrows, heads).  With `weight` the first head's
// workgroups also leave the projection weight behind for the output kernel: 16 bit, as the A operand of OUT^T = W Y^T with the columns
// in accumulator slot order, 32 rows x 16 columns after one another in the order in which a wave reads them.
template <typename Tag>
__global__ __launch_bounds__(64) void complement_row_weights_kernel(const void* __restrict__ lut, int lut64, int topk,
                                                                    uint32_t* __restrict__ w, int* __restrict__ all, int nblk,
                                                                    const float* __restrict__ weight, uint16_t* __restrict__ wo, int D) {
  using E = Elem<Tag>;
  constexpr int SPAN = 1024;             // words at a time (32768 blocks)
  __shared__ uint32_t word[SPAN];
  const int row = blockIdx.x, nrows = gridDim.x, steps = (nblk + WEIGHT_STEP - 1) / WEIGHT_STEP, tid = threadIdx.x;
  const size_t at = (size_t)blockIdx.y * nrows + row;
  if (weight && blockIdx.y == 0)
    for (int p = row * 64 + tid; p < D * D / 8; p += nrows * 64) {
      const int tile = p >> 6, et = tile / (D / 16), c = tile - et * (D / 16);
      const float* const x = weight + (32 * et + (p & 31)) * D + 16 * c + 4 * (p >> 5 & 1);
      i32x4_t y;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const f32x4_t v = *reinterpret_cast<const f32x4_t*>(x + 8 * h);
        y[2 * h] = (int)E::pack2(v[0], v[1]);
        y[2 * h + 1] = (int)E::pack2(v[2], v[3]);
      }
      *reinterpret_cast<i32x4_t*>(wo + 8 * p) = y;
    }
  w += ((size_t)blockIdx.y * ((nrows + 31) >> 5) + (row >> 5)) * steps * 64;
  for (int w0 = 0; w0 < 2 * steps; w0 += SPAN) {
    const int span = min(SPAN, 2 * steps - w0);
    for (int i = tid; i < span; i += 64) {
      const int c0 = ((w0 + i) >> 1) * WEIGHT_STEP + 8 * (i & 1);
      uint32_t x = 0;
#pragma unroll
      for (int e = 0; e < 32; ++e) {
        const int c = 16 * (e >> 3) + (e & 7);
        x |= c0 + c < nblk ? 1u << weight_bit(c) : 0u;
      }
      word[i] = x;
    }
    __syncthreads();
    for (int t = tid; t < topk; t += 64) {
      const int j = lut64 ? (int)reinterpret_cast<const long long*>(lut)[at * topk + t] : reinterpret_cast<const int*>(lut)[at * topk + t];
      const int i = (j >> 6) * 2 + (j >> 3 & 1) - w0;
      if (j >= 0 && i >= 0 && i < span) atomicAnd(&word[i], ~(1u << weight_bit(j & 63)));
    }
    __syncthreads();
    for (int i = tid; i < span; i += 64) w[(w0 + i) * 32 + (row & 31)] = word[i];
    __syncthreads();
  }
  if (tid == 0) all[at] = topk >= nblk;
}

// Columns of the map (key blocks): the query blocks that did not select it.  A workgroup per strip of 64 key blocks and head, a
// lane per key block, a word per wave and pass.  In the workgroups from `strips` x heads on the sum of the heads' weight gradients,
// a wave each, which needs nothing of it: both are bound by latency, 5 us each in launches of their own (forward and backward of 12
// heads x 16380 x 128 1059 us, in one 1057).
__global__ __launch_bounds__(512) void complement_column_weights_kernel(const int8_t* __restrict__ map, uint32_t* __restrict__ w,
                                                                        int* __restrict__ all, int Mblk, int Nblk, int strips,
                                                                        int first_sum, const HeadSums heads) {
  __shared__ uint32_t any[64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if ((int)blockIdx.x >= first_sum) {
    const int job = ((int)blockIdx.x - first_sum) * 8 + wave;
    if (job < heads.wgs) head_sums_body(heads, job);
    return;
  }
  const int head = blockIdx.x / strips, n = (blockIdx.x - head * strips) * 64 + lane;
  const int steps = (Mblk + WEIGHT_STEP - 1) / WEIGHT_STEP;
  const size_t bh = head;
  if (wave == 0) any[lane] = 0;
  __syncthreads();
  if (n < Nblk) {
    const int8_t* const col = map + bh * Mblk * Nblk + n;
    w += (bh * ((Nblk + 31) >> 5) + (n >> 5)) * steps * 64;
    uint32_t seen = 0;
    for (int i = wave; i < 2 * steps; i += 8) {
      const int m0 = (i >> 1) * WEIGHT_STEP + 8 * (i & 1);
      int8_t sel[32];
#pragma unroll
      for (int e = 0; e < 32; ++e) sel[e] = col[(size_t)min(m0 + 16 * (e >> 3) + (e & 7), Mblk - 1) * Nblk];
      uint32_t x = 0;
#pragma unroll
      for (int e = 0; e < 32; ++e) {
        const int c = 16 * (e >> 3) + (e & 7);
        x |= m0 + c < Mblk && sel[e] != 1 ? 1u << weight_bit(c) : 0u;
      }
      w[i * 32 + (n & 31)] = x;
      seen |= x;
    }
    if (seen) atomicOr(&any[lane], 1u);
  }
  __syncthreads();
  if (wave == 0 && n < Nblk) all[bh * Nblk + n] = any[lane] == 0;
}

// Rows' states, states[r] = the sum of the block states whose bit is set in row r (16-bit result), z in fp32: for every query
// block in the forward, for every key block in the backward.
//
// A matrix product of the weights (nrows x nblk) with the block states (nblk x D*D) on the matrix cores, whose products are
// exact (weights 0 and 2, the sum halved at the end), accumulated in fp32.  Bound by memory up to some 400 blocks (every block
// state is read once per workgroup's rows and every state written once: 2 x 32 KB per row at D = 128), by the matrix cores above.
// A workgroup of four waves takes 128 rows x 256 values (RW = 1) or 256 x 128 (RW = 2), a wave 128 x 64 as eight 32 x 32 accumulators
// (parts of 32 rows that the head does not have are left out): eight products for every four transposed LDS reads.  Tiles of 64 blocks
// go through registers, two tiles ahead, into one of two LDS buffers.  Even and odd values of a row are parked apart, so that a lane's
// two column tiles hold neighbouring values and 32 lanes store whole 128-byte lines.
// z: workgroups of their own (the first ones of a head), 128 RW rows x 32 values, fp32 matrix products.
// Against `total - sum of the listed states` on the vector ALU, the union of eight rows' lists at a time, and its totals in two
// launches: 12 heads x 16380 x 128, 12 of 256 blocks selected 70 us where that took 101 + 23 + 8; forward and backward of 12 heads
// x 75600 x 128 with 5 % selected 12.2 ms (15.5), 10.7 (11.8) where neighbouring rows select alike, 6.6 (6.8) with 2 %; 8 heads x
// 4096 x 128 with 20 % 309 us (382).  64 x 64 values per wave: the same up to 256 blocks, 7.0 ms for the one with 2 %.
// A row that leaves every block out is exactly zero, whatever the block states hold.
template <typename Tag, int D, int RW>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void complement_states_kernel(
    const uint16_t* __restrict__ blocks, const float* __restrict__ zblocks, const uint32_t* __restrict__ w,
    const int* __restrict__ all, uint16_t* __restrict__ states, float* __restrict__ zstates, int nrows, int nblk, int ntotal) {
  using E = Elem<Tag>;
  constexpr int DD = D * D;
  constexpr int MI = 4, BM = 128 * RW, BN = 256 / RW, KS = WEIGHT_STEP;
  constexpr int CPR = BN / 8, NP = KS * CPR / 256;   // 16-byte pieces of a row; pieces per thread and tile
  constexpr int STR = BN + 16;                       // transposed reads of 4 rows hit disjoint banks
  constexpr int ZT = D / 32, CT = DD / BN;
  __shared__ __attribute__((aligned(16))) uint16_t sB[2][KS * STR];
  __shared__ int sAll[BM];
  const int logical = xcd_remap(blockIdx.x, gridDim.x, ntotal);
  if (logical < 0) return;
  const int rtiles = (nrows + BM - 1) / BM, per_head = (ZT + CT) * rtiles;
  const int bh = logical / per_head, rest = logical - bh * per_head;
  const int ct = rest / rtiles, row0 = (rest - ct * rtiles) * BM;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int g = lane >> 5, r = lane & 31;
  const int steps = (nblk + KS - 1) / KS;
  const uint32_t* const wb = w + (size_t)bh * ((nrows + 31) >> 5) * steps * 64 + lane;
  if (tid < BM) sAll[tid] = all[(size_t)bh * nrows + min(row0 + tid, nrows - 1)];          // (BM <= 256)
  __syncthreads();

  if (ct < ZT) {
    // ---- z: rows row0 + 32 wave .. (and 128 further), values 32 ct .. ----
#pragma unroll 1
    for (int rw = 0; rw < RW; ++rw) {
      const int local = 128 * rw + 32 * wave, base = row0 + local;
      if (base >= nrows) return;
      const uint32_t* wr = wb + (size_t)(base >> 5) * steps * 64;
      const float* zb = zblocks + (size_t)bh * nblk * D;
      f32x16_t acc;
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[i] = 0.f;
      uint32_t a[2];
      float z[2][32];
      // (lane group g holds blocks 16 c + 8 g + u of a step)
      const auto fetch = [&](int st, int s) __attribute__((always_inline)) {
        const __amdgpu_buffer_rsrc_t rs = make_rsrc(zb + (size_t)st * KS * D, (uint32_t)min(nblk - st * KS, KS) * D * 4u);
        a[s] = wr[st * 64];
#pragma unroll
        for (int u = 0; u < 32; ++u)
          z[s][u] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
              rs, (int)(((16 * (u >> 3) + 8 * g + (u & 7)) * D + 32 * ct + r) * 4), 0, 0));
      };
      fetch(0, 0);
      for (int s0 = 0; s0 < steps; s0 += 2)
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          if (s0 + s >= steps) break;
          if (s0 + s + 1 < steps) fetch(s0 + s + 1, s ^ 1);
#pragma unroll
          for (int u = 0; u < 32; ++u) {
            const int bit = (u >> 1) + 16 * (u & 1);             // (u = 8 c + e: weight_bit(16 c + e))
            const float x = __uint_as_float((bit <= 30 ? a[s] << (30 - bit) : a[s] >> 1) & 0x40000000u);
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(x, z[s][u], acc, 0, 0, 0);
          }
        }
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int row = 8 * (i >> 2) + 4 * g + (i & 3);
        if (base + row < nrows)
          zstates[((size_t)bh * nrows + base + row) * D + 32 * ct + r] = sAll[local + row] ? 0.f : 0.5f * acc[i];
      }
    }
    return;
  }

  const int col0 = (ct - ZT) * BN;
  const int tr_row = (lane & 15) >> 2, tr_col = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
  const int brow = tid / CPR, bch = tid % CPR;       // this thread's piece of rows brow + 256 / CPR p
  const uint16_t* const hb = blocks + (size_t)bh * nblk * DD + col0;
  const int mrow = 128 * (wave % RW), cgrp = wave / RW;          // this wave's rows and 64 values
  const int mine = min(MI, (nrows - row0 - mrow + 31) / 32);     // 32-row parts with rows
  const uint32_t* wp[MI];                             // (a part without rows reads the last one with rows, to no end)
#pragma unroll
  for (int m = 0; m < MI; ++m) wp[m] = wb + (size_t)(min(row0 + mrow + 32 * m, nrows - 1) >> 5) * steps * 64;

  f32x16_t acc[MI][2];
#pragma unroll
  for (int m = 0; m < MI; ++m)
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[m][t][i] = 0.f;
  i16x8_t breg[2][NP];
  uint32_t areg[2][MI];
  const auto fetch_b = [&](int k0, int s) __attribute__((always_inline)) {
    const int rows = min(KS, nblk - k0);             // (rows past the last block read as zero)
    const __amdgpu_buffer_rsrc_t rs = make_rsrc(hb + (size_t)k0 * DD, rows > 0 ? ((uint32_t)(rows - 1) * DD + BN) * 2u : 0u);
#pragma unroll
    for (int p = 0; p < NP; ++p) breg[s][p] = buf_load_b128(rs, ((uint32_t)(brow + 256 / CPR * p) * DD + 8u * (uint32_t)bch) * 2u);
  };
  const auto park_b = [&](int s) __attribute__((always_inline)) {
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const i32x4_t x = __builtin_bit_cast(i32x4_t, breg[s][p]);
      i32x2_t even, odd;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        even[h] = (int)__builtin_amdgcn_perm((uint32_t)x[2 * h + 1], (uint32_t)x[2 * h], 0x05040100u);
        odd[h] = (int)__builtin_amdgcn_perm((uint32_t)x[2 * h + 1], (uint32_t)x[2 * h], 0x07060302u);
      }
      uint16_t* at = &sB[s][(brow + 256 / CPR * p) * STR + 4 * bch];
      *reinterpret_cast<i32x2_t*>(at) = even;
      *reinterpret_cast<i32x2_t*>(at + BN / 2) = odd;
    }
  };
  const auto fetch_a = [&](int k0, int s) __attribute__((always_inline)) {
#pragma unroll
    for (int m = 0; m < MI; ++m) areg[s][m] = wp[m][k0];
  };
  const auto operand = [](uint32_t x, int c) __attribute__((always_inline)) {
    i32x4_t a;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int d = 4 * c + i;
      a[i] = (int)((d <= 14 ? x << (14 - d) : x >> 1) & 0x40004000u);
    }
    return __builtin_bit_cast(i16x8_t, a);
  };
  fetch_b(0, 0);
  fetch_b(KS, 1);
  fetch_a(0, 0);
  park_b(0);
  fetch_b(2 * KS, 0);
  lds_barrier();
  const auto step = [&](int k0, int s) __attribute__((always_inline)) {
    if (k0 + KS < nblk) fetch_a(k0 + KS, s ^ 1);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      if (k0 + 16 * c >= nblk) break;
      i16x8_t b[2];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const uint16_t* p = &sB[s][(16 * c + 8 * g + tr_row) * STR + (BN / 2) * t + 32 * cgrp + tr_col];
        b[t] = concat4(lds_read_tr16(p), lds_read_tr16(p + 4 * STR));
      }
#pragma unroll
      for (int m = 0; m < MI; ++m)
        if (m < mine) {
          const i16x8_t a = operand(areg[s][m], c);
#pragma unroll
          for (int t = 0; t < 2; ++t) acc[m][t] = E::mfma32(a, b[t], acc[m][t]);
        }
    }
    if (k0 + KS < nblk) {
      park_b(s ^ 1);
      fetch_b(k0 + 3 * KS, s ^ 1);
      lds_barrier();
    }
  };
  for (int k0 = 0; k0 < nblk; k0 += 2 * KS)
#pragma unroll
    for (int s = 0; s < 2; ++s)
      if (s == 0 || k0 + KS < nblk) step(k0 + s * KS, s);

#pragma unroll
  for (int m = 0; m < MI; ++m)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int row = mrow + 32 * m + 8 * (i >> 2) + 4 * g + (i & 3);
      if (row0 + row < nrows) {
        uint32_t v = E::pack2(0.5f * acc[m][0][i], 0.5f * acc[m][1][i]);
        if (sAll[row]) v = 0u;
        *reinterpret_cast<uint32_t*>(states + ((size_t)bh * nrows + row0 + row) * DD + col0 + 64 * cgrp + 2 * r) = v;
      }
    }
}

// A row's state on its way from memory into an LDS matrix of D rows with row stride STR, by NT threads.
template <int D, int NT = 256>
struct StateRows {
  static constexpr int NCH = D * D / 8 / NT;
  static_assert(D * D / 8 % NT == 0 && NT >= D, "state does not divide among the threads");
  i16x8_t x[NCH];
  float z;
  __device__ __forceinline__ void fetch(const uint16_t* states, const float* zstates, size_t row, int tid) {
    const __amdgpu_buffer_rsrc_t rs = make_rsrc(states + row * D * D, 2 * D * D);        // (the pieces share one offset register)
#pragma unroll
    for (int c = 0; c < NCH; ++c) x[c] = buf_load_b128(rs, 16u * (uint32_t)(tid + NT * c));
    z = tid < D ? zstates[row * D + tid] : 0.f;
  }
  template <int STR>
  __device__ __forceinline__ void park(uint16_t* sH, int tid) const {
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
      const int idx = (tid + NT * c) * 8;
      *reinterpret_cast<i16x8_t*>(&sH[idx / D * STR + idx % D]) = x[c];
    }
  }
};

// 32 contiguous rows of which rows_valid (possibly none) are there, through a buffer descriptor: the others read as zero and are not
// written, without a branch, and a lane's pieces share one offset.
template <int D>
struct ContiguousRows {
  __amdgpu_buffer_rsrc_t rs;
  uint32_t at;
  __device__ __forceinline__ ContiguousRows(const uint16_t* rows, int rows_valid, int lane)
      : rs(make_rsrc(rows, (uint32_t)max(rows_valid, 0) * D * 2u)), at(16u * (uint32_t)lane) {}
  __device__ __forceinline__ TileRows<D> fetch() const {
    TileRows<D> t;
#pragma unroll
    for (int i = 0; i < TileRows<D>::N; ++i) t.x[i] = buf_load_b128(rs, at + 1024u * i);
    return t;
  }
  __device__ __forceinline__ void store(const TileRows<D>& t) const {
#pragma unroll
    for (int i = 0; i < TileRows<D>::N; ++i)
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, t.x[i]), rs, (int)(at + 1024u * i), 0, 0);
  }
};

// A tile packed to 16 bit in accumulator order (word 2 h + i of w[dt][c2]: columns 32 dt + 16 c2 + 8 h + 4 g + 2 i ..), by way
// of the wave's staging tile to its rows; with `add` old's rows are added to the rounded values.
template <typename E, int D>
static __device__ __forceinline__ void store_packed_tile(uint16_t* stage, const i32x4_t (&w)[D / 32][2],
                                                         const ContiguousRows<D>& rows, int lane, bool add,
                                                         const TileRows<D>& old) {
  const int g = lane >> 5, r = lane & 31;
#pragma unroll
  for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
    for (int i4 = 0; i4 < 4; ++i4)
      *reinterpret_cast<i32x2_t*>(&stage[r * TileRows<D>::SSTR + 32 * dt + 8 * i4 + 4 * g]) =
          i32x2_t{w[dt][i4 >> 1][2 * (i4 & 1)], w[dt][i4 >> 1][2 * (i4 & 1) + 1]};
  wave_lds_fence();
  TileRows<D> t;
  t.unpark(stage, lane);
  if (add) t.template add<E>(old);
  rows.store(t);
  wave_lds_fence();
}

// The staging tile in accumulator order, as floats
template <typename E, int D>
static __device__ __forceinline__ void read_acc_tile(const uint16_t* stage, float (&x)[D / 32][16], int lane) {
  const int g = lane >> 5, r = lane & 31;
#pragma unroll
  for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
    for (int i4 = 0; i4 < 4; ++i4) {
      const i16x4_t w = *reinterpret_cast<const i16x4_t*>(&stage[r * TileRows<D>::SSTR + 32 * dt + 8 * i4 + 4 * g]);
#pragma unroll
      for (int j = 0; j < 4; ++j) x[dt][4 * i4 + j] = E::to_float((uint16_t)w[j]);
    }
  wave_lds_fence();
}

template <typename E>
static __device__ __forceinline__ i32x4_t pack_half(const float (&x)[16], int c2) {
  i32x4_t w;
#pragma unroll
  for (int j = 0; j < 4; ++j) w[j] = (int)E::pack2(x[8 * c2 + 2 * j], x[8 * c2 + 2 * j + 1]);
  return w;
}

// The output kernel and the backward's two are bound by latency: a workgroup waits for its state and rows, and what hides that is
// other workgroups on the compute unit.  So every wave has 32 rows, the registers allow two waves per SIMD, and the state's buffer is
// all the LDS there is: rows pass through it on their way into operand order before the state takes it, and on their way out when
// the last wave is done with the state; W comes in operand order from memory.  Four workgroups of 64 rows fit a compute unit (two
// before, with half of each one's waves idle in the products): at 12 heads x 16380 x 128 out 79 -> 56 us, rows 110 -> 97, kv 113 -> 75;
// the whole backward, adding to existing gradients, 386 -> 357 us there, with 128-row blocks 328 -> 301, at 24 heads x 10000 x 64
// 200 -> 159 and 187 -> 150.  No spills in bf16; in half precision at head dim 128, whose feature map and conversions hold more at a
// time, the compiler keeps 13 registers of the rows' kernel and 17 of the keys' in scratch memory.

// 1-D grid over (head, query block), XCD-aware order, one wave per 32 query rows.  wo: W in operand order.
template <typename Tag, int D, int BLKQ>
__global__ __launch_bounds__(BLKQ * 2) __attribute__((amdgpu_waves_per_eu(2, 2))) void complement_out_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ states, const float* __restrict__ zstates,
    const uint16_t* __restrict__ wo, const float* __restrict__ bias, const uint16_t* __restrict__ residual,
    uint16_t* __restrict__ out, int L, int Mblk, int fmap, int total) {
  using E = Elem<Tag>;
  constexpr int DC = D / 16;
  constexpr int DT = D / 32;
  constexpr int STR = TileRows<D>::SSTR;
  __shared__ __attribute__((aligned(16))) uint16_t sH[(D > BLKQ ? D : BLKQ) * STR];    // staging tiles, H_i^T [d2][d1], staging tiles
  __shared__ float sZ[D], sBias[D];

  const int logical = xcd_remap(blockIdx.x, gridDim.x, total);
  if (logical < 0) return;
  const int bh = __builtin_amdgcn_readfirstlane(logical / Mblk), mb = logical - bh * Mblk;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 5, r = lane & 31;
  const int row0 = mb * BLKQ + wave * 32;
  const int rows_valid = __builtin_amdgcn_readfirstlane(min(32, L - row0));             // (rows past L read as zero and are not written)
  const size_t toff = first_lane64(((size_t)bh * L + row0) * D);
  const auto rows_of = [&](const uint16_t* x, bool there = true) __attribute__((always_inline)) {
    return ContiguousRows<D>(x + toff, there ? rows_valid : 0, lane);
  };
  uint16_t* const stage = sH + wave * 32 * STR;

  i16x8_t xq[DC];                        // q in B-operand order (d = 16c + 8g + j)
  StateRows<D, BLKQ * 2> h;
  {
    const TileRows<D> qt = rows_of(q).fetch();
    h.fetch(states, zstates, (size_t)bh * Mblk + mb, tid);
    qt.park(stage, lane);
#pragma unroll
    for (int c = 0; c < DC; ++c) xq[c] = *reinterpret_cast<const i16x8_t*>(&stage[r * STR + 16 * c + 8 * g]);
  }
  __syncthreads();                       // the tiles have been read: the buffer takes H_i^T
  h.template park<STR>(sH, tid);
  if (tid < D) sZ[tid] = round16<Tag>(h.z);
  if (tid < D) sBias[tid] = round16<Tag>(bias[tid]);
  const TileRows<D> res = rows_of(residual, residual != nullptr).fetch();
  __syncthreads();                       // H_i^T, z_i visible

  i16x8_t qf[DC];
  float den = phi_pack_den<Tag, DC>(fmap, xq, qf, [&](int c, int j) { return sZ[16 * c + 8 * g + j]; });
  den += __shfl_xor(den, 32);
  den = round16<Tag>(1e-5f + round16<Tag>(den));
  const float inv_den = 1.0f / den;

  // N^T = H_i^T phi(Q)^T ; Y^T = round(round(N^T) / den) packed straight into B-operand fragments
  i16x8_t yf[DT][2];
#pragma unroll
  for (int t = 0; t < DT; ++t) {
    f32x16_t nacc;
#pragma unroll
    for (int i = 0; i < 16; ++i) nacc[i] = 0.f;
#pragma unroll
    for (int c = 0; c < DC; ++c)
      nacc = E::mfma32(*reinterpret_cast<const i16x8_t*>(&sH[(32 * t + r) * STR + 16 * c + 8 * g]), qf[c], nacc);
#pragma unroll
    for (int c2 = 0; c2 < 2; ++c2) {
      i32x4_t pw;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        pw[j] = (int)E::pack2(round16<Tag>(nacc[8 * c2 + 2 * j]) * inv_den, round16<Tag>(nacc[8 * c2 + 2 * j + 1]) * inv_den);
      yf[t][c2] = __builtin_bit_cast(i16x8_t, pw);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  // OUT^T = W Y^T : contraction chunk (t, c2) covers d2 = 32t + 16c2 .. +15 in slot order
  i32x4_t op[DT][2];
#pragma unroll
  for (int et = 0; et < DT; ++et) {
    f32x16_t oacc;
#pragma unroll
    for (int i = 0; i < 16; ++i) oacc[i] = 0.f;
#pragma unroll
    for (int c = 0; c < DC; ++c)
      oacc = E::mfma32(*reinterpret_cast<const i16x8_t*>(wo + ((et * DC + c) * 64 + lane) * 8), yf[c >> 1][c & 1], oacc);
    float y[16];
#pragma unroll
    for (int i4 = 0; i4 < 4; ++i4)
#pragma unroll
      for (int j = 0; j < 4; ++j) y[4 * i4 + j] = oacc[4 * i4 + j] + sBias[32 * et + 8 * i4 + 4 * g + j];
#pragma unroll
    for (int c2 = 0; c2 < 2; ++c2) op[et][c2] = pack_half<E>(y, c2);
  }
  __syncthreads();                       // H_i^T consumed: the buffer holds staging tiles again
  store_packed_tile<E, D>(stage, op, rows_of(out), lane, residual != nullptr, res);
}

// ---- backward ----------------------------------------------------------------------------
// With a = phi(q), c = phi(k), the states h_j, z_j, H_i, z_i as above, n = a H_i, den = 1e-5 + a . z_i, y = n / den,
// out = y W^T + b and G = d(out):
//   db = sum G ; dW = G^T y ; dy = G W ; dn = dy / den ; dden = -sum_d(dy * y) / den
//   da = dn H_i^T + dden z_i ; dq = phi'(q) da
//   dH_i = a_i^T dn_i (rows of query block i), dz_i = sum_rows dden a
//   G_j = sum_{i : j not in S_i} dH_i = sum_i dH_i - sum_{i in C_j} dH_i  (C_j = query blocks that selected j), gz_j likewise
//   dc = v G_j^T + gz_j ; dv = c G_j ; dk = phi'(k) dc                     (rows of key block j)
// Kernels (the per-block products and dW / db reuse kernels of the forward and of the global backward):
//   rows   : one workgroup per query block: y, dy, dn, dden, da, dq for its rows from the forward's H_i, z_i on the MFMA in
//            transposed form; writes dq and the row-wise temporaries dn, y (16 bit), dden
//   states : the forward's kernel, with the map's columns as weights: G_j, gz_j
//   kv     : one workgroup per key block: dv, dc, dk for its 64 rows

// 1-D grid over (head, query block), XCD-aware order, one wave per 32 query rows.  wt: W^T in operand order.
template <typename Tag, int D, int BLKQ>
__global__ __launch_bounds__(BLKQ * 2) __attribute__((amdgpu_waves_per_eu(2, 2))) void complement_bwd_rows_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ gout, const uint16_t* __restrict__ states,
    const float* __restrict__ zstates, const uint16_t* __restrict__ wt, uint16_t* __restrict__ dq, uint16_t* __restrict__ dn_out,
    uint16_t* __restrict__ y_out, float* __restrict__ dden_out, int L, int Mblk, int fmap, int total, int accumulate) {
  using E = Elem<Tag>;
  constexpr int DC = D / 16;
  constexpr int DT = D / 32;
  constexpr int HSTR = D + 16;           // H_i^T is read row-wise (n^T = H^T a^T) and transposed (da^T = H dn^T)
  constexpr int XSTR = TileRows<D>::SSTR;
  constexpr int SIZE = D * HSTR > BLKQ * XSTR ? D * HSTR : BLKQ * XSTR;
  __shared__ __attribute__((aligned(16))) uint16_t sHT[SIZE];    // staging tiles (q, then G), H_i^T [d2][d1], staging tiles (out)
  __shared__ float sZ[D];

  const int logical = xcd_remap(blockIdx.x, gridDim.x, total);
  if (logical < 0) return;
  const int bh = __builtin_amdgcn_readfirstlane(logical / Mblk), mb = logical - bh * Mblk;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 5, r = lane & 31;
  const int row0 = mb * BLKQ + wave * 32;
  const int rows_valid = __builtin_amdgcn_readfirstlane(min(32, L - row0));             // (rows past L read as zero and are not written)
  const int qrow = row0 + r;
  const size_t toff = first_lane64(((size_t)bh * L + row0) * D);
  const auto rows_of = [&](const uint16_t* x, bool there = true) __attribute__((always_inline)) {
    return ContiguousRows<D>(x + toff, there ? rows_valid : 0, lane);
  };
  uint16_t* const stage = sHT + wave * 32 * XSTR;

  // q and G in B-operand order (d = 16c + 8g + j)
  i16x8_t qx[DC], gf[DC];
  StateRows<D, BLKQ * 2> h;
  {
    const TileRows<D> qt = rows_of(q).fetch(), gt = rows_of(gout).fetch();
    h.fetch(states, zstates, (size_t)bh * Mblk + mb, tid);
    qt.park(stage, lane);
#pragma unroll
    for (int c = 0; c < DC; ++c) qx[c] = *reinterpret_cast<const i16x8_t*>(&stage[r * XSTR + 16 * c + 8 * g]);
    wave_lds_fence();
    gt.park(stage, lane);
#pragma unroll
    for (int c = 0; c < DC; ++c) gf[c] = *reinterpret_cast<const i16x8_t*>(&stage[r * XSTR + 16 * c + 8 * g]);
  }
  __syncthreads();                       // the tiles have been read: the buffer takes H_i^T
  h.template park<HSTR>(sHT, tid);
  if (tid < D) sZ[tid] = round16<Tag>(h.z);
  __syncthreads();                       // H_i^T, z_i visible

  // dy^T = W^T G^T
  float yv[DT][16], dnv[DT][16];
#pragma unroll
  for (int t = 0; t < DT; ++t) {
    f32x16_t acc;
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = 0.f;
#pragma unroll
    for (int c = 0; c < DC; ++c)
      acc = E::mfma32(*reinterpret_cast<const i16x8_t*>(wt + ((t * DC + c) * 64 + lane) * 8), gf[c], acc);
#pragma unroll
    for (int i = 0; i < 16; ++i) dnv[t][i] = acc[i];
    __builtin_amdgcn_sched_barrier(0);
  }
  // a = phi(q) as B operand and the divisor
  i16x8_t af[DC];
  float row_mx = 0.f, row_inv = 1.f, inv_den;
  {
    float f[DC][8];
#pragma unroll
    for (int c = 0; c < DC; ++c)
#pragma unroll
      for (int j = 0; j < 8; ++j) f[c][j] = E::to_float((uint16_t)qx[c][j]);
    phi_row_pair<Tag, DC>(fmap, f, row_mx, row_inv);
    float den = 0.f;
#pragma unroll
    for (int c = 0; c < DC; ++c) {
      i32x4_t pw;
#pragma unroll
      for (int j = 0; j < 8; ++j) den += f[c][j] * sZ[16 * c + 8 * g + j];
#pragma unroll
      for (int j = 0; j < 4; ++j) pw[j] = (int)E::pack2(f[c][2 * j], f[c][2 * j + 1]);
      af[c] = __builtin_bit_cast(i16x8_t, pw);
    }
    den += __shfl_xor(den, 32);
    den += 1e-5f;
    inv_den = 1.0f / den;
  }
  // y^T = (H_i^T a^T) / den
#pragma unroll
  for (int t = 0; t < DT; ++t) {
    f32x16_t acc;
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = 0.f;
#pragma unroll
    for (int c = 0; c < DC; ++c)
      acc = E::mfma32(*reinterpret_cast<const i16x8_t*>(&sHT[(32 * t + r) * HSTR + 16 * c + 8 * g]), af[c], acc);
#pragma unroll
    for (int i = 0; i < 16; ++i) yv[t][i] = acc[i];
    __builtin_amdgcn_sched_barrier(0);
  }

  float dden = 0.f;
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      yv[t][i] *= inv_den;
      dden += dnv[t][i] * yv[t][i];
      dnv[t][i] *= inv_den;          // dn^T
    }
  dden += __shfl_xor(dden, 32);
  dden = -dden * inv_den;
  if (qrow < L && g == 0) dden_out[(size_t)bh * L + qrow] = dden;

  // dn^T as B operand: register 8c2+j of tile t is d2 = 32t + 16c2 + 8(j/4) + 4g + j%4
  i32x4_t dnp[DT][2], yp[DT][2];
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int c2 = 0; c2 < 2; ++c2) {
      dnp[t][c2] = pack_half<E>(dnv[t], c2);
      yp[t][c2] = pack_half<E>(yv[t], c2);
    }

  // da^T = H_i dn^T + z_i dden: rows d1 of H_i come out of H_i^T through the transposing read, the contraction
  // index d2 in the slot order of dn^T above
  const int tr_row = (lane & 15) >> 2;
  const int tr_col = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
  float da[DT][16];
#pragma unroll
  for (int t1 = 0; t1 < DT; ++t1) {
    f32x16_t acc;
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = 0.f;
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int c2 = 0; c2 < 2; ++c2) {
        const uint16_t* p0 = &sHT[(16 * (2 * t + c2) + 4 * g + tr_row) * HSTR + 32 * t1 + tr_col];
        acc = E::mfma32(concat4(lds_read_tr16(p0), lds_read_tr16(p0 + 8 * HSTR)), __builtin_bit_cast(i16x8_t, dnp[t][c2]), acc);
      }
#pragma unroll
    for (int i4 = 0; i4 < 4; ++i4) {
      const int d0 = 32 * t1 + 8 * i4 + 4 * g;
#pragma unroll
      for (int j = 0; j < 4; ++j) da[t1][4 * i4 + j] = acc[4 * i4 + j] + sZ[d0 + j] * dden;
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  // (q again, in accumulator order, for the gradient through phi: from L2, and no registers held through the products)
  const TileRows<D> again = rows_of(q).fetch();
  __syncthreads();                       // H_i^T consumed: the buffer holds staging tiles again
  int lane_e = lane;
  asm volatile("" : "+v"(lane_e));       // (addresses are formed again: none is worth a register through the products)
  store_packed_tile<E, D>(stage, dnp, rows_of(dn_out), lane_e, false, again);
  store_packed_tile<E, D>(stage, yp, rows_of(y_out), lane_e, false, again);
  again.park(stage, lane_e);
  const TileRows<D> old = rows_of(dq, accumulate).fetch();
  float xq[DT][16];
  read_acc_tile<E, D>(stage, xq, lane_e);
  phi_backward<DT>(fmap, xq, da, row_mx, row_inv);
  i32x4_t dqp[DT][2];
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int c2 = 0; c2 < 2; ++c2) dqp[t][c2] = pack_half<E>(da[t], c2);
  store_packed_tile<E, D>(stage, dqp, rows_of(dq), lane_e, accumulate, old);
}

// 1-D grid over (head, key block), XCD-aware order, two waves of 32 key rows.
// states: per key block G_j^T [d2][d1] (16 bit), zstates: gz_j (fp32).
template <typename Tag, int D>
__global__ __launch_bounds__(128) __attribute__((amdgpu_waves_per_eu(2, 2))) void complement_bwd_kv_kernel(
    const uint16_t* __restrict__ k, const uint16_t* __restrict__ v, const uint16_t* __restrict__ states,
    const float* __restrict__ zstates, uint16_t* __restrict__ dk, uint16_t* __restrict__ dv, int L, int N, int fmap, int total,
    int accumulate) {
  using E = Elem<Tag>;
  constexpr int DC = D / 16;
  constexpr int DT = D / 32;
  constexpr int GSTR = D + 16;           // G_j^T is read row-wise (dv^T = G^T c^T) and transposed (dc^T = G v^T)
  constexpr int SSTR = TileRows<D>::SSTR;
  static_assert(64 * SSTR <= D * GSTR, "staging tiles exceed the state buffer");
  __shared__ __attribute__((aligned(16))) uint16_t sGT[D * GSTR];      // staging tiles (k, then v), G_j^T [d2][d1], staging tiles
  __shared__ float sGZ[D];

  const int logical = xcd_remap(blockIdx.x, gridDim.x, total);
  if (logical < 0) return;
  const int bh = __builtin_amdgcn_readfirstlane(logical / N), nb = logical - bh * N;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 5, r = lane & 31;
  const int row0 = nb * 64 + wave * 32;
  const int rows_valid = __builtin_amdgcn_readfirstlane(min(32, L - row0));             // (rows past L read as zero and are not written)
  const size_t toff = first_lane64(((size_t)bh * L + row0) * D);
  const auto rows_of = [&](const uint16_t* x, bool there = true) __attribute__((always_inline)) {
    return ContiguousRows<D>(x + toff, there ? rows_valid : 0, lane);
  };
  uint16_t* const stage = sGT + wave * 32 * SSTR;
  i16x8_t kx[DC], vf[DC];
  StateRows<D, 128> h;
  {
    const TileRows<D> kt = rows_of(k).fetch(), vt = rows_of(v).fetch();
    h.fetch(states, zstates, (size_t)bh * N + nb, tid);
    kt.park(stage, lane);
#pragma unroll
    for (int c = 0; c < DC; ++c) kx[c] = *reinterpret_cast<const i16x8_t*>(&stage[r * SSTR + 16 * c + 8 * g]);
    wave_lds_fence();
    vt.park(stage, lane);
#pragma unroll
    for (int c = 0; c < DC; ++c) vf[c] = *reinterpret_cast<const i16x8_t*>(&stage[r * SSTR + 16 * c + 8 * g]);
  }
  __syncthreads();                       // the tiles have been read: the buffer takes G_j^T
  h.template park<GSTR>(sGT, tid);
  if (tid < D) sGZ[tid] = h.z;
  __syncthreads();

  float row_mx, row_inv;
  i32x4_t dvp[DT][2];
  {
    // dv^T = G^T c^T
    float f[DC][8];
#pragma unroll
    for (int c = 0; c < DC; ++c)
#pragma unroll
      for (int j = 0; j < 8; ++j) f[c][j] = E::to_float((uint16_t)kx[c][j]);
    phi_row_pair<Tag, DC>(fmap, f, row_mx, row_inv);
    i16x8_t cf[DC];
#pragma unroll
    for (int c = 0; c < DC; ++c) {
      i32x4_t pw;
#pragma unroll
      for (int j = 0; j < 4; ++j) pw[j] = (int)E::pack2(f[c][2 * j], f[c][2 * j + 1]);
      cf[c] = __builtin_bit_cast(i16x8_t, pw);
    }
#pragma unroll
    for (int t = 0; t < DT; ++t) {
      f32x16_t vacc;
#pragma unroll
      for (int i = 0; i < 16; ++i) vacc[i] = 0.f;
#pragma unroll
      for (int c = 0; c < DC; ++c) {
        const i16x8_t a2 = *reinterpret_cast<const i16x8_t*>(&sGT[(32 * t + r) * GSTR + 16 * c + 8 * g]);
        vacc = E::mfma32(a2, cf[c], vacc);
      }
      float dvv[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) dvv[i] = vacc[i];
#pragma unroll
      for (int c2 = 0; c2 < 2; ++c2) dvp[t][c2] = pack_half<E>(dvv, c2);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  // dc^T = G v^T + gz ; dk = phi'(k) dc  (rows d1 of G through the transposing read, d2 in the order of v's fragments)
  const int tr_row = (lane & 15) >> 2;
  const int tr_col = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
  float dc[DT][16];
#pragma unroll
  for (int t = 0; t < DT; ++t) {
    f32x16_t acc;
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = 0.f;
#pragma unroll
    for (int c = 0; c < DC; ++c) {
      const uint16_t* pa = &sGT[(16 * c + 8 * g + tr_row) * GSTR + 32 * t + tr_col];
      acc = E::mfma32(concat4(lds_read_tr16(pa), lds_read_tr16(pa + 4 * GSTR)), vf[c], acc);
    }
#pragma unroll
    for (int i4 = 0; i4 < 4; ++i4) {
      const int d0 = 32 * t + 8 * i4 + 4 * g;
#pragma unroll
      for (int j = 0; j < 4; ++j) dc[t][4 * i4 + j] = acc[4 * i4 + j] + sGZ[d0 + j];
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  const TileRows<D> again = rows_of(k).fetch();       // (k again, in accumulator order, as q above)
  const TileRows<D> old_v = rows_of(dv, accumulate).fetch();
  __syncthreads();                       // G_j^T consumed: the buffer holds staging tiles again
  int lane_e = lane;
  asm volatile("" : "+v"(lane_e));       // (addresses are formed again: none is worth a register through the products)
  store_packed_tile<E, D>(stage, dvp, rows_of(dv), lane_e, accumulate, old_v);
  again.park(stage, lane_e);
  const TileRows<D> old_k = rows_of(dk, accumulate).fetch();
  float xk[DT][16];
  read_acc_tile<E, D>(stage, xk, lane_e);
  phi_backward<DT>(fmap, xk, dc, row_mx, row_inv);
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int c2 = 0; c2 < 2; ++c2) dvp[t][c2] = pack_half<E>(dc[t], c2);
  store_packed_tile<E, D>(stage, dvp, rows_of(dk), lane_e, accumulate, old_k);
}

// ---- host ---------------------------------------------------------------------------------
struct ComplWs {
  size_t hblk, zblk, w, all, wo, total;                  // total: without the query blocks' states
};
// The query blocks' states: what the backward reads of the forward.
struct ComplStates {
  size_t h, z, total;
};
static ComplStates compl_states(int BH, int L, int D, int BLKQ) {
  const int64_t M = cdiv(L, BLKQ);
  ComplStates w;
  w.h = 0;
  w.z = align_up((int64_t)BH * M * D * D * 2, 256);
  w.total = w.z + align_up((int64_t)BH * M * D * 4, 256);
  return w;
}
int64_t linear_complement_states_bytes(int BH, int L, int D, int BLKQ) { return (int64_t)compl_states(BH, L, D, BLKQ).total; }
static ComplWs compl_ws(int BH, int L, int D) {
  const int64_t N = cdiv(L, 64);
  ComplWs w;
  size_t off = 0;
  w.hblk = off; off += align_up((int64_t)BH * N * D * D * 2, 256);
  w.zblk = off; off += align_up((int64_t)BH * N * D * 4, 256);
  // (weights of up to N rows over up to N blocks: the backward's take the place of the forward's)
  w.w = off;    off += align_up(BH * weight_words((int)N, (int)N) * 4, 256);
  w.all = off;  off += align_up((int64_t)BH * N * 4, 256);
  w.wo = off;   off += align_up((int64_t)D * D * 2, 256);
  w.total = off;
  return w;
}
// A call that does not keep the query blocks' states (twice the bytes of q at 64-row blocks and head dim 128) forms them for a
// few heads at a time, in up to CPL_STATES_AT_ONCE bytes, so that short problems stay one launch.
// 40 heads x 75600 x 128: 1.57 GiB of workspace (all at once 3.0), in 14 groups.
constexpr int64_t CPL_STATES_AT_ONCE = 128ll << 20;
struct ComplGroups {
  int heads;             // per group
  size_t extra;          // bytes their states add behind the rest of the workspace
};
static ComplGroups compl_groups(int BH, int L, int D, int BLKQ) {
  const size_t room = (size_t)CPL_STATES_AT_ONCE, one = compl_states(1, L, D, BLKQ).total;
  ComplGroups g;
  g.heads = (int)(room / one < 1 ? 1 : room / one > (size_t)BH ? BH : room / one);
  g.heads = cdiv(BH, cdiv(BH, g.heads));                    // (even groups)
  g.extra = compl_states(g.heads, L, D, BLKQ).total;
  return g;
}
int64_t linear_complement_apart_bytes(int BH, int L, int D) { return (int64_t)compl_ws(BH, L, D).total; }
int64_t linear_complement_workspace_bytes(int BH, int L, int D, int BLKQ) {
  return (int64_t)(compl_ws(BH, L, D).total + compl_groups(BH, L, D, BLKQ).extra);
}

// The states of nrows rows of every head from its nblk block states (see complement_states_kernel)
template <typename Tag, int D>
static void launch_states(const uint16_t* blocks, const float* zblocks, const uint32_t* w, const int* all, uint16_t* states,
                          float* zstates, int BH, int nrows, int nblk, hipStream_t st) {
#define SLA_STATES_LAUNCH(RW)                                                                                                \
  do {                                                                                                                     \
    const int units = BH * (D / 32 + D * D / (256 / RW)) * cdiv(nrows, 128 * RW);                                          \
    hipLaunchKernelGGL((complement_states_kernel<Tag, D, RW>), dim3(xcd_grid(units)), dim3(256), 0, st, blocks, zblocks,   \
                       w, all, states, zstates, nrows, nblk, units);                                                      \
  } while (0)
  // (twice the rows and half the values per workgroup: every block state is fetched for half as many tiles of rows.  Forward and
  //  backward of the branch, one / two: 12 heads x 32760 x 128, 512 rows, 975 / 948 us, 4 x 75600 x 128, 1182 rows, 967 / 950, 16 x
  //  30000 x 64, 469 rows, 427 / 419.  Up to 256 rows the two tiles run side by side and share what they fetch in L2: 12 x 16380 x 128,
  //  256 rows, 490 / 492, with 128-row blocks 407 / 411, 2 x 12000 x 128, 188 rows, 128 / 132)
  if (nrows > 256) SLA_STATES_LAUNCH(2);
  else SLA_STATES_LAUNCH(1);
#undef SLA_STATES_LAUNCH
}

// Block states.
template <typename Tag, int D>
static void complement_blocks_run(const void* k, const void* v, int fmap, int BH, int L, char* ws, hipStream_t st) {
  const ComplWs w = compl_ws(BH, L, D);
  hipLaunchKernelGGL((linear_state_partial_kernel<Tag, D, true>), dim3(cdiv(L, 64), BH), dim3(256), 0, st, (const uint16_t*)k,
                     (const uint16_t*)v, contiguous_layout(BH, L, D), (void*)(ws + w.hblk), (float*)(ws + w.zblk), L, 64, fmap,
                     (const float*)nullptr);
}

// The query blocks' states of `heads` heads from head h0 on, laid out as compl_states(heads, ..) says, and with `weight` its operand.
template <typename Tag, int D>
static void complement_states_run(const void* lut, int lut64, int BH, int L, int BLKQ, int topk, char* ws, int h0, int heads,
                                  char* states, const float* weight, hipStream_t st) {
  const ComplWs w = compl_ws(BH, L, D);
  const ComplStates s = compl_states(heads, L, D, BLKQ);
  const int N = cdiv(L, 64), M = cdiv(L, BLKQ);
  const size_t head = h0;
  uint32_t* const wt = (uint32_t*)(ws + w.w);
  int* const all = (int*)(ws + w.all);
  hipLaunchKernelGGL((complement_row_weights_kernel<Tag>), dim3(M, heads), dim3(64), 0, st,
                     lut ? (const char*)lut + head * M * topk * (lut64 ? 8 : 4) : nullptr, lut64, topk, wt, all, N, weight,
                     (uint16_t*)(ws + w.wo), D);
  launch_states<Tag, D>((const uint16_t*)(ws + w.hblk) + head * N * D * D, (const float*)(ws + w.zblk) + head * N * D, wt, all,
                        (uint16_t*)(states + s.h), (float*)(states + s.z), heads, M, N, st);
}

// (kept: where the caller wants every head's states; null: they are formed in the workspace, a group of heads at a time)
template <typename Tag, int D, int BLKQ>
static int complement_impl(const void* q, const void* k, const void* v, const void* lut, int lut64, const float* weight,
                           const float* bias, const void* residual, void* out, int fmap, int BH, int L, int topk, char* ws,
                           char* kept, hipStream_t st) {
  const int Mblk = cdiv(L, BLKQ);
  complement_blocks_run<Tag, D>(k, v, fmap, BH, L, ws, st);
  const ComplGroups g = compl_groups(BH, L, D, BLKQ);
  const int step = kept ? BH : g.heads;
  char* const states = kept ? kept : ws + compl_ws(BH, L, D).total;
  for (int h0 = 0; h0 < BH; h0 += step) {
    const int heads = BH - h0 < step ? BH - h0 : step;
    const ComplStates s = compl_states(heads, L, D, BLKQ);
    const size_t rows = (size_t)h0 * L * D;
    complement_states_run<Tag, D>(lut, lut64, BH, L, BLKQ, topk, ws, h0, heads, states, h0 == 0 ? weight : nullptr, st);
    const int total = heads * Mblk;
    hipLaunchKernelGGL((complement_out_kernel<Tag, D, BLKQ>), dim3(xcd_grid(total)), dim3(BLKQ * 2), 0, st, (const uint16_t*)q + rows,
                       (const uint16_t*)(states + s.h), (const float*)(states + s.z), (const uint16_t*)(ws + compl_ws(BH, L, D).wo), bias,
                       residual ? (const uint16_t*)residual + rows : nullptr, (uint16_t*)out + rows, L, Mblk, fmap, total);
  }
  return check_launch("linear_complement_fwd");
}

// ---- backward, host -------------------------------------------------------------------------
struct ComplBwdWs {
  ComplWs fwd;
  size_t wt, dn, y, dden, dhblk, dzblk, wg, total;
};
static ComplBwdWs compl_bwd_ws(int BH, int L, int D, int BLKQ) {
  const int64_t M = cdiv(L, BLKQ);
  ComplBwdWs w;
  w.fwd = compl_ws(BH, L, D);
  size_t off = w.fwd.total;
  w.wt = off;    off += align_up((int64_t)D * D * 2, 256);
  w.dn = off;    off += align_up((int64_t)BH * L * D * 2, 256);
  w.y = off;     off += align_up((int64_t)BH * L * D * 2, 256);
  w.dden = off;  off += align_up((int64_t)BH * L * 4, 256);
  w.dhblk = off; off += align_up((int64_t)BH * M * D * D * 2, 256);
  w.dzblk = off; off += align_up((int64_t)BH * M * D * 4, 256);
  w.wg = off;    off += align_up(weight_grads_workspace_bytes(BH, L, D), 256);
  w.total = off;
  return w;
}
int64_t linear_complement_bwd_apart_bytes(int BH, int L, int D, int BLKQ) { return (int64_t)compl_bwd_ws(BH, L, D, BLKQ).total; }
int64_t linear_complement_bwd_workspace_bytes(int BH, int L, int D, int BLKQ) {
  return (int64_t)(compl_bwd_ws(BH, L, D, BLKQ).total + compl_groups(BH, L, D, BLKQ).extra);
}

template <typename Tag, int D, int BLKQ>
static int complement_bwd_impl(const void* q, const void* k, const void* v, const int8_t* sparse_map, const void* lut, int lut64,
                               const float* weight, const void* d_out, void* dq, void* dk, void* dv, float* d_weight,
                               float* d_bias, int dtype, int fmap, int BH, int L, int topk, int accumulate, char* ws,
                               const char* kept, hipStream_t st) {
  const ComplBwdWs w = compl_bwd_ws(BH, L, D, BLKQ);
  const int N = cdiv(L, 64), Mblk = cdiv(L, BLKQ);
  const RowLayout lay = contiguous_layout(BH, L, D);
  // (the forward's block states are done with when the key blocks' take their place)
  uint16_t* gst = (uint16_t*)(ws + w.fwd.hblk);
  float* gzst = (float*)(ws + w.fwd.zblk);
  uint16_t* wt = (uint16_t*)(ws + w.wt);
  uint16_t* dn = (uint16_t*)(ws + w.dn);
  uint16_t* y = (uint16_t*)(ws + w.y);
  float* dden = (float*)(ws + w.dden);
  uint16_t* dhblk = (uint16_t*)(ws + w.dhblk);
  float* dzblk = (float*)(ws + w.dzblk);
  hipLaunchKernelGGL((linear_prep_weight_kernel<Tag>), dim3(cdiv(D * D, 256)), dim3(256), 0, st, weight, wt, D);
  // rows: dq and the row temporaries (with the forward's states, kept or formed again)
  if (!kept) complement_blocks_run<Tag, D>(k, v, fmap, BH, L, ws, st);
  const ComplGroups g = compl_groups(BH, L, D, BLKQ);
  const int step = kept ? BH : g.heads;
  for (int h0 = 0; h0 < BH; h0 += step) {
    const int heads = BH - h0 < step ? BH - h0 : step;
    const ComplStates s = compl_states(heads, L, D, BLKQ);
    const size_t rows = (size_t)h0 * L * D;
    if (!kept) complement_states_run<Tag, D>(lut, lut64, BH, L, BLKQ, topk, ws, h0, heads, ws + w.total, nullptr, st);
    const char* const states = kept ? kept : ws + w.total;
    const int total_q = heads * Mblk;
    hipLaunchKernelGGL((complement_bwd_rows_kernel<Tag, D, BLKQ>), dim3(xcd_grid(total_q)), dim3(BLKQ * 2), 0, st,
                       (const uint16_t*)q + rows, (const uint16_t*)d_out + rows, (const uint16_t*)(states + s.h),
                       (const float*)(states + s.z), wt, (uint16_t*)dq + rows, dn + rows, y + rows, dden + (size_t)h0 * L, L, Mblk,
                       fmap, total_q, accumulate);
  }
  // per query block dH_i^T = (a_i^T dn_i)^T and dz_i = sum dden a (the state kernel with q, dn in the place of k, v)
  hipLaunchKernelGGL((linear_state_partial_kernel<Tag, D, true, true>), dim3(Mblk, BH), dim3(256), 0, st, (const uint16_t*)q,
                     (const uint16_t*)dn, lay, (void*)dhblk, dzblk, L, BLKQ, fmap, (const float*)dden);
  // dW, db of every head
  const HeadSums heads = launch_weight_grads(dtype, D, d_out, y, BH, L, ws + w.wg, d_weight, d_bias, st);
  // their sum; dk, dv
  uint32_t* const wk = (uint32_t*)(ws + w.fwd.w);
  int* const all = (int*)(ws + w.fwd.all);
  const int strips = cdiv(N, 64);
  hipLaunchKernelGGL(complement_column_weights_kernel, dim3(strips * BH + cdiv(heads.wgs, 8)), dim3(512), 0, st, sparse_map, wk, all,
                     Mblk, N, strips, strips * BH, heads);
  launch_states<Tag, D>(dhblk, dzblk, wk, all, gst, gzst, BH, N, Mblk, st);
  const int total_k = BH * N;
  hipLaunchKernelGGL((complement_bwd_kv_kernel<Tag, D>), dim3(xcd_grid(total_k)), dim3(128), 0, st, (const uint16_t*)k,
                     (const uint16_t*)v, gst, gzst, (uint16_t*)dk, (uint16_t*)dv, L, N, fmap, total_k, accumulate);
  return check_launch("linear_complement_bwd");
}

}  // namespace sla

using namespace sla;

static int complement_bwd_entry(const void* q, const void* k, const void* v, const int8_t* sparse_map, const void* lut,
                                int lut_elem_bytes, const float* weight, const float* bias, const void* d_out, void* dq, void* dk,
                                void* dv, float* d_weight, float* d_bias, int dtype, int fmap, int B, int H, int L, int D, int BLKQ,
                                int BLKK, int topk, int flags, void* workspace, int64_t workspace_bytes,
                                const char* states, bool apart, void* stream) {
  int rc = validate_linear(dtype, fmap, B, H, L, D);
  if (rc) return rc;
  rc = validate_attn_shape(dtype, B, H, L, D, BLKQ, BLKK, topk, lut_elem_bytes);
  if (rc) return rc;
  (void)bias;  // the bias does not enter any gradient
  SLA_REQUIRE((flags & ~SLA_BWD_ACCUMULATE) == 0, SLA_ERR_BAD_ARG, "unknown flag bits in %d", flags);
  SLA_REQUIRE(q && k && v && sparse_map && weight && d_out && dq && dk && dv && d_weight && d_bias && workspace &&
                  (lut || topk == 0),
              SLA_ERR_BAD_ARG, "null pointer");
  SLA_REQUIRE(((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)d_out | (uintptr_t)dq | (uintptr_t)dk | (uintptr_t)dv |
               (uintptr_t)weight | (uintptr_t)workspace) % 16 == 0,
              SLA_ERR_BAD_ARG, "pointers must be 16-byte aligned");
  SLA_REQUIRE(!apart || (states && (uintptr_t)states % 16 == 0), SLA_ERR_BAD_ARG, "states null or not 16-byte aligned");
  SLA_REQUIRE((int64_t)H * B <= 65535, SLA_ERR_UNSUPPORTED, "B*H exceeds 65535");
  const int BH = B * H;
  const int64_t need = apart ? linear_complement_bwd_apart_bytes(BH, L, D, BLKQ) : linear_complement_bwd_workspace_bytes(BH, L, D, BLKQ);
  SLA_REQUIRE(workspace_bytes >= need, SLA_ERR_WORKSPACE, "workspace of %lld bytes, need %lld", (long long)workspace_bytes,
              (long long)need);
  hipStream_t st = (hipStream_t)stream;
  char* ws = (char*)workspace;
  const int lut64 = lut_elem_bytes == 8;
  const int accumulate = flags & SLA_BWD_ACCUMULATE;
#define SLA_CPLB_CASE(TAG, DD, BQ)                                                                                      \
  if (D == DD && BLKQ == BQ)                                                                                            \
  return complement_bwd_impl<TAG, DD, BQ>(q, k, v, sparse_map, lut, lut64, weight, d_out, dq, dk, dv, d_weight, d_bias, \
                                          dtype, fmap, BH, L, topk, accumulate, ws, states, st)
  if (dtype == SLA_BF16) {
    SLA_CPLB_CASE(bf16_tag, 128, 64);
    SLA_CPLB_CASE(bf16_tag, 128, 128);
    SLA_CPLB_CASE(bf16_tag, 64, 64);
    SLA_CPLB_CASE(bf16_tag, 64, 128);
  } else {
    SLA_CPLB_CASE(f16_tag, 128, 64);
    SLA_CPLB_CASE(f16_tag, 128, 128);
    SLA_CPLB_CASE(f16_tag, 64, 64);
    SLA_CPLB_CASE(f16_tag, 64, 128);
  }
#undef SLA_CPLB_CASE
  set_error("unsupported D=%d BLKQ=%d", D, BLKQ);
  return SLA_ERR_UNSUPPORTED;
}

extern "C" int sla_linear_complement_bwd(const void* q, const void* k, const void* v, const int8_t* sparse_map, const void* lut,
                                         int lut_elem_bytes, const float* weight, const float* bias, const void* d_out, void* dq,
                                         void* dk, void* dv, float* d_weight, float* d_bias, int dtype, int fmap, int B, int H,
                                         int L, int D, int BLKQ, int BLKK, int topk, int flags, void* workspace,
                                         int64_t workspace_bytes, void* stream) {
  return complement_bwd_entry(q, k, v, sparse_map, lut, lut_elem_bytes, weight, bias, d_out, dq, dk, dv, d_weight, d_bias, dtype,
                              fmap, B, H, L, D, BLKQ, BLKK, topk, flags, workspace, workspace_bytes, nullptr, false, stream);
}

extern "C" int sla_linear_complement_bwd_states(const void* q, const void* k, const void* v, const int8_t* sparse_map,
                                                const void* lut, int lut_elem_bytes, const float* weight, const float* bias,
                                                const void* d_out, const void* states, void* dq, void* dk, void* dv,
                                                float* d_weight, float* d_bias, int dtype, int fmap, int B, int H, int L, int D,
                                                int BLKQ, int BLKK, int topk, int flags, void* workspace,
                                                int64_t workspace_bytes, void* stream) {
  return complement_bwd_entry(q, k, v, sparse_map, lut, lut_elem_bytes, weight, bias, d_out, dq, dk, dv, d_weight, d_bias, dtype,
                              fmap, B, H, L, D, BLKQ, BLKK, topk, flags, workspace, workspace_bytes, (const char*)states, true,
                              stream);
}

static int complement_fwd_entry(const void* q, const void* k, const void* v, const void* lut, int lut_elem_bytes,
                                const float* weight, const float* bias, const void* residual, void* out, int dtype, int fmap,
                                int B, int H, int L, int D, int BLKQ, int BLKK, int topk, void* workspace,
                                int64_t workspace_bytes, char* states, bool apart, void* stream) {
  int rc = validate_linear(dtype, fmap, B, H, L, D);
  if (rc) return rc;
  rc = validate_attn_shape(dtype, B, H, L, D, BLKQ, BLKK, topk, lut_elem_bytes);
  if (rc) return rc;
  SLA_REQUIRE(q && k && v && weight && bias && out && workspace && (lut || topk == 0), SLA_ERR_BAD_ARG, "null pointer");
  SLA_REQUIRE(((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)out | (uintptr_t)residual | (uintptr_t)weight |
               (uintptr_t)workspace) % 16 == 0,
              SLA_ERR_BAD_ARG, "pointers must be 16-byte aligned");
  SLA_REQUIRE(!apart || (states && (uintptr_t)states % 16 == 0), SLA_ERR_BAD_ARG, "states null or not 16-byte aligned");
  SLA_REQUIRE((int64_t)H * B <= 65535 && cdiv(L, BLKQ) <= 65535 * 32, SLA_ERR_UNSUPPORTED, "grid too large");
  const int BH = B * H;
  const int64_t need = apart ? linear_complement_apart_bytes(BH, L, D) : linear_complement_workspace_bytes(BH, L, D, BLKQ);
  SLA_REQUIRE(workspace_bytes >= need, SLA_ERR_WORKSPACE, "workspace of %lld bytes, need %lld", (long long)workspace_bytes,
              (long long)need);
  hipStream_t st = (hipStream_t)stream;
  char* ws = (char*)workspace;
  const int lut64 = lut_elem_bytes == 8;
#define SLA_CPL_CASE(TAG, DD, BQ) \
  if (D == DD && BLKQ == BQ)      \
  return complement_impl<TAG, DD, BQ>(q, k, v, lut, lut64, weight, bias, residual, out, fmap, BH, L, topk, ws, states, st)
  if (dtype == SLA_BF16) {
    SLA_CPL_CASE(bf16_tag, 128, 64);
    SLA_CPL_CASE(bf16_tag, 128, 128);
    SLA_CPL_CASE(bf16_tag, 64, 64);
    SLA_CPL_CASE(bf16_tag, 64, 128);
  } else {
    SLA_CPL_CASE(f16_tag, 128, 64);
    SLA_CPL_CASE(f16_tag, 128, 128);
    SLA_CPL_CASE(f16_tag, 64, 64);
    SLA_CPL_CASE(f16_tag, 64, 128);
  }
#undef SLA_CPL_CASE
  set_error("unsupported D=%d BLKQ=%d", D, BLKQ);
  return SLA_ERR_UNSUPPORTED;
}

extern "C" int sla_linear_complement_fwd(const void* q, const void* k, const void* v, const void* lut, int lut_elem_bytes,
                                         const float* weight, const float* bias, const void* residual, void* out, int dtype,
                                         int fmap, int B, int H, int L, int D, int BLKQ, int BLKK, int topk, void* workspace,
                                         int64_t workspace_bytes, void* stream) {
  return complement_fwd_entry(q, k, v, lut, lut_elem_bytes, weight, bias, residual, out, dtype, fmap, B, H, L, D, BLKQ, BLKK, topk,
                              workspace, workspace_bytes, nullptr, false, stream);
}

extern "C" int sla_linear_complement_fwd_states(const void* q, const void* k, const void* v, const void* lut, int lut_elem_bytes,
                                                const float* weight, const float* bias, const void* residual, void* out,
                                                void* states, int dtype, int fmap, int B, int H, int L, int D, int BLKQ,
                                                int BLKK, int topk, void* workspace, int64_t workspace_bytes, void* stream) {
  return complement_fwd_entry(q, k, v, lut, lut_elem_bytes, weight, bias, residual, out, dtype, fmap, B, H, L, D, BLKQ, BLKK, topk,
                              workspace, workspace_bytes, (char*)states, true, stream);
}
