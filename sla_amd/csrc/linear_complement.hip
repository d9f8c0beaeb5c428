// Linear branch over the NON-selected key blocks ("complement" mode), projection and final sum, for gfx950.
//
// The mounted reference computes the linear branch over all keys (sparse_linear_attention/core.py:92-96);
// the variant in which query block i only sees the key blocks it did not select for the sparse branch has no
// code there.  Definition used here (per head, S_i = look-up row of query block i, block size BLKK = 64):
//   h_j = phi(K_j)^T V_j (D x D),  z_j = sum_rows phi(K_j)            per key block j
//   H_i = sum_j h_j - sum_{j in S_i} h_j,   z_i likewise              per query block i
//   o_l = phi(Q_i) H_i / (1e-5 + phi(Q_i) . z_i);  out = residual + o_l W^T + b
// Rounding: phi, h_j, H_i, z_i, o_l are rounded to the 16-bit dtype where the global path rounds its
// counterparts; all sums of states are fp32 in a fixed order (ascending j, then the look-up row in order).
//
// Kernels:
//   block states : linear_state_partial_kernel with one 64-row slice per workgroup, 16-bit h_j^T, fp32 z_j
//   totals       : sum_j h_j, sum_j z_j in fp32 (groups of 16 blocks, then the groups)
//   gather       : H_i, z_i = totals - the T selected states, per query block (H_i rounded); the backward reads them again
//   out          : N^T = H_i^T phi(Q)^T, OUT^T = W Y^T for the rows of a query block in the transposed
//                  formulation of the global output kernel.
// At 12 heads of 16380 rows, head dim 128, 12 of 256 blocks selected, with the gathers inside the kernels of the rows (a
// workgroup per query or key block, the whole state in 64 fp32 registers per thread, two waves per SIMD): out 236 us,
// rows 171 us, kv 171 us, and the backward formed the forward's states again (88 us).  With the
// gathers in a kernel of their own: gather 101 us (twice), out 77 us, rows 110 us, kv 112 us.
#include "linear_state.h"

namespace sla {

int validate_attn_shape(int dtype, int B, int H, int L, int D, int BLKQ, int BLKK, int topk, int lut_elem_bytes);
void launch_col_lists(const int8_t* sparse_map, int* list, int* count, int BH, int Mblk, int Nblk, hipStream_t st);
int64_t weight_grads_workspace_bytes(int BH, int L, int D);
void launch_weight_grads(int dtype, int D, const void* q, const void* dn, const void* gout, const void* y, const float* dden,
                         int BH, int L, int fmap, char* ws, float* d_weight, float* d_bias, hipStream_t st);

// Totals in two fixed-order levels: groups of TOTAL_GROUP consecutive key blocks, then the groups in order.
// level 1: grid (cdiv(D*D/8, 256), ngroup, BH), thread owns 8 adjacent elements of one group's D x D sum;
// level 2: grid (cdiv(D*D, 256), BH), thread owns one element.
constexpr int TOTAL_GROUP = 16;

template <typename Tag>
__global__ __launch_bounds__(256) void complement_group_kernel(const uint16_t* __restrict__ hblk,
                                                               const float* __restrict__ zblk, float* __restrict__ hgrp,
                                                               float* __restrict__ zgrp, int N, int D) {
  using E = Elem<Tag>;
  const int DD = D * D;
  const int grp = blockIdx.y, ngroup = gridDim.y, bh = blockIdx.z;
  const int j0 = grp * TOTAL_GROUP, j1 = min(N, j0 + TOTAL_GROUP);
  const int i = (blockIdx.x * 256 + threadIdx.x) * 8;
  if (i < DD) {
    float acc[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] = 0.f;
    const uint16_t* p = hblk + (size_t)bh * N * DD + i;
#pragma unroll 8
    for (int j = j0; j < j1; ++j) {
      const i16x8_t x = *reinterpret_cast<const i16x8_t*>(p + (size_t)j * DD);
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[e] += E::to_float((uint16_t)x[e]);
    }
    float* o = hgrp + ((size_t)bh * ngroup + grp) * DD + i;
    *reinterpret_cast<f32x4_t*>(o) = f32x4_t{acc[0], acc[1], acc[2], acc[3]};
    *reinterpret_cast<f32x4_t*>(o + 4) = f32x4_t{acc[4], acc[5], acc[6], acc[7]};
  }
  const int d = blockIdx.x * 256 + threadIdx.x;
  if (d < D) {
    float s = 0.f;
    for (int j = j0; j < j1; ++j) s += zblk[((size_t)bh * N + j) * D + d];
    zgrp[((size_t)bh * ngroup + grp) * D + d] = s;
  }
}

__global__ __launch_bounds__(256) void complement_total_kernel(const float* __restrict__ hgrp, const float* __restrict__ zgrp,
                                                               float* __restrict__ hall, float* __restrict__ zall, int ngroup,
                                                               int D) {
  const int DD = D * D;
  const int bh = blockIdx.y;
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < DD) {
    float s = 0.f;
#pragma unroll 4
    for (int gi = 0; gi < ngroup; ++gi) s += hgrp[((size_t)bh * ngroup + gi) * DD + i];
    hall[(size_t)bh * DD + i] = s;
  }
  if (i < D) {
    float s = 0.f;
    for (int gi = 0; gi < ngroup; ++gi) s += zgrp[((size_t)bh * ngroup + gi) * D + i];
    zall[(size_t)bh * D + i] = s;
  }
}

// Rows' states: `total - sum of the listed block states` for every query block (its look-up row) or, in the backward, for
// every key block (the query blocks that selected it); 16-bit result, z in fp32.
//
// Bound by the traffic of the listed states (32 KB each at D = 128; a head's do not fit an XCD's L2).  Neighbouring lists
// share many entries (6.8 of 12 between two rows at 12 heads x 16380 rows), so a workgroup takes GATHER_ROWS consecutive rows
// at once: it walks the union of their lists and applies every block's state to all the rows that name it.  It holds a slice
// of 4 KB of the state, 8 values per row and thread.  Applying the difference of a row's list against the previous one's
// instead (one state in registers, 10.2 of 12 loads per row left) took 124 us there,
// the union takes 101.
// Every row's sum runs in the order of the union (the first row's list, what the second adds to it, ...).  Lists longer than
// GATHER_TMAX are walked by themselves.  A list that names every block gives exactly zero by definition, not the rounding
// residue of two fp32 sums formed in different orders, which the 1e-5 of the divisor would turn into an arbitrary result.
constexpr int GATHER_ROWS = 8;
constexpr int GATHER_TMAX = 256;

// list: row (head, r) starts `stride` entries after the previous one and has count[r] entries (`fixed` where count is null).
// 1-D grid over (head, slice, group of rows), 256 threads; thread t owns 16-byte chunk t of its slice.
template <typename Tag, int D>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void complement_gather_kernel(
    const uint16_t* __restrict__ blocks, const float* __restrict__ zblocks, const float* __restrict__ total,
    const float* __restrict__ ztotal, const void* __restrict__ list, int list64, const int* __restrict__ count, int fixed,
    int stride, uint16_t* __restrict__ states, float* __restrict__ zstates, int nrows, int nblk, int ntotal) {
  using E = Elem<Tag>;
  constexpr int DD = D * D;
  constexpr int SLICES = DD / 2048;
  constexpr int R = GATHER_ROWS;
  constexpr int BATCH = 8;               // listed states in flight
  constexpr int CHUNKS = GATHER_TMAX / 64;
  static_assert(DD % 2048 == 0, "slices of 2048 values");
  static_assert(R == 8, "a wave builds the union's share of two rows");
  __shared__ int sRow[R][GATHER_TMAX];
  __shared__ uint32_t sUnion[R * GATHER_TMAX];       // block in the lower 24 bits, the rows that name it above
  __shared__ int sCnt[R * CHUNKS];
  const int logical = xcd_remap(blockIdx.x, gridDim.x, ntotal);
  if (logical < 0) return;
  const int groups = (nrows + R - 1) / R;
  const int unit = logical / groups, row0 = (logical - unit * groups) * R;
  const int bh = unit / SLICES, slice = unit - bh * SLICES;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const bool has_z = slice == 0 && tid < D;
  const size_t off = (size_t)slice * 2048 + tid * 8;
  const uint16_t* hb = blocks + (size_t)bh * nblk * DD + off;
  const float* zb = zblocks + (size_t)bh * nblk * D + (has_z ? tid : 0);
  auto entry = [&](int row, int i) -> int {
    const size_t at = ((size_t)bh * nrows + row) * stride + i;
    return list64 ? (int)reinterpret_cast<const long long*>(list)[at] : reinterpret_cast<const int*>(list)[at];
  };

  int cnt[R];                            // (uniform over the workgroup)
#pragma unroll
  for (int s = 0; s < R; ++s) {
    cnt[s] = row0 + s < nrows ? __builtin_amdgcn_readfirstlane(count ? count[(size_t)bh * nrows + row0 + s] : fixed) : 0;
    if (cnt[s] <= GATHER_TMAX && cnt[s] < nblk && tid < cnt[s]) sRow[s][tid] = entry(row0 + s, tid);
  }
  auto listed = [&](int s) { return cnt[s] <= GATHER_TMAX && cnt[s] < nblk ? cnt[s] : 0; };     // entries in LDS
  __syncthreads();
  // the union: wave w finds which entries of rows w and w + 4 no earlier row names, and who else names them
  uint32_t word[2][CHUNKS];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int s = wave + 4 * h;
    int mine = 0;
#pragma unroll
    for (int x = 0; x < R; ++x) mine = x == s ? listed(x) : mine;
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
      word[h][c] = 0;
      if (c * 64 < mine) {
        const bool has = c * 64 + lane < mine;
        const int j = has ? sRow[s][c * 64 + lane] : -1;
        uint32_t rows = has ? 1u << s : 0u;
#pragma unroll
        for (int x = 0; x < R; ++x) {
          bool hit = false;
          if (x != s)
            for (int u = 0, n = listed(x); u < n; ++u) hit |= sRow[x][u] == j;
          rows |= hit ? 1u << x : 0u;
        }
        if (has && (rows & ((1u << s) - 1)) == 0) word[h][c] = (uint32_t)j | rows << 24;
      }
      const unsigned long long m = __ballot(word[h][c] != 0);
      if (lane == 0) sCnt[s * CHUNKS + c] = __popcll(m);
    }
  }
  __syncthreads();
  int n = 0;
  {
    int before[2][CHUNKS];
    for (int i = 0; i < R * CHUNKS; ++i) {
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int c = 0; c < CHUNKS; ++c)
          if (i == (wave + 4 * h) * CHUNKS + c) before[h][c] = n;
      n += sCnt[i];
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int c = 0; c < CHUNKS; ++c) {
        const unsigned long long m = __ballot(word[h][c] != 0);
        if (word[h][c] != 0) sUnion[before[h][c] + __popcll(m & ((1ull << lane) - 1))] = word[h][c];
      }
    n = __builtin_amdgcn_readfirstlane(n);
  }
  __syncthreads();

  float acc[R][8], zacc[R];
  {
    const float* tot = total + (size_t)bh * DD + off;
    const f32x4_t a = *reinterpret_cast<const f32x4_t*>(tot), b = *reinterpret_cast<const f32x4_t*>(tot + 4);
    const float z = has_z ? ztotal[(size_t)bh * D + tid] : 0.f;
#pragma unroll
    for (int s = 0; s < R; ++s) {
      zacc[s] = z;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        acc[s][e] = a[e];
        acc[s][4 + e] = b[e];
      }
    }
  }
  // subtracts the blocks of words at(0 .. n-1) from the rows they name
  auto walk = [&](int n, auto at) {
    for (int i0 = 0; i0 < n; i0 += BATCH) {
      i16x8_t x[BATCH];
      float zx[BATCH];
      uint32_t rows[BATCH];
#pragma unroll
      for (int u = 0; u < BATCH; ++u) {
        rows[u] = 0;
        if (i0 + u >= n) continue;
        const uint32_t w = (uint32_t)__builtin_amdgcn_readfirstlane((int)at(i0 + u));
        const uint32_t j = w & 0xffffffu;
        rows[u] = w >> 24;
        x[u] = *reinterpret_cast<const i16x8_t*>(hb + (size_t)j * DD);
        zx[u] = has_z ? zb[(size_t)j * D] : 0.f;
      }
#pragma unroll
      for (int u = 0; u < BATCH; ++u) {
        if (i0 + u >= n) continue;
        float f[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) f[e] = E::to_float((uint16_t)x[u][e]);
#pragma unroll
        for (int s = 0; s < R; ++s)
          if (rows[u] >> s & 1) {
#pragma unroll
            for (int e = 0; e < 8; ++e) acc[s][e] -= f[e];
            zacc[s] -= zx[u];
          }
      }
    }
  };
  walk(n, [&](int i) { return sUnion[i]; });
  for (int s = 0; s < R; ++s) {          // lists too long for the union, one at a time
    int longer = 0;
#pragma unroll
    for (int x = 0; x < R; ++x) longer = x == s && cnt[x] > GATHER_TMAX && cnt[x] < nblk ? cnt[x] : longer;
    if (longer) walk(longer, [&](int i) { return (uint32_t)entry(row0 + s, i) | (1u << s) << 24; });
  }
#pragma unroll
  for (int s = 0; s < R; ++s) {
    if (row0 + s >= nrows) break;
    const bool all = cnt[s] >= nblk;
    const size_t at_row = (size_t)bh * nrows + row0 + s;
    i32x4_t w;
#pragma unroll
    for (int e = 0; e < 4; ++e) w[e] = all ? 0 : (int)E::pack2(acc[s][2 * e], acc[s][2 * e + 1]);
    *reinterpret_cast<i32x4_t*>(states + at_row * DD + off) = w;
    if (has_z) zstates[at_row * D + tid] = all ? 0.f : zacc[s];
  }
}

// A row's state on its way from memory into an LDS matrix of D rows with row stride STR.
template <int D>
struct StateRows {
  static constexpr int NCH = D * D / 8 / 256;
  static_assert(D * D / 8 % 256 == 0, "state does not divide among the threads");
  i16x8_t x[NCH];
  float z;
  __device__ __forceinline__ void fetch(const uint16_t* states, const float* zstates, size_t row, int tid) {
#pragma unroll
    for (int c = 0; c < NCH; ++c) x[c] = *reinterpret_cast<const i16x8_t*>(states + row * D * D + (tid + 256 * c) * 8);
    z = tid < D ? zstates[row * D + tid] : 0.f;
  }
  template <int STR>
  __device__ __forceinline__ void park(uint16_t* sH, int tid) const {
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
      const int idx = (tid + 256 * c) * 8;
      *reinterpret_cast<i16x8_t*>(&sH[idx / D * STR + idx % D]) = x[c];
    }
  }
};

// 1-D grid over (head, run of OUT_RUN query blocks: the projection weight is converted once per run), XCD-aware order, 256
// threads; the next block's state is requested beside the products of the present one.
constexpr int OUT_RUN = 4;

template <typename Tag, int D, int BLKQ>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void complement_out_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ states, const float* __restrict__ zstates,
    const float* __restrict__ weight, const float* __restrict__ bias, const uint16_t* __restrict__ residual,
    uint16_t* __restrict__ out, int L, int Mblk, int fmap, int total) {
  using E = Elem<Tag>;
  constexpr int DC = D / 16;
  constexpr int DT = D / 32;
  constexpr int STR = D + 8;
  constexpr int DD = D * D;
  __shared__ __attribute__((aligned(16))) uint16_t sH[D * STR];    // H_i^T [d2][d1]
  __shared__ __attribute__((aligned(16))) uint16_t sW[D * STR];    // W [e][d2 in accumulator slot order]
  __shared__ float sBias[D];
  __shared__ float sZ[D];

  const int logical = xcd_remap(blockIdx.x, gridDim.x, total);
  if (logical < 0) return;
  const int runs = (Mblk + OUT_RUN - 1) / OUT_RUN;
  const int bh = logical / runs, mb0 = (logical - bh * runs) * OUT_RUN;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int g = lane >> 5, r = lane & 31;

  StateRows<D> h;
  h.fetch(states, zstates, (size_t)bh * Mblk + mb0, tid);
  // projection weight, 16 bit, columns in accumulator slot order; bias
#pragma unroll
  for (int i = 0; i < DD / 1024; ++i) {
    const int idx = (tid + 256 * i) * 4, e = idx / D, d = idx % D;       // (four adjacent columns stay adjacent)
    const f32x4_t x = *reinterpret_cast<const f32x4_t*>(weight + idx);
    i32x2_t w;
    w[0] = (int)E::pack2(x[0], x[1]);
    w[1] = (int)E::pack2(x[2], x[3]);
    *reinterpret_cast<i32x2_t*>(&sW[e * STR + slot_order_pos(d)]) = w;
  }
  if (tid < D) sBias[tid] = round16<Tag>(bias[tid]);

  // this wave's 32 queries of a block: rows in operand order
  i16x8_t xq[DC];
  auto fetch_q = [&](int mb) {
    const int qrow = mb * BLKQ + wave * 32 + r;
    const bool ok = wave < BLKQ / 32 && qrow < L;
#pragma unroll
    for (int c = 0; c < DC; ++c) {
      xq[c] = i16x8_t{0, 0, 0, 0, 0, 0, 0, 0};
      if (ok) xq[c] = *reinterpret_cast<const i16x8_t*>(q + ((size_t)bh * L + qrow) * D + 16 * c + 8 * g);
    }
  };
  fetch_q(mb0);

#pragma nounroll
  for (int step = 0; step < OUT_RUN; ++step) {
    const int mb = mb0 + step;
    if (mb >= Mblk) break;
    h.template park<STR>(sH, tid);
    if (tid < D) sZ[tid] = round16<Tag>(h.z);
    __syncthreads();
    const bool more = step + 1 < OUT_RUN && mb + 1 < Mblk;
    if (more) h.fetch(states, zstates, (size_t)bh * Mblk + mb + 1, tid);
    if (wave < BLKQ / 32) {
      // ---- this wave's 32 queries ----
      const int qrow = mb * BLKQ + wave * 32 + r;
      const bool ok = qrow < L;
      const size_t off = ((size_t)bh * L + qrow) * D;
      i32x2_t res[DT][4];
#pragma unroll
      for (int et = 0; et < DT; ++et)
#pragma unroll
        for (int i4 = 0; i4 < 4; ++i4)
          if (residual && ok) res[et][i4] = *reinterpret_cast<const i32x2_t*>(residual + off + 32 * et + 8 * i4 + 4 * g);
      i16x8_t qf[DC];
      float den = phi_pack_den<Tag, DC>(fmap, xq, qf, [&](int c, int j) { return sZ[16 * c + 8 * g + j]; });
      if (more) fetch_q(mb + 1);
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
        for (int c = 0; c < DC; ++c) {
          const i16x8_t a = *reinterpret_cast<const i16x8_t*>(&sH[(32 * t + r) * STR + 16 * c + 8 * g]);
          nacc = E::mfma32(a, qf[c], nacc);
        }
#pragma unroll
        for (int c2 = 0; c2 < 2; ++c2) {
          i32x4_t pw;
#pragma unroll
          for (int j = 0; j < 4; ++j)
            pw[j] = (int)E::pack2(round16<Tag>(nacc[8 * c2 + 2 * j]) * inv_den, round16<Tag>(nacc[8 * c2 + 2 * j + 1]) * inv_den);
          yf[t][c2] = __builtin_bit_cast(i16x8_t, pw);
        }
      }
      // OUT^T = W Y^T : contraction chunk (t, c2) covers d2 = 32t + 16c2 .. +15 in slot order
#pragma unroll
      for (int et = 0; et < DT; ++et) {
        f32x16_t oacc;
#pragma unroll
        for (int i = 0; i < 16; ++i) oacc[i] = 0.f;
#pragma unroll
        for (int t = 0; t < DT; ++t)
#pragma unroll
          for (int c2 = 0; c2 < 2; ++c2) {
            const i16x8_t a = *reinterpret_cast<const i16x8_t*>(&sW[(32 * et + r) * STR + 16 * (2 * t + c2) + 8 * g]);
            oacc = E::mfma32(a, yf[t][c2], oacc);
          }
        if (ok) {
#pragma unroll
          for (int i4 = 0; i4 < 4; ++i4) {
            const int e0 = 32 * et + 8 * i4 + 4 * g;
            float y[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) y[j] = round16<Tag>(oacc[4 * i4 + j] + sBias[e0 + j]);
            if (residual) {
              const uint16_t* rp = reinterpret_cast<const uint16_t*>(&res[et][i4]);
#pragma unroll
              for (int j = 0; j < 4; ++j) y[j] += E::to_float(rp[j]);
            }
            i32x2_t w;
            w[0] = (int)E::pack2(y[0], y[1]);
            w[1] = (int)E::pack2(y[2], y[3]);
            *reinterpret_cast<i32x2_t*>(out + off + e0) = w;
          }
        }
      }
    }
    __syncthreads();                       // H_i^T and z_i are rewritten by the next block of the run
  }
}

// ---- backward ----------------------------------------------------------------------------
// With a = phi(q), c = phi(k), the states h_j, z_j, H_i, z_i as above, n = a H_i, den = 1e-5 + a . z_i, y = n / den,
// out = y W^T + b and G = d(out):
//   db = sum G ; dW = G^T y ; dy = G W ; dn = dy / den ; dden = -sum_d(dy * y) / den
//   da = dn H_i^T + dden z_i ; dq = phi'(q) da
//   dH_i = a_i^T dn_i (rows of query block i), dz_i = sum_rows dden a
//   G_j = sum_{i : j not in S_i} dH_i = sum_i dH_i - sum_{i in C_j} dH_i  (C_j = query blocks that selected j), gz_j likewise
//   dc = v G_j^T + gz_j ; dv = c G_j ; dk = phi'(k) dc                     (rows of key block j)
// Kernels (the totals, the per-block products and dW / db reuse kernels of the forward and of the global backward):
//   rows   : one workgroup per query block: y, dy, dn, dden, da, dq for its rows from the forward's H_i, z_i on the MFMA in
//            transposed form; writes dq and the row-wise temporaries dn, y (16 bit), dden
//   gather : the forward's kernel: G_j, gz_j = total - listed dH_i, dz_i
//   kv     : one workgroup per key block: dv, dc, dk for its 64 rows

// 1-D grid over (head, query block), XCD-aware order, 256 threads; waves 0 .. BLKQ/32-1 own 32 query rows each.
template <typename Tag, int D, int BLKQ>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void complement_bwd_rows_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ gout, const uint16_t* __restrict__ states,
    const float* __restrict__ zstates, const uint16_t* __restrict__ wt, uint16_t* __restrict__ dq, uint16_t* __restrict__ dn_out,
    uint16_t* __restrict__ y_out, float* __restrict__ dden_out, int L, int Mblk, int fmap, int total, int accumulate) {
  using E = Elem<Tag>;
  constexpr int DC = D / 16;
  constexpr int DT = D / 32;
  constexpr int HSTR = D + 16;           // H_i^T is read row-wise (n^T = H^T a^T) and transposed (da^T = H dn^T)
  constexpr int XSTR = D + 8;
  constexpr int DD = D * D;
  constexpr int XROWS = D > BLKQ ? D : BLKQ;
  __shared__ __attribute__((aligned(16))) uint16_t sHT[D * HSTR];      // H_i^T [d2][d1]
  // first the waves' staging tiles (q, G in), then W^T [d][e] (A of dy^T = W^T G^T), then staging tiles again (out)
  __shared__ __attribute__((aligned(16))) uint16_t sX[XROWS * XSTR];
  __shared__ float sZ[D];
  static_assert(TileRows<D>::SSTR == XSTR, "staging tiles and W^T share one row stride");

  const int logical = xcd_remap(blockIdx.x, gridDim.x, total);
  if (logical < 0) return;
  const int bh = logical / Mblk, mb = logical - bh * Mblk;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int g = lane >> 5, r = lane & 31;
  const int row0 = mb * BLKQ + wave * 32;
  const bool active = wave < BLKQ / 32 && row0 < L;     // (uniform per wave)
  const int rows_valid = min(32, L - row0);
  const int qrow = row0 + r;
  const bool ok = active && qrow < L;
  const size_t toff = ((size_t)bh * L + row0) * D;
  uint16_t* const stage = sX + wave * 32 * XSTR;

  // This wave's q and G rows take their operand order through LDS: q in the wave's staging tile, G in the still unused
  // H_i^T buffer.  The state is on its way meanwhile.
  constexpr bool G_IN_H = (BLKQ / 32) * 32 * XSTR <= D * HSTR;
  uint16_t* const gstage = G_IN_H ? sHT + wave * 32 * XSTR : stage;
  TileRows<D> gt;
  StateRows<D> h;
  h.fetch(states, zstates, (size_t)bh * Mblk + mb, tid);
  if (active) {
    TileRows<D> qt;
    qt.fetch(q + toff, rows_valid, lane);
    gt.fetch(gout + toff, rows_valid, lane);
    qt.park(stage, lane);
    if (G_IN_H) gt.park(gstage, lane);
  }
  // G in B-operand order (d = 16c + 8g + j)
  i16x8_t gf[DC];
  if (active && G_IN_H) {
#pragma unroll
    for (int c = 0; c < DC; ++c) gf[c] = *reinterpret_cast<const i16x8_t*>(&gstage[r * XSTR + 16 * c + 8 * g]);
  }
  if (G_IN_H) __syncthreads();           // the G tiles have been read: the buffer takes H_i^T
  h.template park<HSTR>(sHT, tid);
  if (tid < D) sZ[tid] = round16<Tag>(h.z);
  __syncthreads();                       // H_i^T, z_i visible
  // q in B-operand order (d = 16c + 8g + j) -> a = phi(q) as B operand and the divisor; raw q in accumulator order
  // (d = 32t + 8i4 + 4g + j) for the gradient through phi
  i32x2_t xraw[DT][4];
  i16x8_t af[DC];
  float row_mx = 0.f, row_inv = 1.f, inv_den = 0.f;
  if (active) {
    float f[DC][8];
#pragma unroll
    for (int c = 0; c < DC; ++c) {
      const i16x8_t x = *reinterpret_cast<const i16x8_t*>(&stage[r * XSTR + 16 * c + 8 * g]);
#pragma unroll
      for (int j = 0; j < 8; ++j) f[c][j] = E::to_float((uint16_t)x[j]);
    }
#pragma unroll
    for (int t1 = 0; t1 < DT; ++t1)
#pragma unroll
      for (int i4 = 0; i4 < 4; ++i4)
        xraw[t1][i4] = *reinterpret_cast<const i32x2_t*>(&stage[r * XSTR + 32 * t1 + 8 * i4 + 4 * g]);
    if (!G_IN_H) {
      wave_lds_fence();
      gt.park(stage, lane);
#pragma unroll
      for (int c = 0; c < DC; ++c) gf[c] = *reinterpret_cast<const i16x8_t*>(&stage[r * XSTR + 16 * c + 8 * g]);
    }
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
  __syncthreads();                       // every wave has read its staging tile: the buffer takes W^T
  for (int idx = tid; idx < DD / 8; idx += 256) {
    const int row = idx / (D / 8), col = (idx % (D / 8)) * 8;
    *reinterpret_cast<i16x8_t*>(&sX[row * XSTR + col]) = *reinterpret_cast<const i16x8_t*>(wt + (size_t)row * D + col);
  }
  __syncthreads();                       // W^T visible

  float yv[DT][16], dnv[DT][16];
  if (active) {
    // y^T = (H_i^T a^T) / den ; dy^T = W^T G^T
#pragma unroll
    for (int t = 0; t < DT; ++t) {
      f32x16_t yacc, dyacc;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        yacc[i] = 0.f;
        dyacc[i] = 0.f;
      }
#pragma unroll
      for (int c = 0; c < DC; ++c) {
        const i16x8_t a1 = *reinterpret_cast<const i16x8_t*>(&sHT[(32 * t + r) * HSTR + 16 * c + 8 * g]);
        yacc = E::mfma32(a1, af[c], yacc);
        const i16x8_t a2 = *reinterpret_cast<const i16x8_t*>(&sX[(32 * t + r) * XSTR + 16 * c + 8 * g]);
        dyacc = E::mfma32(a2, gf[c], dyacc);
      }
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        yv[t][i] = yacc[i];
        dnv[t][i] = dyacc[i];
      }
    }
  }
  __syncthreads();                       // W^T consumed: its rows are staging tiles again
  if (!active) return;

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
  if (ok && g == 0) dden_out[(size_t)bh * L + qrow] = dden;

  // dn^T as B operand: register 8c2+j of tile t is d2 = 32t + 16c2 + 8(j/4) + 4g + j%4
  i16x8_t dnf[DT][2];
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int c2 = 0; c2 < 2; ++c2) {
      i32x4_t pw;
#pragma unroll
      for (int j = 0; j < 4; ++j) pw[j] = (int)E::pack2(dnv[t][8 * c2 + 2 * j], dnv[t][8 * c2 + 2 * j + 1]);
      dnf[t][c2] = __builtin_bit_cast(i16x8_t, pw);
    }
  TileRows<D> dq_old;
  if (accumulate) dq_old.fetch(dq + toff, rows_valid, lane);
  store_acc_tile<E, D>(stage, dnv, dn_out + toff, nullptr, rows_valid, lane);
  store_acc_tile<E, D>(stage, yv, y_out + toff, nullptr, rows_valid, lane);

  // da^T = H_i dn^T + z_i dden: rows d1 of H_i come out of H_i^T through the transposing read, the contraction
  // index d2 in the slot order of dn^T above
  const int tr_row = (lane & 15) >> 2;
  const int tr_col = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
  float da[DT][16], xq[DT][16];
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
        acc = E::mfma32(concat4(lds_read_tr16(p0), lds_read_tr16(p0 + 8 * HSTR)), dnf[t][c2], acc);
      }
#pragma unroll
    for (int i4 = 0; i4 < 4; ++i4) {
      const int d0 = 32 * t1 + 8 * i4 + 4 * g;
      const uint16_t* xp = reinterpret_cast<const uint16_t*>(&xraw[t1][i4]);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        da[t1][4 * i4 + j] = acc[4 * i4 + j] + sZ[d0 + j] * dden;
        xq[t1][4 * i4 + j] = E::to_float(xp[j]);
      }
    }
  }
  phi_backward<DT>(fmap, xq, da, row_mx, row_inv);
  store_acc_tile<E, D>(stage, da, dq + toff, accumulate ? &dq_old : nullptr, rows_valid, lane);
}

// 1-D grid over (head, key block), XCD-aware order, 256 threads; waves 0 and 1 own 32 key rows each.
// states: per key block G_j^T [d2][d1] (16 bit), zstates: gz_j (fp32).
template <typename Tag, int D>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void complement_bwd_kv_kernel(
    const uint16_t* __restrict__ k, const uint16_t* __restrict__ v, const uint16_t* __restrict__ states,
    const float* __restrict__ zstates, uint16_t* __restrict__ dk, uint16_t* __restrict__ dv, int L, int N, int fmap, int total,
    int accumulate) {
  using E = Elem<Tag>;
  constexpr int DC = D / 16;
  constexpr int DT = D / 32;
  constexpr int GSTR = D + 16;           // G_j^T is read row-wise (dv^T = G^T c^T) and transposed (dc^T = G v^T)
  constexpr int SSTR = TileRows<D>::SSTR;
  __shared__ __attribute__((aligned(16))) uint16_t sGT[D * GSTR];      // G_j^T [d2][d1]
  __shared__ __attribute__((aligned(16))) uint16_t sStage[2][32 * SSTR];
  __shared__ float sGZ[D];

  const int logical = xcd_remap(blockIdx.x, gridDim.x, total);
  if (logical < 0) return;
  const int bh = logical / N, nb = logical - bh * N;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int g = lane >> 5, r = lane & 31;
  const int row0 = nb * 64 + wave * 32;
  const bool active = wave < 2 && row0 < L;
  const int rows_valid = min(32, L - row0);
  const size_t toff = ((size_t)bh * L + row0) * D;
  // this wave's k and v rows take their operand order through LDS: k in the wave's staging tile, v in the still unused
  // G_j^T buffer; the state is on its way meanwhile
  static_assert(2 * 32 * SSTR <= D * GSTR, "v tiles exceed the state buffer");
  uint16_t* const stage = sStage[wave & 1];
  uint16_t* const vstage = sGT + (wave & 1) * 32 * SSTR;
  StateRows<D> h;
  h.fetch(states, zstates, (size_t)bh * N + nb, tid);
  if (active) {
    TileRows<D> kt, vt;
    kt.fetch(k + toff, rows_valid, lane);
    vt.fetch(v + toff, rows_valid, lane);
    kt.park(stage, lane);
    vt.park(vstage, lane);
  }
  i16x8_t vf[DC];
  if (active) {
#pragma unroll
    for (int c = 0; c < DC; ++c) vf[c] = *reinterpret_cast<const i16x8_t*>(&vstage[r * SSTR + 16 * c + 8 * g]);
  }
  __syncthreads();                       // the v tiles have been read: the buffer takes G_j^T
  h.template park<GSTR>(sGT, tid);
  if (tid < D) sGZ[tid] = h.z;
  __syncthreads();
  if (!active) return;

  float f[DC][8];
#pragma unroll
  for (int c = 0; c < DC; ++c) {
    const i16x8_t x = *reinterpret_cast<const i16x8_t*>(&stage[r * SSTR + 16 * c + 8 * g]);
#pragma unroll
    for (int j = 0; j < 8; ++j) f[c][j] = E::to_float((uint16_t)x[j]);
  }
  i32x2_t xraw[DT][4];
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int i4 = 0; i4 < 4; ++i4) xraw[t][i4] = *reinterpret_cast<const i32x2_t*>(&stage[r * SSTR + 32 * t + 8 * i4 + 4 * g]);
  wave_lds_fence();
  float row_mx, row_inv;
  phi_row_pair<Tag, DC>(fmap, f, row_mx, row_inv);
  {
    // dv^T = G^T c^T
    i16x8_t cf[DC];
#pragma unroll
    for (int c = 0; c < DC; ++c) {
      i32x4_t pw;
#pragma unroll
      for (int j = 0; j < 4; ++j) pw[j] = (int)E::pack2(f[c][2 * j], f[c][2 * j + 1]);
      cf[c] = __builtin_bit_cast(i16x8_t, pw);
    }
    float dvv[DT][16];
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
#pragma unroll
      for (int i = 0; i < 16; ++i) dvv[t][i] = vacc[i];
    }
    if (accumulate)
      store_acc_tile<E, D, true>(stage, dvv, dv + toff, nullptr, rows_valid, lane);
    else
      store_acc_tile<E, D, false>(stage, dvv, dv + toff, nullptr, rows_valid, lane);
  }
  // dc^T = G v^T + gz ; dk = phi'(k) dc  (rows d1 of G through the transposing read, d2 in the order of v's fragments)
  const int tr_row = (lane & 15) >> 2;
  const int tr_col = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
  float dc[DT][16], xk[DT][16];
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
      const uint16_t* xp = reinterpret_cast<const uint16_t*>(&xraw[t][i4]);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        dc[t][4 * i4 + j] = acc[4 * i4 + j] + sGZ[d0 + j];
        xk[t][4 * i4 + j] = E::to_float(xp[j]);
      }
    }
  }
  phi_backward<DT>(fmap, xk, dc, row_mx, row_inv);
  if (accumulate)
    store_acc_tile<E, D, true>(stage, dc, dk + toff, nullptr, rows_valid, lane);
  else
    store_acc_tile<E, D, false>(stage, dc, dk + toff, nullptr, rows_valid, lane);
}

// ---- host ---------------------------------------------------------------------------------
struct ComplWs {
  int ngroup;
  size_t hblk, zblk, hgrp, zgrp, hall, zall, total;      // total: without the query blocks' states
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
  w.ngroup = cdiv((int)N, TOTAL_GROUP);
  w.hgrp = off; off += align_up((int64_t)BH * w.ngroup * D * D * 4, 256);
  w.zgrp = off; off += align_up((int64_t)BH * w.ngroup * D * 4, 256);
  w.hall = off; off += align_up((int64_t)BH * D * D * 4, 256);
  w.zall = off; off += align_up((int64_t)BH * D * 4, 256);
  w.total = off;
  return w;
}
// A call that does not keep the query blocks' states (twice the bytes of q at 64-row blocks and head dim 128) forms them for a
// few heads at a time: in the place of the groups' sums, which nobody reads any more (an eighth of the block states), or,
// where those hold less, in up to CPL_STATES_AT_ONCE bytes of their own, so that short problems stay one launch.
// 40 heads x 75600 x 128: 1.65 GiB of workspace (all at once 3.1), in 10 groups, inference 17.3 ms (16.5).  12 heads x 32760
// x 128, in us: 64 MiB at once 1222, 128 MiB 1118, all (201 MiB) 1090; up to 12 heads x 16380 are one group.
constexpr int64_t CPL_STATES_AT_ONCE = 128ll << 20;
struct ComplGroups {
  int heads;             // per group
  size_t at, extra;      // where the states lie; bytes they add behind `end`, the end of the rest of the workspace
};
static ComplGroups compl_groups(int BH, int L, int D, int BLKQ, size_t end) {
  const ComplWs w = compl_ws(BH, L, D);
  const size_t sums = w.zgrp - w.hgrp, one = compl_states(1, L, D, BLKQ).total;
  const size_t room = sums > (size_t)CPL_STATES_AT_ONCE ? sums : (size_t)CPL_STATES_AT_ONCE;
  ComplGroups g;
  g.heads = (int)(room / one < 1 ? 1 : room / one > (size_t)BH ? BH : room / one);
  g.heads = cdiv(BH, cdiv(BH, g.heads));                    // (even groups)
  const size_t bytes = compl_states(g.heads, L, D, BLKQ).total;
  g.extra = bytes <= sums ? 0 : bytes;
  g.at = bytes <= sums ? w.hgrp : end;
  return g;
}
int64_t linear_complement_apart_bytes(int BH, int L, int D) { return (int64_t)compl_ws(BH, L, D).total; }
int64_t linear_complement_workspace_bytes(int BH, int L, int D, int BLKQ) {
  const size_t end = compl_ws(BH, L, D).total;
  return (int64_t)(end + compl_groups(BH, L, D, BLKQ, end).extra);
}

// `total - listed` for nrows rows of every head (see complement_gather_kernel)
template <typename Tag, int D>
static void launch_gather(const uint16_t* blocks, const float* zblocks, const float* total, const float* ztotal, const void* list,
                          int list64, const int* count, int fixed, int stride, uint16_t* states, float* zstates, int BH, int nrows,
                          int nblk, hipStream_t st) {
  const int units = BH * (D * D / 2048) * cdiv(nrows, GATHER_ROWS);
  hipLaunchKernelGGL((complement_gather_kernel<Tag, D>), dim3(xcd_grid(units)), dim3(256), 0, st, blocks, zblocks, total, ztotal,
                     list, list64, count, fixed, stride, states, zstates, nrows, nblk, units);
}

// Block states and their totals.
template <typename Tag, int D>
static void complement_totals_run(const void* k, const void* v, int fmap, int BH, int L, char* ws, hipStream_t st) {
  const ComplWs w = compl_ws(BH, L, D);
  const int N = cdiv(L, 64);
  uint16_t* hblk = (uint16_t*)(ws + w.hblk);
  float* zblk = (float*)(ws + w.zblk);
  float* hgrp = (float*)(ws + w.hgrp);
  float* zgrp = (float*)(ws + w.zgrp);
  hipLaunchKernelGGL((linear_state_partial_kernel<Tag, D, true>), dim3(N, BH), dim3(256), 0, st, (const uint16_t*)k,
                     (const uint16_t*)v, contiguous_layout(BH, L, D), (void*)hblk, zblk, L, 64, fmap, (const float*)nullptr);
  hipLaunchKernelGGL((complement_group_kernel<Tag>), dim3(cdiv(D * D / 8, 256), w.ngroup, BH), dim3(256), 0, st, hblk, zblk,
                     hgrp, zgrp, N, D);
  hipLaunchKernelGGL(complement_total_kernel, dim3(cdiv(D * D, 256), BH), dim3(256), 0, st, hgrp, zgrp, (float*)(ws + w.hall),
                     (float*)(ws + w.zall), w.ngroup, D);
}

// The query blocks' states of `heads` heads from head h0 on, laid out as compl_states(heads, ..) says.
template <typename Tag, int D>
static void complement_gather_run(const void* lut, int lut64, int BH, int L, int BLKQ, int topk, const char* ws, int h0, int heads,
                                  char* states, hipStream_t st) {
  const ComplWs w = compl_ws(BH, L, D);
  const ComplStates s = compl_states(heads, L, D, BLKQ);
  const int N = cdiv(L, 64), M = cdiv(L, BLKQ);
  const size_t head = h0;
  launch_gather<Tag, D>((const uint16_t*)(ws + w.hblk) + head * N * D * D, (const float*)(ws + w.zblk) + head * N * D,
                        (const float*)(ws + w.hall) + head * D * D, (const float*)(ws + w.zall) + head * D,
                        lut ? (const char*)lut + head * M * topk * (lut64 ? 8 : 4) : nullptr, lut64, nullptr, topk, topk,
                        (uint16_t*)(states + s.h), (float*)(states + s.z), heads, M, N, st);
}

// (kept: where the caller wants every head's states; null: they are formed in the workspace, a group of heads at a time)
template <typename Tag, int D, int BLKQ>
static int complement_impl(const void* q, const void* k, const void* v, const void* lut, int lut64, const float* weight,
                           const float* bias, const void* residual, void* out, int fmap, int BH, int L, int topk, char* ws,
                           char* kept, hipStream_t st) {
  const int Mblk = cdiv(L, BLKQ);
  complement_totals_run<Tag, D>(k, v, fmap, BH, L, ws, st);
  const ComplGroups g = compl_groups(BH, L, D, BLKQ, compl_ws(BH, L, D).total);
  const int step = kept ? BH : g.heads;
  char* const states = kept ? kept : ws + g.at;
  for (int h0 = 0; h0 < BH; h0 += step) {
    const int heads = BH - h0 < step ? BH - h0 : step;
    const ComplStates s = compl_states(heads, L, D, BLKQ);
    const size_t rows = (size_t)h0 * L * D;
    complement_gather_run<Tag, D>(lut, lut64, BH, L, BLKQ, topk, ws, h0, heads, states, st);
    const int total = heads * cdiv(Mblk, OUT_RUN);
    hipLaunchKernelGGL((complement_out_kernel<Tag, D, BLKQ>), dim3(xcd_grid(total)), dim3(256), 0, st, (const uint16_t*)q + rows,
                       (const uint16_t*)(states + s.h), (const float*)(states + s.z), weight, bias,
                       residual ? (const uint16_t*)residual + rows : nullptr, (uint16_t*)out + rows, L, Mblk, fmap, total);
  }
  return check_launch("linear_complement_fwd");
}

// ---- backward, host -------------------------------------------------------------------------
struct ComplBwdWs {
  ComplWs fwd;
  int ngroup_q;
  size_t wt, dn, y, dden, dhblk, dzblk, dgrp, dzgrp, gall, gzall, wg, count, list, total;
};
static ComplBwdWs compl_bwd_ws(int BH, int L, int D, int BLKQ) {
  const int64_t N = cdiv(L, 64), M = cdiv(L, BLKQ);
  ComplBwdWs w;
  w.fwd = compl_ws(BH, L, D);
  w.ngroup_q = cdiv((int)M, TOTAL_GROUP);
  size_t off = w.fwd.total;
  w.wt = off;    off += align_up((int64_t)D * D * 2, 256);
  w.dn = off;    off += align_up((int64_t)BH * L * D * 2, 256);
  w.y = off;     off += align_up((int64_t)BH * L * D * 2, 256);
  w.dden = off;  off += align_up((int64_t)BH * L * 4, 256);
  w.dhblk = off; off += align_up((int64_t)BH * M * D * D * 2, 256);
  w.dzblk = off; off += align_up((int64_t)BH * M * D * 4, 256);
  w.dgrp = off;  off += align_up((int64_t)BH * w.ngroup_q * D * D * 4, 256);
  w.dzgrp = off; off += align_up((int64_t)BH * w.ngroup_q * D * 4, 256);
  w.gall = off;  off += align_up((int64_t)BH * D * D * 4, 256);
  w.gzall = off; off += align_up((int64_t)BH * D * 4, 256);
  w.wg = off;    off += align_up(weight_grads_workspace_bytes(BH, L, D), 256);
  w.count = off; off += align_up((int64_t)BH * N * 4, 256);
  w.list = off;  off += align_up((int64_t)BH * N * M * 4, 256);
  w.total = off;
  return w;
}
int64_t linear_complement_bwd_apart_bytes(int BH, int L, int D, int BLKQ) { return (int64_t)compl_bwd_ws(BH, L, D, BLKQ).total; }
int64_t linear_complement_bwd_workspace_bytes(int BH, int L, int D, int BLKQ) {
  const size_t end = compl_bwd_ws(BH, L, D, BLKQ).total;
  return (int64_t)(end + compl_groups(BH, L, D, BLKQ, end).extra);
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
  float* gall = (float*)(ws + w.gall);
  float* gzall = (float*)(ws + w.gzall);
  int* count = (int*)(ws + w.count);
  int* list = (int*)(ws + w.list);
  hipLaunchKernelGGL((linear_prep_weight_kernel<Tag>), dim3(cdiv(D * D, 256)), dim3(256), 0, st, weight, wt, D);
  launch_col_lists(sparse_map, list, count, BH, Mblk, N, st);
  // rows: dq and the row temporaries (with the forward's states, kept or formed again)
  if (!kept) complement_totals_run<Tag, D>(k, v, fmap, BH, L, ws, st);
  const ComplGroups g = compl_groups(BH, L, D, BLKQ, w.total);
  const int step = kept ? BH : g.heads;
  for (int h0 = 0; h0 < BH; h0 += step) {
    const int heads = BH - h0 < step ? BH - h0 : step;
    const ComplStates s = compl_states(heads, L, D, BLKQ);
    const size_t rows = (size_t)h0 * L * D;
    if (!kept) complement_gather_run<Tag, D>(lut, lut64, BH, L, BLKQ, topk, ws, h0, heads, ws + g.at, st);
    const char* const states = kept ? kept : ws + g.at;
    const int total_q = heads * Mblk;
    hipLaunchKernelGGL((complement_bwd_rows_kernel<Tag, D, BLKQ>), dim3(xcd_grid(total_q)), dim3(256), 0, st,
                       (const uint16_t*)q + rows, (const uint16_t*)d_out + rows, (const uint16_t*)(states + s.h),
                       (const float*)(states + s.z), wt, (uint16_t*)dq + rows, dn + rows, y + rows, dden + (size_t)h0 * L, L, Mblk,
                       fmap, total_q, accumulate);
  }
  // per query block dH_i^T = (a_i^T dn_i)^T and dz_i = sum dden a (the state kernel with q, dn in the place of k, v),
  // then their totals
  hipLaunchKernelGGL((linear_state_partial_kernel<Tag, D, true, true>), dim3(Mblk, BH), dim3(256), 0, st, (const uint16_t*)q,
                     (const uint16_t*)dn, lay, (void*)dhblk, dzblk, L, BLKQ, fmap, (const float*)dden);
  hipLaunchKernelGGL((complement_group_kernel<Tag>), dim3(cdiv(D * D / 8, 256), w.ngroup_q, BH), dim3(256), 0, st, dhblk, dzblk,
                     (float*)(ws + w.dgrp), (float*)(ws + w.dzgrp), Mblk, D);
  hipLaunchKernelGGL(complement_total_kernel, dim3(cdiv(D * D, 256), BH), dim3(256), 0, st, (const float*)(ws + w.dgrp),
                     (const float*)(ws + w.dzgrp), gall, gzall, w.ngroup_q, D);
  // dW, db
  launch_weight_grads(dtype, D, q, dn, d_out, y, dden, BH, L, fmap, ws + w.wg, d_weight, d_bias, st);
  // dk, dv
  launch_gather<Tag, D>(dhblk, dzblk, gall, gzall, list, 0, count, 0, Mblk, gst, gzst, BH, N, Mblk, st);
  const int total_k = BH * N;
  hipLaunchKernelGGL((complement_bwd_kv_kernel<Tag, D>), dim3(xcd_grid(total_k)), dim3(256), 0, st, (const uint16_t*)k,
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
