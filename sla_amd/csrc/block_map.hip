// Block-mask builder for Sparse-Linear Attention on gfx950.
//
// Stands in for sparse_linear_attention/utils.py:21-67 of the reference:
//   arg_k = k - mean_L(k); pooled_q = mean_pool(q, BLKQ); pooled_k = mean_pool(arg_k, BLKK);
//   score = pooled_q @ pooled_k^T; lut = topk(score); map = scatter(lut).
//
// All of this is HBM-bound streaming or tiny, so it runs on the vector ALUs with a
// FIXED fp32 summation order that a CPU checker can follow bit for bit:
//   block mean : rows added one at a time in ascending order, one IEEE division;
//   column mean: 64-row chunk sums (same order); groups of 32 consecutive chunk sums added in
//                ascending order; group sums added in ascending order; one IEEE division by L;
//   score      : acc = acc + (a_d * b_d), d ascending, no fused multiply-add.
// Selection is by (score descending, index ascending); -0.0 == +0.0.
#include <type_traits>
#include "block_map.h"
#include "block_pool.h"
#include "fwd_steps.h"

#include <mutex>

#pragma clang fp contract(off)

namespace sla {

template <typename IO, int MODE, int W>
__global__ __launch_bounds__(256) void pool_kernel(const typename IO::raw* __restrict__ x, const RowLayout lay,
                                                   const typename IO::raw* __restrict__ colmean,
                                                   void* __restrict__ out, int L, int D, int BLK, int nblk, int tiled) {
  pool_body<IO, MODE, W, 256>(x, lay, colmean, out, L, D, BLK, nblk, tiled, blockIdx.x, blockIdx.y);
}

// The two independent first passes of the mask builder in one launch (neither fills the memory system alone).
template <typename IO, int W>
__global__ __launch_bounds__(256) void pool_pair_kernel(const typename IO::raw* __restrict__ k, float* __restrict__ chunk_sums,
                                                        int nchunk, const typename IO::raw* __restrict__ q,
                                                        const RowLayout lay, typename IO::raw* __restrict__ pq, int BLKQ,
                                                        int nblkq, int L, int D, int tiled) {
  pool_pair_body<IO, W>(k, chunk_sums, nchunk, q, lay, pq, BLKQ, nblkq, L, D, tiled, blockIdx.x, blockIdx.y, blockIdx.z);
}

// Column mean of K, levels 2 and 3 of the fixed summation order:
//   group_sums[bh][g][d] = chunk sums of group g (KMEAN_GROUP consecutive chunks) added in ascending order;
//   colmean[bh][d]       = (group sums added in ascending order) / L, rounded to the input dtype.
__global__ __launch_bounds__(128) void colmean_group_kernel(const float* __restrict__ chunk_sums,
                                                            float* __restrict__ group_sums, int nchunk, int ngroup, int D) {
  const int g = blockIdx.x, bh = blockIdx.y;
  const int c0 = g * KMEAN_GROUP;
  const int n = min(KMEAN_GROUP, nchunk - c0);
  for (int d = threadIdx.x; d < D; d += 128) {
    const float* p = chunk_sums + ((size_t)bh * nchunk + c0) * D + d;
    float acc = 0.f;
#pragma unroll 8
    for (int i = 0; i < n; ++i) acc = acc + p[(size_t)i * D];
    group_sums[((size_t)bh * ngroup + g) * D + d] = acc;
  }
}

template <typename IO>
__global__ __launch_bounds__(128) void colmean_kernel(const float* __restrict__ group_sums,
                                                      typename IO::raw* __restrict__ colmean, int ngroup, int D, int L) {
  const int bh = blockIdx.y;
  const int d = blockIdx.x * blockDim.x + threadIdx.x;
  if (d >= D) return;
  const float* p = group_sums + (size_t)bh * ngroup * D + d;
  float acc = 0.f;
#pragma unroll 8
  for (int i = 0; i < ngroup; ++i) acc = acc + p[(size_t)i * D];
  colmean[(size_t)bh * D + d] = IO::st(acc / (float)L);
}

// Levels 2 and 3 in one launch when the group sums of a column slab fit in LDS.
template <typename IO>
__global__ __launch_bounds__(256) void colmean_fused_kernel(const float* __restrict__ chunk_sums,
                                                            typename IO::raw* __restrict__ colmean, int nchunk, int ngroup,
                                                            int D, int L) {
  __shared__ float gs[COLMEAN_MAX_GROUPS * COLMEAN_SLAB];
  colmean_body<IO, 256>(chunk_sums, colmean, nchunk, ngroup, D, L, blockIdx.x, blockIdx.y, gs);
}

// score[bh][m][n] = round_dtype( sum_d pq[m][d]*pk[n][d] ), d ascending, every product and every sum rounded to fp32.
// 64x64 outputs per workgroup, 4x4 per thread, operands staged through LDS 32 columns at a time.
// VECD (D a multiple of 32): every thread fetches eight adjacent d of one row of each operand with 16-byte loads,
// one chunk ahead of the chunk being accumulated.
template <typename IO, bool VECD>
__global__ __launch_bounds__(256) void score_kernel(const typename IO::raw* __restrict__ pq,
                                                    const typename IO::raw* __restrict__ pk,
                                                    typename IO::raw* __restrict__ score, int M, int N, int D) {
  constexpr int TS = 64, DC = 32, LD = TS + 4;
  constexpr int NV = 8 / IO::VEC;          // 16-byte loads per eight elements
  __shared__ __attribute__((aligned(16))) float sa[DC][LD];
  __shared__ __attribute__((aligned(16))) float sb[DC][LD];
  const int bh = blockIdx.z;
  const int m0 = blockIdx.y * TS, n0 = blockIdx.x * TS;
  const int tid = threadIdx.x;
  const int ty = tid >> 4, tx = tid & 15;
  float acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = 0.f;
  const typename IO::raw* aq = pq + (size_t)bh * M * D;
  const typename IO::raw* bk = pk + (size_t)bh * N * D;
  const int lrow = tid >> 2, lseg = (tid & 3) * 8;
  Vec16<IO> va[NV], vb[NV];
  auto fetch = [&](int d0) {
#pragma unroll
    for (int v = 0; v < NV; ++v) {
#pragma unroll
      for (int e = 0; e < IO::VEC; ++e) {
        va[v].e[e] = 0;
        vb[v].e[e] = 0;
      }
      if (m0 + lrow < M) va[v] = reinterpret_cast<const Vec16<IO>*>(aq + (size_t)(m0 + lrow) * D + d0 + lseg)[v];
      if (n0 + lrow < N) vb[v] = reinterpret_cast<const Vec16<IO>*>(bk + (size_t)(n0 + lrow) * D + d0 + lseg)[v];
    }
  };
  if (VECD) fetch(0);
  for (int d0 = 0; d0 < D; d0 += DC) {
    __syncthreads();
    if (VECD) {
#pragma unroll
      for (int v = 0; v < NV; ++v)
#pragma unroll
        for (int e = 0; e < IO::VEC; ++e) {
          sa[lseg + v * IO::VEC + e][lrow] = IO::ld(va[v].e[e]);
          sb[lseg + v * IO::VEC + e][lrow] = IO::ld(vb[v].e[e]);
        }
    } else {
      for (int idx = tid; idx < TS * DC; idx += 256) {
        const int row = idx / DC, dd = idx % DC;
        const bool dok = d0 + dd < D;
        sa[dd][row] = (m0 + row < M && dok) ? IO::ld(aq[(size_t)(m0 + row) * D + d0 + dd]) : 0.f;
        sb[dd][row] = (n0 + row < N && dok) ? IO::ld(bk[(size_t)(n0 + row) * D + d0 + dd]) : 0.f;
      }
    }
    __syncthreads();
    if (VECD && d0 + DC < D) fetch(d0 + DC);
    const int dn = min(DC, D - d0);
    for (int dd = 0; dd < dn; ++dd) {
      const f32x4_t a = *reinterpret_cast<const f32x4_t*>(&sa[dd][ty * 4]);
      const f32x4_t b = *reinterpret_cast<const f32x4_t*>(&sb[dd][tx * 4]);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          if (sizeof(typename IO::raw) == 2) {
            // the product of two 16-bit values is exact in fp32 (above the subnormal range), so the fused
            // form rounds the same sum once, exactly as the separate addition does, in half the instructions
            acc[i][j] = __builtin_fmaf(a[i], b[j], acc[i][j]);
          } else {
            const float prod = a[i] * b[j];
            acc[i][j] = acc[i][j] + prod;
          }
        }
    }
  }
  typename IO::raw* out = score + (size_t)bh * M * N;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int m = m0 + ty * 4 + i;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = n0 + tx * 4 + j;
      if (n < N) out[(size_t)m * N + n] = IO::st(acc[i][j]);
    }
  }
}

// The same scores from the matrix cores, for 16-bit dtypes.  v_mfma_f32_32x32x2_f32 adds its two products to the
// accumulator one after the other, each with a single rounding: k = 0 first, then k = 1.  A chain of them over
// d = 0, 2, 4, ... therefore is the d-ascending chain of fp32 fused multiply-adds of score_kernel, bit for bit (the
// product of two 16-bit values is exact in fp32, so fused or not makes no difference; values whose products fall
// into the fp32 subnormal range aside), at twice the rate of the vector ALU.
// The operands arrive in the order the products read them (tiled_pos, written by the pooling kernels): a fragment is one
// coalesced load, straight into registers.  TILED = false: the means lie as rows (a workspace with no room for whole tiles);
// a lane then reads all columns of its block and keeps the odd or the even ones.  The same bits.
template <typename IO, int D, bool TILED>
struct ScoreFrags {
  static constexpr int NC = D / 16;              // fragments (16 d of 32 blocks) per tile
  i32x4_t w[NC];
  __device__ __forceinline__ void load(const typename IO::raw* p, int bh, int nblk, int tile, int lane) {
    if constexpr (TILED) {
      const i16x8_t* t = reinterpret_cast<const i16x8_t*>(p + tiled_head(bh, nblk, D)) + (size_t)tile * (NC * 64) + lane;
#pragma unroll
      for (int c = 0; c < NC; ++c) w[c] = __builtin_bit_cast(i32x4_t, t[c * 64]);
    } else {
      const int blk = min(32 * tile + (lane & 31), nblk - 1);      // (blocks past the end: scores nobody looks at)
      const int sh = 16 * (lane >> 5);
      const i32x4_t* t = reinterpret_cast<const i32x4_t*>(p + ((size_t)bh * nblk + blk) * D);
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const i32x4_t a = t[2 * c], b = t[2 * c + 1];
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          const uint32_t lo = (uint32_t)(x < 2 ? a[2 * x] : b[2 * x - 4]), hi = (uint32_t)(x < 2 ? a[2 * x + 1] : b[2 * x - 3]);
          w[c][x] = (int)(((lo >> sh) & 0xffffu) | (hi >> sh) << 16);
        }
      }
    }
  }
  __device__ __forceinline__ float at(int c, int j) const {      // column 16 c + 2 j + lane / 32 of the lane's block
    return IO::ld((typename IO::raw)((uint32_t)w[c][j >> 1] >> (16 * (j & 1))));
  }
};
template <typename IO, int D, bool TILED>
static __device__ __forceinline__ f32x16_t score_tile(const ScoreFrags<IO, D, TILED>& a, const ScoreFrags<IO, D, TILED>& b) {
  __builtin_amdgcn_sched_barrier(0);             // (every load of both tiles first)
  f32x16_t acc;
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[i] = 0.f;
#pragma unroll
  for (int c = 0; c < D / 16; ++c)
#pragma unroll
    for (int j = 0; j < 8; ++j) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a.at(c, j), b.at(c, j), acc, 0, 0, 0);
  return acc;                                    // register i of lane (r, h): query block 8 (i / 4) + i % 4 + 4 h, key block r
}

// 64 x 64 scores per workgroup, one wave per 32 x 32 part; the rounded scores go through LDS and leave in 128-byte runs.
// Bound by the fp32 matrix rate (40 heads x 1182 x 1182: 91 us at the nominal rate); with both operand tiles through LDS
// 158 us, now 140.
template <typename IO, int D, bool TILED>
__global__ __launch_bounds__(256) void score_mfma_kernel(const typename IO::raw* __restrict__ pq,
                                                         const typename IO::raw* __restrict__ pk,
                                                         typename IO::raw* __restrict__ score, int M, int N) {
  constexpr int OS = 64 + 2;             // staged scores between rows
  __shared__ __attribute__((aligned(16))) typename IO::raw sm[64 * OS];
  const int bh = blockIdx.z, tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int r = lane & 31, h = lane >> 5;
  const int m0 = blockIdx.y * 64, n0 = blockIdx.x * 64;
  const int wm = wave >> 1, wn = wave & 1;
  if (m0 + 32 * wm < M && n0 + 32 * wn < N) {
    ScoreFrags<IO, D, TILED> a, b;
    a.load(pq, bh, M, (m0 >> 5) + wm, lane);
    b.load(pk, bh, N, (n0 >> 5) + wn, lane);
    const f32x16_t acc = score_tile<IO, D, TILED>(a, b);
#pragma unroll
    for (int i = 0; i < 16; ++i) sm[(wm * 32 + 8 * (i >> 2) + (i & 3) + 4 * h) * OS + wn * 32 + r] = IO::st(acc[i]);
  }
  __syncthreads();
  typename IO::raw* out = score + (size_t)bh * M * N;
  const int orow = tid >> 5, ocol = (tid & 31) * 2;      // two scores per thread and pass
#pragma unroll
  for (int pass = 0; pass < 8; ++pass) {
    const int ml = pass * 8 + orow, m = m0 + ml, n = n0 + ocol;
    if (m >= M || n >= N) continue;
    const uint32_t two = *reinterpret_cast<const uint32_t*>(&sm[ml * OS + ocol]);
    typename IO::raw* dst = out + (size_t)m * N + n;
    if (!(N & 1) && n + 1 < N) {
      *reinterpret_cast<uint32_t*>(dst) = two;          // (N even: every pair starts 4-byte aligned)
    } else {
      dst[0] = (typename IO::raw)(two & 0xffffu);
      if (n + 1 < N) dst[1] = (typename IO::raw)(two >> 16);
    }
  }
}

template <typename IO>
static void launch_score(const typename IO::raw* pq, const typename IO::raw* pk, int tiled, typename IO::raw* score, int BH, int M,
                         int N, int D, hipStream_t st) {
  const dim3 grid(cdiv(N, 64), cdiv(M, 64), BH);
  if constexpr (sizeof(typename IO::raw) == 2) {
#define SLA_SCORE_CASE(DD, TILED)                                                                                  \
  if (D == DD && (tiled != 0) == TILED) {                                                                          \
    hipLaunchKernelGGL((score_mfma_kernel<IO, DD, TILED>), grid, dim3(256), 0, st, pq, pk, score, M, N);            \
    return;                                                                                                        \
  }
    SLA_SCORE_CASE(128, true)
    SLA_SCORE_CASE(64, true)
    SLA_SCORE_CASE(128, false)
    SLA_SCORE_CASE(64, false)
#undef SLA_SCORE_CASE
  }
  if (D % 32 == 0)
    hipLaunchKernelGGL((score_kernel<IO, true>), grid, dim3(256), 0, st, pq, pk, score, M, N, D);
  else
    hipLaunchKernelGGL((score_kernel<IO, false>), grid, dim3(256), 0, st, pq, pk, score, M, N, D);
}

// Monotone map float -> uint32 (larger float = larger key); -0.0 is folded onto +0.0.  The LOW_BIT
// low bits (zero in the fp32 image of every value of the score dtype) are cleared, also for negative
// values where the complement would set them, so the radix select can stop at LOW_BIT.
template <int LOW_BIT>
static __device__ __forceinline__ uint32_t order_key(float f) {
  uint32_t u = __float_as_uint(f);
  if (u == 0x80000000u) u = 0u;
  u = (u & 0x80000000u) ? ~u : (u | 0x80000000u);
  return u & ~((1u << LOW_BIT) - 1u);
}

// Inclusive prefix sum over the 64 lanes of a wave (data-parallel-primitive moves inside rows of 16 lanes, then the
// row totals are handed on).
static __device__ __forceinline__ int wave_inclusive_sum(int x, int lane) {
  const int rl = lane & 15;
  int t;
  t = __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false);      // row_shr:1
  if (rl >= 1) x += t;
  t = __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false);      // row_shr:2
  if (rl >= 2) x += t;
  t = __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false);      // row_shr:4
  if (rl >= 4) x += t;
  t = __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false);      // row_shr:8
  if (rl >= 8) x += t;
  t = __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);      // row_bcast:15 (last lane of a row -> the next row)
  if ((lane & 31) >= 16) x += t;
  t = __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);      // row_bcast:31 (lane 31 -> the upper half)
  if (lane >= 32) x += t;
  return x;
}

static __device__ __forceinline__ int lanes_before(unsigned long long b) {       // set bits of b below this lane
  return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(b >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)b, 0u));
}

// Writes the selection of a row whose keys lie in EPL registers per lane (key e of lane l: index 64 e + l): everything above
// `thr` and the first `need_eq` keys equal to it, in ascending index order, into the look-up row and the int8 map row (null:
// not wanted).
template <int EPL>
static __device__ __forceinline__ void emit_row(const uint32_t (&keys)[EPL], uint32_t thr, int need_eq, int8_t* mrow, void* lut,
                                                int lut64, size_t lut_row, int N, int T, int lane) {
  int run_eq = 0, run_sel = 0;
#pragma unroll
  for (int e = 0; e < EPL; ++e) {
    if (e * 64 >= N) break;
    const int i = e * 64 + lane;
    const bool in = i < N;
    const bool gt = in && keys[e] > thr;
    const bool eq = in && keys[e] == thr;
    const unsigned long long beq = __ballot(eq);
    const int eq_rank = run_eq + lanes_before(beq);
    const bool sel = gt || (eq && eq_rank < need_eq);
    const unsigned long long bsel = __ballot(sel);
    const int pos = run_sel + lanes_before(bsel);
    if (in && mrow) mrow[i] = sel ? 1 : 0;
    if (sel && pos < T) {              // (pos < T always holds; the test keeps a wrong count from ever leaving the row)
      if (lut64)
        reinterpret_cast<long long*>(lut)[lut_row + pos] = i;
      else
        reinterpret_cast<int*>(lut)[lut_row + pos] = i;
    }
    run_eq += __popcll(beq);
    run_sel += __popcll(bsel);
    __builtin_amdgcn_sched_barrier(0);      // (not every ballot first: a pair of scalar registers each)
  }
}

// The T-th largest of W keys per lane, for R rows at once, built bit by bit from the top (a bit stays when at least T keys are
// at or above the value it gives; counts through the wave's ballots).  The rows' chains hide each other's latency.
// Missing keys are 0.  FOUR: four bits at a time.  (Rows of one or two keys per lane: left alone, the compiler lays out all the bits
// and keeps 23 to 103 scalar registers elsewhere; mask builder of 8 heads x 4096 x 128 in fp32 25.7 -> 24.5 us, of 32 x 7813 x 64 25.8 ->
// 24.9.  With four keys it does not, and is faster for it: 8 heads x 16000 x 64 19.9 us, 20.3 four bits at a time.)
template <int R, int W, int LOW_BIT, bool FOUR = false>
static __device__ __forceinline__ void kth_largest(const uint32_t (&kx)[R][W], int T, uint32_t (&thr)[R]) {
#pragma unroll
  for (int x = 0; x < R; ++x) thr[x] = 0;
  const auto bit = [&](int b) __attribute__((always_inline)) {
    int cnt[R];
#pragma unroll
    for (int x = 0; x < R; ++x) {
      cnt[x] = 0;
#pragma unroll
      for (int e = 0; e < W; ++e) cnt[x] += __popcll(__ballot(kx[x][e] >= (thr[x] | (1u << b))));
    }
#pragma unroll
    for (int x = 0; x < R; ++x)
      if (cnt[x] >= T) thr[x] |= 1u << b;
  };
  if constexpr (FOUR) {
#pragma unroll 4
    for (int b = 31; b >= LOW_BIT; --b) bit(b);
  } else {
    for (int b = 31; b >= LOW_BIT; --b) bit(b);
  }
}
template <int W>
static __device__ __forceinline__ int count_above(const uint32_t (&k)[W], uint32_t thr) {
  int n = 0;
#pragma unroll
  for (int e = 0; e < W; ++e) n += __popcll(__ballot(k[e] > thr));
  return n;
}

constexpr int SELECT_CAND = 128;       // candidates a short list holds

// Selection for R rows (wave-wide; row x's keys: kx[x][e] of lane l is index 64 e + l, 0 past the end of the row).
// The instructions of a threshold search grow with the keys per lane, so it runs twice on few of them where T allows: first on
// S group maxima per lane, whose T-th largest value is at most the row's; the keys not below it, usually little more than
// T, go into a short list in LDS in index order, and the exact search and the emission run on that.  (S 64 T-th maxima:
// T <= 32 with one group, T <= 80 with two leave about 1.2 T .. 1.6 T candidates of distinct random scores.)  Longer rows of
// selected blocks, and lists that overflow because many scores are equal, search all keys.
// Kernel of 12 heads x 512 rows x 512, T = 25: 13.8 -> 11.2 us; of 40 x 1182 x 1182, T = 59: 129 -> 89 us.
// `list`: SELECT_CAND keys, then SELECT_CAND indices, then the map row; private to the wave.
template <int EPL, int LOW_BIT, int R>
static __device__ __forceinline__ void select_rows(const uint32_t (&kx)[R][EPL], uint32_t* list, int8_t* sparse_map, void* lut,
                                                   int lut64, size_t row0, int rows, int N, int T, int lane) {
  uint32_t thr[R];
  bool short_list = EPL > 2 && T <= 80;
  if constexpr (EPL > 2) {
    if (short_list) {
      if (T <= 32) {
        uint32_t mx[R][1];
#pragma unroll
        for (int x = 0; x < R; ++x) {
          mx[x][0] = kx[x][0];
#pragma unroll
          for (int e = 1; e < EPL; ++e) mx[x][0] = max(mx[x][0], kx[x][e]);
        }
        kth_largest<R, 1, LOW_BIT>(mx, T, thr);
      } else {
        uint32_t mx[R][2];
#pragma unroll
        for (int x = 0; x < R; ++x)
#pragma unroll
          for (int s = 0; s < 2; ++s) {
            mx[x][s] = kx[x][s];
#pragma unroll
            for (int e = 2 + s; e < EPL; e += 2) mx[x][s] = max(mx[x][s], kx[x][e]);
          }
        kth_largest<R, 2, LOW_BIT>(mx, T, thr);
      }
    }
  }
  if (!short_list) kth_largest<R, EPL, LOW_BIT, EPL <= 2>(kx, T, thr);
#pragma unroll
  for (int x = 0; x < R; ++x) {
    if (x >= rows) break;
    const size_t row = row0 + x;
    int8_t* const mrow = sparse_map ? sparse_map + row * N : nullptr;
    if constexpr (EPL > 2) {
      if (short_list) {
        const uint32_t lb = thr[x];
        uint32_t* const li = list + SELECT_CAND;
        int n = 0;
#pragma unroll
        for (int e = 0; e < EPL; ++e) {
          const bool in = kx[x][e] >= lb && 64 * e + lane < N;
          const unsigned long long b = __ballot(in);
          const int pos = n + lanes_before(b);
          if (in && pos < SELECT_CAND) {
            list[pos] = kx[x][e];
            li[pos] = (uint32_t)(64 * e + lane);
          }
          n += __popcll(b);
        }
        if (n <= SELECT_CAND) {
          int8_t* const lm = reinterpret_cast<int8_t*>(list + 2 * SELECT_CAND);
          if (mrow)
#pragma unroll
            for (int e = 0; e < EPL / 4; ++e) reinterpret_cast<uint32_t*>(lm)[64 * e + lane] = 0u;
          wave_lds_fence();
          uint32_t ck[1][2], idx[2];
#pragma unroll
          for (int w = 0; w < 2; ++w) {
            const bool in = 64 * w + lane < n;
            ck[0][w] = in ? list[64 * w + lane] : 0u;
            idx[w] = in ? li[64 * w + lane] : 0u;
          }
          uint32_t t1[1];
          kth_largest<1, 2, LOW_BIT>(ck, T, t1);
          const int need_eq = T - count_above<2>(ck[0], t1[0]);
          int run_eq = 0, run_sel = 0;
#pragma unroll
          for (int w = 0; w < 2; ++w) {
            const bool in = 64 * w + lane < n;
            const bool eq = in && ck[0][w] == t1[0];
            const unsigned long long beq = __ballot(eq);
            const bool sel = (in && ck[0][w] > t1[0]) || (eq && run_eq + lanes_before(beq) < need_eq);
            const unsigned long long bsel = __ballot(sel);
            const int pos = run_sel + lanes_before(bsel);
            if (sel && pos < T) {            // (pos < T always holds; the test keeps a wrong count from ever leaving the row)
              if (lut64)
                reinterpret_cast<long long*>(lut)[row * T + pos] = (int)idx[w];
              else
                reinterpret_cast<int*>(lut)[row * T + pos] = (int)idx[w];
              if (mrow) lm[idx[w]] = 1;
            }
            run_eq += __popcll(beq);
            run_sel += __popcll(bsel);
          }
          if (mrow) {
            wave_lds_fence();
            if (!(((uintptr_t)mrow | (uint32_t)N) & 3)) {        // (a map may start at any byte)
#pragma unroll
              for (int e = 0; e < EPL / 4; ++e)
                if (4 * (64 * e + lane) < N) reinterpret_cast<uint32_t*>(mrow)[64 * e + lane] = reinterpret_cast<const uint32_t*>(lm)[64 * e + lane];
            } else {
#pragma unroll
              for (int e = 0; e < EPL; ++e)
                if (64 * e + lane < N) mrow[64 * e + lane] = lm[64 * e + lane];
            }
          }
          wave_lds_fence();                  // (the next row's list goes over this one)
          continue;
        }
        wave_lds_fence();
        const uint32_t (&k1)[1][EPL] = reinterpret_cast<const uint32_t (&)[1][EPL]>(kx[x]);
        uint32_t t1[1];
        kth_largest<1, EPL, LOW_BIT>(k1, T, t1);
        thr[x] = t1[0];
      }
    }
    emit_row<EPL>(kx[x], thr[x], T - count_above<EPL>(kx[x], thr[x]), mrow, lut, lut64, row * T, N, T, lane);
  }
}

// One wavefront per (bh, m) row (four rows per workgroup): find the T-th largest key, then emit
// winners in ascending index order (ties at the threshold value go to the lowest indices).  Writes the int8 map row and the look-up-table row.
// EPL > 0: the row's keys live in EPL registers per lane (N <= 64*EPL; select_rows); EPL == 0: keys in LDS.
// LOW_BIT: lowest key bit that can differ (16 for 16-bit score dtypes, whose low bits are zero).
template <typename IO, int EPL, int LOW_BIT>
__global__ __launch_bounds__(256) void topk_kernel(const typename IO::raw* __restrict__ score,
                                                   int8_t* __restrict__ sparse_map, void* __restrict__ lut, int lut64, int N,
                                                   int T, size_t nrows) {
  extern __shared__ uint32_t lds_keys[];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const size_t row = (size_t)blockIdx.x * 4 + wave;
  if (row >= nrows) return;
  const typename IO::raw* s = score + row * N;
  if (T <= 0) {              // nothing to select (a ratio that rounds to no block at all): an all-zero map row, no table row
    if (sparse_map)
      for (int i = lane; i < N; i += 64) sparse_map[row * N + i] = 0;
    return;
  }
  if constexpr (EPL > 0) {
    __shared__ __attribute__((aligned(16))) uint32_t lists[4][2 * SELECT_CAND + 16 * EPL];
    // (out-of-range slots hold key 0, below every real key but the most negative NaN pattern; the index tests exclude them)
    uint32_t kx[1][EPL];
#pragma unroll
    for (int e = 0; e < EPL; ++e) {
      const int i = e * 64 + lane;
      kx[0][e] = i < N ? order_key<LOW_BIT>(IO::ld(s[i])) : 0u;
    }
    select_rows<EPL, LOW_BIT, 1>(kx, lists[wave], sparse_map, lut, lut64, row, 1, N, T, lane);
  } else {
    // Keys in LDS: radix select, eight key bits per pass (two passes for bf16 scores): the keys that agree with the digits found
    // so far are counted per value of the next digit in a 256-bin histogram (LDS atomics of this wave on its own
    // bins); lane l then owns the four highest undecided digits 255 - 4l .. 252 - 4l, a prefix sum over the lanes
    // gives the number of keys above them, and the one lane whose digits straddle the wanted rank names the digit.
    __shared__ __attribute__((aligned(16))) uint32_t hist_all[4][256];
    uint32_t* keys = lds_keys + (size_t)wave * N;
    const int nit = (N + 63) / 64;
    for (int i = lane; i < N; i += 64) keys[i] = order_key<LOW_BIT>(IO::ld(s[i]));
    uint32_t thr = 0;          // digits decided so far
    int need = T;              // rank of the threshold among the keys that agree with them
    uint32_t* hist = hist_all[wave];
#pragma unroll
    for (int hi = 32; hi > LOW_BIT;) {
      const int w = (hi - LOW_BIT) < 8 ? (hi - LOW_BIT) : 8;
      const int shift = hi - w;
      *reinterpret_cast<i32x4_t*>(&hist[4 * lane]) = i32x4_t{0, 0, 0, 0};
      wave_lds_fence();
      for (int e = 0; e < nit; ++e) {
        const int i = e * 64 + lane;
        const uint32_t kv = i < N ? keys[i] : 0u;
        if (i < N && (hi == 32 || ((kv ^ thr) >> (hi & 31)) == 0)) atomicAdd(&hist[(kv >> shift) & ((1u << w) - 1u)], 1u);
      }
      wave_lds_fence();
      const i32x4_t c4 = *reinterpret_cast<const i32x4_t*>(&hist[252 - 4 * lane]);    // digits 252 - 4l .. 255 - 4l
      const int c[4] = {c4[3], c4[2], c4[1], c4[0]};                                   // in descending order of the digit
      const int mine = c[0] + c[1] + c[2] + c[3];
      const int incl = wave_inclusive_sum(mine, lane);
      const int above = incl - mine;               // keys (among those that agree) whose digit is above all of this lane's
      const bool here = above < need && need <= incl;
      int digit = 0, rest = 0;
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) {             // (at most one of the four digits straddles the rank)
        int before = above;
#pragma unroll
        for (int t = 0; t < jj; ++t) before += c[t];
        if (before < need && need <= before + c[jj]) {
          digit = 255 - 4 * lane - jj;
          rest = need - before;
        }
      }
      const unsigned long long who = __ballot(here);
      const int src = who ? (int)__builtin_ctzll(who) : 0;
      digit = __builtin_amdgcn_readlane(digit, src);
      need = __builtin_amdgcn_readlane(rest, src);
      thr |= (uint32_t)digit << shift;
      hi = shift;
    }
    int run_eq = 0, run_sel = 0;
    for (int e = 0; e < nit; ++e) {
      const int i = e * 64 + lane;
      const bool in = i < N;
      const uint32_t kv = in ? keys[i] : 0u;
      const bool eq = in && kv == thr;
      const unsigned long long beq = __ballot(eq);
      const bool sel = (in && kv > thr) || (eq && run_eq + lanes_before(beq) < need);
      const unsigned long long bsel = __ballot(sel);
      const int pos = run_sel + lanes_before(bsel);
      if (in && sparse_map) sparse_map[row * N + i] = sel ? 1 : 0;
      if (sel && pos < T) {              // (pos < T always holds; the test keeps a wrong count from ever leaving the row)
        if (lut64)
          reinterpret_cast<long long*>(lut)[row * T + pos] = i;
        else
          reinterpret_cast<int*>(lut)[row * T + pos] = i;
      }
      run_eq += __popcll(beq);
      run_sel += __popcll(bsel);
    }
  }
}

// ---- scores and selection in one launch, rows of at most 256 key blocks ------------------------------------------------
// One workgroup of eight waves per 16 query blocks of a head: the waves form the 16 x N scores (16-bit inputs: a tile of 16 x
// 16 each on the matrix cores; fp32 inputs: every product and sum rounded on the vector ALU as in score_kernel), keep them in LDS,
// rounded, and then select for two rows each.  The scores never go to memory and a launch is saved: mask builder of 2
// heads x 1024 x 64 in fp32 25.3 -> 19.6 us, of 32 x 7813 x 64 38.1 -> 35.0.
// Bound by latency: a chain of dependent products, then one of threshold bits.  v_mfma_f32_16x16x4_f32 adds its four products
// one after the other, each with a single rounding, k ascending: the same bits as the 32 x 32 x 2 chain in a quarter of the cycles
// per tile.
// Rows of 129 to 256 key blocks go this way, too, where the workgroups fit the compute units side by side (16-bit inputs; forward, two
// launches / one: 12 heads x 9360 x 128 141.9 / 139.4 us, 8 x 16000 x 64 79.6 / 77.9; 315 workgroups 344.0 / 345.3; fp32 120.7 /
// 121.8).  They are a variant of their own (MAX_N): its short lists take 14 KB of LDS that the shorter rows do not need.
constexpr int SELECT_ONE_N = 256;
static bool select_in_one(int N, int D, int BH, int M, int elem_bytes) {
  return !scores_in_memory(N, D) ||
         ((D == 64 || D == 128) && N <= SELECT_ONE_N && elem_bytes == 2 && (int64_t)BH * cdiv(M, 16) <= 256);
}
template <typename IO, int D, bool TILED>
struct ScoreFrags16 {                            // 16 blocks, a lane's columns are 4 t + lane / 16
  static constexpr int NC = D / 16;
  i32x4_t w[NC];
  __device__ __forceinline__ void load(const typename IO::raw* p, int bh, int nblk, int tile, int lane) {
    const int l = lane & 15, q = lane >> 4;
    if constexpr (TILED) {
      const i16x8_t* t = reinterpret_cast<const i16x8_t*>(p + tiled_head(bh, nblk, D)) + (size_t)(tile >> 1) * (NC * 64) + 32 * (q & 1) +
                         16 * (tile & 1) + l;
#pragma unroll
      for (int c = 0; c < NC; ++c) w[c] = __builtin_bit_cast(i32x4_t, t[c * 64]);
    } else {
      const int blk = min(16 * tile + l, nblk - 1);              // (blocks past the end: scores nobody looks at)
      const i32x4_t* t = reinterpret_cast<const i32x4_t*>(p + ((size_t)bh * nblk + blk) * D);
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const i32x4_t a = t[2 * c], b = t[2 * c + 1];
        w[c] = q & 2 ? i32x4_t{a[1], a[3], b[1], b[3]} : i32x4_t{a[0], a[2], b[0], b[2]};
      }
    }
  }
  __device__ __forceinline__ float at(int c, int t, int q) const {      // column 16 c + 4 t + q
    return IO::ld((typename IO::raw)((uint32_t)w[c][t] >> (16 * (TILED ? q >> 1 : q & 1))));
  }
};
template <typename IO, int D, bool TILED, int MAX_N>
__global__ __launch_bounds__(512) void select_kernel(const typename IO::raw* __restrict__ pq, const typename IO::raw* __restrict__ pk,
                                                     int8_t* __restrict__ sparse_map, void* __restrict__ lut, int lut64, int M,
                                                     int N, int T) {
  typedef typename IO::raw raw;
  constexpr int EB = sizeof(raw), EPL = MAX_N / 64;
  static_assert(MAX_N == SELECT_FUSED_N || (MAX_N == SELECT_ONE_N && EB == 2), "two variants, the one of longer rows for 16-bit inputs");
  constexpr int OS = 64 * EPL + 4 / EB;     // scores between rows
  constexpr int RS = D * 4 + 16;            // bytes between rows of an fp32 q tile
  constexpr int LIST = 2 * SELECT_CAND + 16 * EPL;      // words of a wave's short list
  __shared__ __attribute__((aligned(16))) uint8_t sq[EB == 4 ? 16 * RS : 16];
  __shared__ __attribute__((aligned(16))) raw ss[16 * OS];
  __shared__ uint32_t lists[EPL > 2 ? 8 * LIST : 1];
  const int bh = blockIdx.y, m0 = blockIdx.x * 16;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  if constexpr (EB == 2) {
    for (int t16 = wave; t16 * 16 < N; t16 += 8) {
      const int q = lane >> 4;
      ScoreFrags16<IO, D, TILED> a, b;
      a.load(pq, bh, M, blockIdx.x, lane);
      b.load(pk, bh, N, t16, lane);
      __builtin_amdgcn_sched_barrier(0);    // (every load of both tiles first)
      f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < D / 16; ++c)
#pragma unroll
        for (int t = 0; t < 4; ++t) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a.at(c, t, q), b.at(c, t, q), acc, 0, 0, 0);
#pragma unroll
      for (int i = 0; i < 4; ++i) ss[(4 * q + i) * OS + 16 * t16 + (lane & 15)] = IO::st(acc[i]);
    }
  } else {
    constexpr int NC = D / 4;               // 16-byte pieces per row
    const __amdgpu_buffer_rsrc_t qh = make_rsrc(pq + (size_t)bh * M * D, (uint32_t)M * D * EB);    // rows past the end read as zero
    const __amdgpu_buffer_rsrc_t kh = make_rsrc(pk + (size_t)bh * N * D, (uint32_t)N * D * EB);
    for (int p = tid; p < 16 * NC; p += 512) {
      const int row = p / NC, pc = p % NC;
      *reinterpret_cast<i16x8_t*>(sq + row * RS + pc * 16) = buf_load_b128(qh, (uint32_t)(m0 + row) * (D * EB) + 16 * pc);
    }
    __syncthreads();
    // a wave takes 32 key blocks and 2 RPL query blocks, a lane RPL scores of its key block side by side: every wave has work
    const int r = lane & 31, h = lane >> 5;
    const auto scores = [&](auto rows_per_lane) __attribute__((always_inline)) {
      constexpr int RPL = decltype(rows_per_lane)::value, GROUPS = 8 / RPL;      // tiles of 32 key blocks: RPL
      const int t = wave / GROUPS, row = 2 * RPL * (wave % GROUPS) + RPL * h;
      const uint32_t koff = (uint32_t)(32 * t + r) * (D * EB);
      float acc[RPL] = {};
#pragma unroll 16
      for (int c = 0; c < NC; ++c) {
        const f32x4_t b = __builtin_bit_cast(f32x4_t, buf_load_b128(kh, koff + 16 * c));
#pragma unroll
        for (int i = 0; i < RPL; ++i) {
          const f32x4_t a = *reinterpret_cast<const f32x4_t*>(sq + (row + i) * RS + c * 16);
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const float prod = a[j] * b[j];
            acc[i] = acc[i] + prod;
          }
        }
      }
#pragma unroll
      for (int i = 0; i < RPL; ++i) ss[(row + i) * OS + 32 * t + r] = IO::st(acc[i]);
    };
    if (N <= 32) scores(std::integral_constant<int, 1>{});
    else if (N <= 64) scores(std::integral_constant<int, 2>{});
    else scores(std::integral_constant<int, 4>{});
  }
  __syncthreads();
  const int mw = m0 + 2 * wave;                // this wave's two rows
  if (mw >= M) return;
  const size_t row0 = (size_t)bh * M + mw;
  const int rows = min(2, M - mw);
  if (T <= 0) {              // nothing to select: all-zero map rows, no table rows
    if (sparse_map)
      for (int x = 0; x < rows; ++x)
        for (int i = lane; i < N; i += 64) sparse_map[(row0 + x) * N + i] = 0;
    return;
  }
  const auto key = [&](int x, int i) {
    return i < N ? order_key<IO::KEY_LOW_BIT>(IO::ld(ss[(2 * wave + x) * OS + i])) : 0u;
  };
  if constexpr (EPL > 2) {
    uint32_t kx[2][EPL];
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int e = 0; e < EPL; ++e) kx[x][e] = key(x, 64 * e + lane);
    select_rows<EPL, IO::KEY_LOW_BIT, 2>(kx, lists + wave * LIST, sparse_map, lut, lut64, row0, rows, N, T, lane);
  } else if (N <= 64) {
    const uint32_t kx[2][1] = {{key(0, lane)}, {key(1, lane)}};
    select_rows<1, IO::KEY_LOW_BIT, 2>(kx, nullptr, sparse_map, lut, lut64, row0, rows, N, T, lane);
  } else {
    const uint32_t kx[2][2] = {{key(0, lane), key(0, 64 + lane)}, {key(1, lane), key(1, 64 + lane)}};
    select_rows<2, IO::KEY_LOW_BIT, 2>(kx, nullptr, sparse_map, lut, lut64, row0, rows, N, T, lane);
  }
}

template <typename IO>
static void launch_topk(const typename IO::raw* score, int8_t* sparse_map, void* lut, int lut64, int N, int T, size_t nrows,
                        hipStream_t st) {
  constexpr int LOW = IO::KEY_LOW_BIT;
  const dim3 grid((unsigned)((nrows + 3) / 4)), block(256);
  if (N <= 512)
    hipLaunchKernelGGL((topk_kernel<IO, 8, LOW>), grid, block, 0, st, score, sparse_map, lut, lut64, N, T, nrows);
  else if (N <= 1280)
    hipLaunchKernelGGL((topk_kernel<IO, 20, LOW>), grid, block, 0, st, score, sparse_map, lut, lut64, N, T, nrows);
  else if (N <= 2048)
    hipLaunchKernelGGL((topk_kernel<IO, 32, LOW>), grid, block, 0, st, score, sparse_map, lut, lut64, N, T, nrows);
  else
    hipLaunchKernelGGL((topk_kernel<IO, 0, LOW>), grid, block, (size_t)N * 16, st, score, sparse_map, lut, lut64, N, T, nrows);
}

// scores and selection (map row, look-up row) of every query block from the block means (in tiles where score_takes_tiled)
template <typename IO>
static void launch_select(const typename IO::raw* pq, const typename IO::raw* pk, int tiled, typename IO::raw* score,
                          int8_t* sparse_map, void* lut, int lut64, int BH, int M, int N, int D, int T, hipStream_t st) {
  if (select_in_one(N, D, BH, M, (int)sizeof(typename IO::raw))) {
    const dim3 grid(cdiv(M, 16), BH);
#define SLA_SELECT_CASE(DD, TILED, MAX_N)                                                                                      \
  if (D == DD && (tiled != 0) == TILED && (N > SELECT_FUSED_N) == (MAX_N > SELECT_FUSED_N))                                      \
    hipLaunchKernelGGL((select_kernel<IO, DD, TILED, MAX_N>), grid, dim3(512), 0, st, pq, pk, sparse_map, lut, lut64, M, N, T);
    if constexpr (sizeof(typename IO::raw) == 2) {
      SLA_SELECT_CASE(128, true, SELECT_FUSED_N)
      SLA_SELECT_CASE(64, true, SELECT_FUSED_N)
      SLA_SELECT_CASE(128, true, SELECT_ONE_N)
      SLA_SELECT_CASE(64, true, SELECT_ONE_N)
      SLA_SELECT_CASE(128, false, SELECT_ONE_N)
      SLA_SELECT_CASE(64, false, SELECT_ONE_N)
    }
    SLA_SELECT_CASE(128, false, SELECT_FUSED_N)
    SLA_SELECT_CASE(64, false, SELECT_FUSED_N)
#undef SLA_SELECT_CASE
    return;
  }
  launch_score<IO>(pq, pk, tiled, score, BH, M, N, D, st);
  launch_topk<IO>(score, sparse_map, lut, lut64, N, T, (size_t)BH * M, st);
}

struct MapWs {
  size_t chunk_sums, group_sums, colmean, pq, pk, score, total;
};

// tiled: the block means in whole tiles of 32 blocks per head; otherwise as rows
static MapWs map_ws(int dtype, int BH, int L, int D, int BLKQ, int BLKK, bool tiled) {
  const int64_t M = cdiv(L, BLKQ), N = cdiv(L, BLKK), nchunk = cdiv(L, KMEAN_CHUNK);
  const int unit = tiled ? 32 : 1;
  const int64_t eb = elem_bytes(dtype);
  MapWs w;
  size_t off = 0;
  w.chunk_sums = off; off += align_up((int64_t)BH * nchunk * D * 4, 256);
  w.group_sums = off; off += align_up((int64_t)BH * cdiv((int)nchunk, KMEAN_GROUP) * D * 4, 256);
  w.colmean = off;    off += align_up((int64_t)BH * D * eb, 256);
  w.pq = off;         off += align_up((int64_t)BH * align_up(M, unit) * D * eb, 256);
  w.pk = off;         off += align_up((int64_t)BH * align_up(N, unit) * D * eb, 256);
  w.score = off;      off += scores_in_memory((int)N, D) ? align_up((int64_t)BH * M * N * eb, 256) : 0;
  w.total = off;
  return w;
}

int64_t block_map_workspace_bytes(int dtype, int BH, int L, int D, int BLKQ, int BLKK) {
  return (int64_t)map_ws(dtype, BH, L, D, BLKQ, BLKK, score_takes_tiled(dtype, D)).total;
}
// What a call can make do with: many short heads are mostly padding in tiles (1024 heads of 640 x 128: 21.0 MiB against 10.3).
static int64_t block_map_least_bytes(int dtype, int BH, int L, int D, int BLKQ, int BLKK) {
  return (int64_t)map_ws(dtype, BH, L, D, BLKQ, BLKK, false).total;
}

MapParts block_map_parts(int dtype, int BH, int L, int D, int BLKQ, int BLKK, void* workspace, int64_t workspace_bytes) {
  // (rows cost the score kernels twice the loads: only where the tiles do not fit)
  const bool tiled = score_takes_tiled(dtype, D) && workspace_bytes >= block_map_workspace_bytes(dtype, BH, L, D, BLKQ, BLKK);
  const MapWs w = map_ws(dtype, BH, L, D, BLKQ, BLKK, tiled);
  char* const ws = (char*)workspace;
  return MapParts{(float*)(ws + w.chunk_sums), (float*)(ws + w.group_sums), ws + w.colmean, ws + w.pq, ws + w.pk, ws + w.score,
                  tiled, cdiv(L, BLKQ), cdiv(L, BLKK), cdiv(L, KMEAN_CHUNK)};
}

static int validate_pool(int dtype, int BH, int L, int D, int BLK) {
  SLA_REQUIRE(dtype == SLA_F32 || dtype == SLA_BF16 || dtype == SLA_F16, SLA_ERR_BAD_ARG, "unknown dtype %d", dtype);
  SLA_REQUIRE(BH > 0 && L > 0 && D > 0 && BLK > 0, SLA_ERR_BAD_ARG, "non-positive size (BH=%d L=%d D=%d BLK=%d)", BH, L,
              D, BLK);
  const int vec = dtype == SLA_F32 ? 4 : 8;
  SLA_REQUIRE(D % vec == 0 && D / vec <= 256, SLA_ERR_UNSUPPORTED, "D=%d must be a multiple of %d and at most %d", D, vec,
              256 * vec);
  SLA_REQUIRE(BH <= 65535, SLA_ERR_UNSUPPORTED, "B*H=%d exceeds 65535", BH);
  return SLA_OK;
}

template <typename IO, int MODE>
static void launch_pool(const void* x, const RowLayout& lay, const void* colmean, void* out, int BH, int L, int D, int BLK,
                        hipStream_t st, int tiled = 0) {
  const int nblk = cdiv(L, BLK);
  typedef typename IO::raw raw;
  if (narrow_pools(sizeof(raw) == 4 ? SLA_F32 : SLA_BF16, BH, L, D) && D / (IO::VEC / 4) <= 256)
    hipLaunchKernelGGL((pool_kernel<IO, MODE, IO::VEC / 4>), dim3(cdiv(nblk, 256 / (D / (IO::VEC / 4))), BH), dim3(256), 0, st,
                       (const raw*)x, lay, (const raw*)colmean, out, L, D, BLK, nblk, tiled);
  else
    hipLaunchKernelGGL((pool_kernel<IO, MODE, IO::VEC>), dim3(cdiv(nblk, 256 / (D / IO::VEC)), BH), dim3(256), 0, st, (const raw*)x,
                       lay, (const raw*)colmean, out, L, D, BLK, nblk, tiled);
}

// levels 2 and 3 of the K column mean from the chunk sums
template <typename IO>
static void launch_colmean_reduce(float* chunk_sums, float* group_sums, typename IO::raw* colmean, int BH, int L, int D,
                                  hipStream_t st) {
  const int nchunk = cdiv(L, KMEAN_CHUNK), ngroup = cdiv(nchunk, KMEAN_GROUP);
  if (D % COLMEAN_SLAB == 0 && ngroup <= COLMEAN_MAX_GROUPS) {
    hipLaunchKernelGGL((colmean_fused_kernel<IO>), dim3(D / COLMEAN_SLAB, BH), dim3(256), 0, st, chunk_sums, colmean, nchunk,
                       ngroup, D, L);
    return;
  }
  hipLaunchKernelGGL(colmean_group_kernel, dim3(ngroup, BH), dim3(128), 0, st, chunk_sums, group_sums, nchunk, ngroup, D);
  hipLaunchKernelGGL((colmean_kernel<IO>), dim3(cdiv(D, 128), BH), dim3(128), 0, st, group_sums, colmean, ngroup, D, L);
}

template <typename IO>
static void launch_k_colmean_t(const void* k, const RowLayout& lay, int BH, int L, int D, float* chunk_sums,
                               float* group_sums, typename IO::raw* colmean, hipStream_t st) {
  launch_pool<IO, 0>(k, lay, nullptr, chunk_sums, BH, L, D, KMEAN_CHUNK, st);
  launch_colmean_reduce<IO>(chunk_sums, group_sums, colmean, BH, L, D, st);
}

// scores and selection from the block means in `m` (topk == 0 selects nothing: the map rows are cleared)
void block_map_select(int dtype, const MapParts& m, int BH, int D, int topk, int8_t* sparse_map, void* lut, int lut64,
                      hipStream_t st) {
  if (dtype == SLA_F32)
    launch_select<IoF32>((const float*)m.pq, (const float*)m.pk, m.tiled, (float*)m.score, sparse_map, lut, lut64, BH, m.M, m.N, D, topk, st);
  else if (dtype == SLA_BF16)
    launch_select<IoBf16>((const uint16_t*)m.pq, (const uint16_t*)m.pk, m.tiled, (uint16_t*)m.score, sparse_map, lut, lut64, BH, m.M, m.N, D, topk, st);
  else
    launch_select<IoF16>((const uint16_t*)m.pq, (const uint16_t*)m.pk, m.tiled, (uint16_t*)m.score, sparse_map, lut, lut64, BH, m.M, m.N, D, topk, st);
}

// first_pass = false: the chunk sums of k and the block means of q are there already
template <typename IO>
static void block_map_pool(const void* q, const void* k, const RowLayout& lay, const MapParts& m, int BH, int L, int D, int BLKQ,
                           int BLKK, bool first_pass, hipStream_t st) {
  typename IO::raw* colmean = (typename IO::raw*)m.colmean;
  if (first_pass) {
    // k chunk sums and q block means share one launch
    typedef typename IO::raw raw;
#define SLA_PAIR_CASE(W)                                                                                                     \
  hipLaunchKernelGGL((pool_pair_kernel<IO, W>), dim3(cdiv(max(m.nchunk, m.M), 256 / (D / (W))), BH, 2), dim3(256), 0, st,   \
                     (const raw*)k, m.chunk_sums, m.nchunk, (const raw*)q, lay, (raw*)m.pq, BLKQ, m.M, L, D, m.tiled)
    if (narrow_pools(sizeof(raw) == 4 ? SLA_F32 : SLA_BF16, BH, L, D) && D / (IO::VEC / 4) <= 256) SLA_PAIR_CASE(IO::VEC / 4);
    else SLA_PAIR_CASE(IO::VEC);
#undef SLA_PAIR_CASE
  }
  launch_colmean_reduce<IO>(m.chunk_sums, m.group_sums, colmean, BH, L, D, st);
  launch_pool<IO, 2>(k, lay, colmean, m.pk, BH, L, D, BLKK, st, m.tiled);
}

// Column mean of k over L in the fixed order, rounded to `dtype`.  scratch: fp32, at least
// k_colmean_scratch_floats(BH, L, D) elements; colmean: (BH, D) in `dtype`.
int64_t k_colmean_scratch_floats(int BH, int L, int D) {
  const int64_t nchunk = cdiv(L, KMEAN_CHUNK), ngroup = cdiv((int)nchunk, KMEAN_GROUP);
  return (int64_t)BH * (nchunk + ngroup) * D;
}
void launch_k_colmean(const void* k, const RowLayout& lay, int dtype, int BH, int L, int D, float* scratch, void* colmean,
                      hipStream_t st) {
  const int64_t nchunk = cdiv(L, KMEAN_CHUNK);
  float* chunk_sums = scratch;
  float* group_sums = scratch + (int64_t)BH * nchunk * D;
  if (dtype == SLA_F32)
    launch_k_colmean_t<IoF32>(k, lay, BH, L, D, chunk_sums, group_sums, (float*)colmean, st);
  else if (dtype == SLA_BF16)
    launch_k_colmean_t<IoBf16>(k, lay, BH, L, D, chunk_sums, group_sums, (uint16_t*)colmean, st);
  else
    launch_k_colmean_t<IoF16>(k, lay, BH, L, D, chunk_sums, group_sums, (uint16_t*)colmean, st);
}

// Scores and top-k selection from block means computed elsewhere (the quantisers of the SageSLA path
// produce them on the way): pq (BH, M, D), pk (BH, N, D) in `dtype`, in tiles where score_takes_tiled says so; score:
// (BH, M, N) elements of `dtype`.
void launch_map_from_pooled(int dtype, const void* pq, const void* pk, void* score, int BH, int M, int N, int D, int topk,
                            int8_t* sparse_map, void* lut, int lut64, hipStream_t st) {
  if (dtype == SLA_BF16) {
    const int tiled = score_takes_tiled(dtype, D);
    launch_select<IoBf16>((const uint16_t*)pq, (const uint16_t*)pk, tiled, (uint16_t*)score, sparse_map, lut, lut64, BH, M, N, D, topk, st);
  } else {
    const int tiled = score_takes_tiled(dtype, D);
    launch_select<IoF16>((const uint16_t*)pq, (const uint16_t*)pk, tiled, (uint16_t*)score, sparse_map, lut, lut64, BH, M, N, D, topk, st);
  }
}

// Everything block_map_entry asks of its arguments, for a caller that launches something else before it; `lay` receives the
// layout of q and k.  (want_map = false: the caller needs the look-up table only, sparse_map may be null)
int block_map_check(const void* q, const void* k, const int64_t* strides, int dtype, int B, int H, int L, int D, int BLKQ,
                    int BLKK, int topk, const void* workspace, int64_t workspace_bytes, const int8_t* sparse_map, bool want_map,
                    const void* lut, int lut_elem_bytes, RowLayout* lay) {
  SLA_REQUIRE(B > 0 && H > 0, SLA_ERR_BAD_ARG, "non-positive batch/head count (B=%d H=%d)", B, H);
  const int64_t BH64 = (int64_t)B * H;
  SLA_REQUIRE(BH64 <= 65535, SLA_ERR_UNSUPPORTED, "B*H=%lld exceeds 65535", (long long)BH64);
  const int BH = (int)BH64;
  int rc = validate_pool(dtype, BH, L, D, BLKQ);
  if (rc) return rc;
  rc = validate_pool(dtype, BH, L, D, BLKK);
  if (rc) return rc;
  const int M = cdiv(L, BLKQ), N = cdiv(L, BLKK);
  SLA_REQUIRE(topk >= 0 && topk <= N, SLA_ERR_BAD_ARG, "topk=%d outside [0, %d]", topk, N);
  // (rows longer than the register instances hold keep their keys in LDS: four waves' rows of 4096 keys are 64 KB, plus
  //  4 KB of histograms, of the 160 KB a workgroup of this machine may use; L <= 262144 at 64-row key blocks)
  SLA_REQUIRE(N <= 4096, SLA_ERR_UNSUPPORTED, "more than 4096 key blocks (%d)", N);
  SLA_REQUIRE((int64_t)BH * M < (1ll << 31), SLA_ERR_UNSUPPORTED, "too many query-block rows");
  SLA_REQUIRE(lut_elem_bytes == 4 || lut_elem_bytes == 8, SLA_ERR_BAD_ARG, "lut_elem_bytes must be 4 or 8, got %d",
              lut_elem_bytes);
  SLA_REQUIRE(q && k && workspace && (sparse_map || !want_map) && (lut || topk == 0), SLA_ERR_BAD_ARG, "null pointer");
  SLA_REQUIRE(((uintptr_t)q | (uintptr_t)k | (uintptr_t)workspace | (uintptr_t)lut) % 16 == 0, SLA_ERR_BAD_ARG,
              "pointers must be 16-byte aligned");
  const int64_t need = block_map_least_bytes(dtype, BH, L, D, BLKQ, BLKK);
  SLA_REQUIRE(workspace_bytes >= need, SLA_ERR_WORKSPACE, "workspace of %lld bytes, need %lld", (long long)workspace_bytes,
              (long long)need);
  return make_layout(strides, B, H, L, D, dtype == SLA_F32 ? 4 : 2, lay);
}

int block_map_run(const void* q, const void* k, const RowLayout& lay, int dtype, const MapParts& m, int BH, int L, int D, int BLKQ,
                  int BLKK, int topk, int8_t* sparse_map, void* lut, int lut64, bool first_pass, hipStream_t st) {
  if (dtype == SLA_F32) block_map_pool<IoF32>(q, k, lay, m, BH, L, D, BLKQ, BLKK, first_pass, st);
  else if (dtype == SLA_BF16) block_map_pool<IoBf16>(q, k, lay, m, BH, L, D, BLKQ, BLKK, first_pass, st);
  else block_map_pool<IoF16>(q, k, lay, m, BH, L, D, BLKQ, BLKK, first_pass, st);
  block_map_select(dtype, m, BH, D, topk, sparse_map, lut, lut64, st);
  return check_launch("block map");
}

int block_map_entry(const void* q, const void* k, const int64_t* strides, int dtype, int B, int H, int L, int D, int BLKQ,
                    int BLKK, int topk, void* workspace, int64_t workspace_bytes, int8_t* sparse_map, bool want_map, void* lut,
                    int lut_elem_bytes, void* stream) {
  RowLayout lay;
  const int rc = block_map_check(q, k, strides, dtype, B, H, L, D, BLKQ, BLKK, topk, workspace, workspace_bytes, sparse_map,
                                 want_map, lut, lut_elem_bytes, &lay);
  if (rc) return rc;
  const MapParts m = block_map_parts(dtype, B * H, L, D, BLKQ, BLKK, workspace, workspace_bytes);
  return block_map_run(q, k, lay, dtype, m, B * H, L, D, BLKQ, BLKK, topk, sparse_map, lut, lut_elem_bytes == 8, true,
                       (hipStream_t)stream);
}

}  // namespace sla

using namespace sla;

extern "C" int sla_mean_pool(const void* x, void* out, int dtype, int BH, int L, int D, int BLK, void* stream) {
  int rc = validate_pool(dtype, BH, L, D, BLK);
  if (rc) return rc;
  SLA_REQUIRE(x && out, SLA_ERR_BAD_ARG, "null pointer");
  SLA_REQUIRE(((uintptr_t)x | (uintptr_t)out) % 16 == 0, SLA_ERR_BAD_ARG, "pointers must be 16-byte aligned");
  hipStream_t st = (hipStream_t)stream;
  const RowLayout lay = contiguous_layout(BH, L, D);
  if (dtype == SLA_F32) launch_pool<IoF32, 1>(x, lay, nullptr, out, BH, L, D, BLK, st);
  else if (dtype == SLA_BF16) launch_pool<IoBf16, 1>(x, lay, nullptr, out, BH, L, D, BLK, st);
  else launch_pool<IoF16, 1>(x, lay, nullptr, out, BH, L, D, BLK, st);
  return check_launch("mean_pool");
}

extern "C" int sla_block_map_fwd(const void* q, const void* k, int dtype, int B, int H, int L, int D, int BLKQ, int BLKK,
                                 int topk, void* workspace, int64_t workspace_bytes, int8_t* sparse_map, void* lut,
                                 int lut_elem_bytes, void* stream) {
  return block_map_entry(q, k, nullptr, dtype, B, H, L, D, BLKQ, BLKK, topk, workspace, workspace_bytes, sparse_map, true, lut,
                         lut_elem_bytes, stream);
}

// ---- the block-mask builder for callers that cannot allocate ---------------------------------------------------
// Same kernels as sla_block_map_fwd; the workspace is a fixed array in device memory that every GPU the library runs
// on holds from the moment the code object is loaded until the process ends.
static __device__ __align__(256) unsigned char scratch[SLA_STATIC_SCRATCH_BYTES];

namespace {
constexpr int MAX_DEVICES = 64;
std::mutex g_scratch_mutex;
void* g_scratch_ptr[MAX_DEVICES];   // device address of `scratch` on each GPU, resolved on the first call there

// The array's name is only a handle on the host: its address in the current GPU's memory is looked up once per GPU.
int static_scratch(void** out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  SLA_REQUIRE(e == hipSuccess && dev >= 0 && dev < MAX_DEVICES, SLA_ERR_LAUNCH, "hipGetDevice: %s (device %d)",
              hipGetErrorString(e), dev);
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    SLA_REQUIRE(e == hipSuccess && p, SLA_ERR_LAUNCH, "hipGetSymbolAddress(scratch) on device %d: %s", dev,
                hipGetErrorString(e));
    g_scratch_ptr[dev] = p;
  }
  *out = g_scratch_ptr[dev];
  return SLA_OK;
}
}  // namespace

extern "C" int sla_block_map_fwd_static(const void* q, const void* k, int dtype, int B, int H, int L, int D, int BLKQ,
                                        int BLKK, int topk, int8_t* sparse_map, void* lut, int lut_elem_bytes,
                                        void* stream) {
  // sizes first (testable without a GPU): the problem must fit the fixed array
  SLA_REQUIRE(B > 0 && H > 0 && L > 0 && D > 0 && BLKQ > 0 && BLKK > 0 && (int64_t)B * H <= 65535, SLA_ERR_BAD_ARG,
              "bad size (B=%d H=%d L=%d D=%d BLKQ=%d BLKK=%d)", B, H, L, D, BLKQ, BLKK);
  SLA_REQUIRE(dtype == SLA_F32 || dtype == SLA_BF16 || dtype == SLA_F16, SLA_ERR_BAD_ARG, "unknown dtype %d", dtype);
  const int64_t need = block_map_least_bytes(dtype, B * H, L, D, BLKQ, BLKK);
  SLA_REQUIRE(need <= (int64_t)SLA_STATIC_SCRATCH_BYTES, SLA_ERR_WORKSPACE,
              "this problem needs %lld bytes of scratch, the static buffer holds %lld: use sla_block_map_fwd with a "
              "workspace of the caller's",
              (long long)need, (long long)SLA_STATIC_SCRATCH_BYTES);
  SLA_REQUIRE(q && k && sparse_map && (lut || topk == 0), SLA_ERR_BAD_ARG, "null pointer");
  void* ws = nullptr;
  int rc = static_scratch(&ws);
  if (rc) return rc;
  // every part of the scratch is written by one kernel of the sequence before a later one reads it: nothing
  // has to be cleared between calls
  return block_map_entry(q, k, nullptr, dtype, B, H, L, D, BLKQ, BLKK, topk, ws, (int64_t)SLA_STATIC_SCRATCH_BYTES,
                         sparse_map, true, lut, lut_elem_bytes, stream);
}

extern "C" int sla_block_map_fwd_strided(const void* q, const void* k, const int64_t* qk_strides, int dtype, int B, int H,
                                         int L, int D, int BLKQ, int BLKK, int topk, void* workspace,
                                         int64_t workspace_bytes, int8_t* sparse_map, void* lut, int lut_elem_bytes,
                                         void* stream) {
  SLA_REQUIRE(qk_strides, SLA_ERR_BAD_ARG, "null strides");
  return block_map_entry(q, k, qk_strides, dtype, B, H, L, D, BLKQ, BLKK, topk, workspace, workspace_bytes, sparse_map, true, lut,
                         lut_elem_bytes, stream);
}
