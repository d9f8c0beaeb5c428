// The pooling passes of the mask builder (block_map.hip) as bodies that other launches take along (module_fwd.hip).
//
// Everything here is sums and divisions in a FIXED fp32 order (block_map.hip states it); there is no multiply-add to contract.
#pragma once
#include "block_map.h"

namespace sla {

constexpr int KMEAN_CHUNK = 64;   // rows per level-1 sum
constexpr int KMEAN_GROUP = 32;   // level-1 sums per level-2 sum

// KEY_LOW_BIT: lowest bit of the fp32 image of a value of this type that can be non-zero.
struct IoF32 {
  typedef float raw;
  static constexpr int VEC = 4;
  static constexpr int KEY_LOW_BIT = 0;
  static __device__ __forceinline__ float ld(raw x) { return x; }
  static __device__ __forceinline__ raw st(float x) { return x; }
};
struct IoBf16 {
  typedef uint16_t raw;
  static constexpr int VEC = 8;
  static constexpr int KEY_LOW_BIT = 16;
  static __device__ __forceinline__ float ld(raw x) { return Elem<bf16_tag>::to_float(x); }
  static __device__ __forceinline__ raw st(float x) { return Elem<bf16_tag>::from_float(x); }
};
struct IoF16 {
  typedef uint16_t raw;
  static constexpr int VEC = 8;
  static constexpr int KEY_LOW_BIT = 13;
  static __device__ __forceinline__ float ld(raw x) { return Elem<f16_tag>::to_float(x); }
  static __device__ __forceinline__ raw st(float x) { return Elem<f16_tag>::from_float(x); }
};

template <typename IO, int W>
struct alignas(W * sizeof(typename IO::raw)) VecIo {
  typename IO::raw e[W];
};
template <typename IO>
using Vec16 = VecIo<IO, IO::VEC>;

// No 16-bit copy is wanted of what is pooled.
struct NoCast {};

// MODE 0: fp32 block sums (no division)        -> out_f32 (BH, nblk, D)
// MODE 1: block mean in the input dtype        -> out     (BH, nblk, D)
// MODE 2: block mean of round(x - colmean)     -> out     (BH, nblk, D); colmean: this head's
// One thread owns W adjacent columns of one block and walks its rows in order; NT threads per workgroup.
//   W = 16 bytes: sixteen rows in flight per thread, the form for inputs that fill the chip;
//   W = 4 bytes: 64 rows in flight per thread (32 in workgroups of 512, beside bodies that want the registers) and four times the
//   threads, for inputs that do not: there a pass is as long as its chain of loads (first pass over 8 heads x 4096 x 128: 8.0 -> 5.6 us).
//   Where it rides with other jobs (module_fwd.hip) it is the form for all sizes.
// tiled: the means go out in operand order (16-bit dtypes; tiled_pos) instead of as rows.
// Cast = a 16-bit tag: the rows also leave rounded to 16 bit, at the same place of `cast` (contiguous tensors).
template <typename IO, int MODE, int W, int NT, typename Cast = NoCast>
static __device__ __forceinline__ void pool_body(const typename IO::raw* __restrict__ x, const RowLayout lay,
                                                 const typename IO::raw* __restrict__ colmean, void* __restrict__ out, int L,
                                                 int D, int BLK, int nblk, int tiled, int bx, int bh,
                                                 uint16_t* __restrict__ cast = nullptr) {
  typedef VecIo<IO, W> Vec;
  constexpr bool NARROW = W * sizeof(typename IO::raw) == 4;
  const int tpr = D / W;
  const int bpw = NT / tpr;
  const int sub = threadIdx.x / tpr;
  const int blk = bx * bpw + sub;
  const int c = (threadIdx.x - sub * tpr) * W;
  if (sub >= bpw || blk >= nblk) return;
  const int row0 = blk * BLK;
  const int nrows = min(BLK, L - row0);
  float acc[W];
  float cm[W];
#pragma unroll
  for (int e = 0; e < W; ++e) acc[e] = 0.f;
  if (MODE == 2) {
    const Vec m = *reinterpret_cast<const Vec*>(colmean + c);
#pragma unroll
    for (int e = 0; e < W; ++e) cm[e] = IO::ld(m.e[e]);
  }
  const size_t pitch = (size_t)lay.sl;
  const size_t at = lay.head(bh) + (size_t)row0 * pitch + c;
  const typename IO::raw* p = x + at;
  const auto add_row = [&](const Vec& v, int r) __attribute__((always_inline)) {
#pragma unroll
    for (int e = 0; e < W; ++e) {
      float f = IO::ld(v.e[e]);
      if (MODE == 2) f = IO::ld(IO::st(f - cm[e]));
      acc[e] = acc[e] + f;
    }
    if constexpr (!__is_same(Cast, NoCast)) {
      VecIo<IoBf16, W> h;
#pragma unroll
      for (int e = 0; e < W; ++e) h.e[e] = Elem<Cast>::from_float(IO::ld(v.e[e]));
      *reinterpret_cast<VecIo<IoBf16, W>*>(cast + at + (size_t)r * pitch) = h;
    }
  };
  // a batch of rows is fetched (all its loads in flight together), then added in row order
  constexpr int BATCH = NARROW ? (NT == 512 ? 32 : 64) : 16;
  int r = 0;
  for (; r + BATCH <= nrows; r += BATCH) {
    Vec v[BATCH];
#pragma unroll
    for (int i = 0; i < BATCH; ++i) v[i] = *reinterpret_cast<const Vec*>(p + (size_t)(r + i) * pitch);
#pragma unroll
    for (int i = 0; i < BATCH; ++i) add_row(v[i], r + i);
  }
  if (r < nrows) {             // the rest of a ragged block likewise, its last row again where there is none
    Vec v[BATCH];
#pragma unroll
    for (int i = 0; i < BATCH; ++i) v[i] = *reinterpret_cast<const Vec*>(p + (size_t)min(r + i, nrows - 1) * pitch);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < BATCH; ++i)
      if (r + i < nrows) add_row(v[i], r + i);
  }
  const size_t o = ((size_t)bh * nblk + blk) * D + c;
  if (MODE == 0) {
    float* of = reinterpret_cast<float*>(out) + o;
#pragma unroll
    for (int e = 0; e < W; ++e) of[e] = acc[e];
  } else {
    const float cnt = (float)nrows;
    Vec m;
#pragma unroll
    for (int e = 0; e < W; ++e) m.e[e] = IO::st(acc[e] / cnt);
    if constexpr (IO::VEC == 8) {
      if (tiled) {             // even and odd columns, each kind adjacent in its places
        uint16_t* t = reinterpret_cast<uint16_t*>(out) + tiled_head(bh, nblk, D);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          if constexpr (W == 8) {
            i16x4_t w;
#pragma unroll
            for (int j = 0; j < 4; ++j) w[j] = (short)m.e[2 * j + h];
            *reinterpret_cast<i16x4_t*>(t + tiled_pos(blk, c + h, D)) = w;
          } else {
            t[tiled_pos(blk, c + h, D)] = m.e[h];
          }
        }
        return;
      }
    }
    *reinterpret_cast<Vec*>(reinterpret_cast<typename IO::raw*>(out) + o) = m;
  }
}

// kind 0: block means of q (MODE 1); kind 1: fp32 chunk sums of k (MODE 0, chunks of KMEAN_CHUNK rows).  K comes
// second because the next pass reads it again: what of it is still in the memory-side cache then is the part read last
// (module forward at B1 H12 L32760: 0.493 against 0.498 ms with k first).  cast: 16-bit copies of q, then of k, n elements each.
template <typename IO, int W, typename Cast = NoCast>
static __device__ __forceinline__ void pool_pair_body(const typename IO::raw* __restrict__ k, float* __restrict__ chunk_sums,
                                                      int nchunk, const typename IO::raw* __restrict__ q, const RowLayout lay,
                                                      typename IO::raw* __restrict__ pq, int BLKQ, int nblkq, int L, int D,
                                                      int tiled, int bx, int bh, int kind, uint16_t* __restrict__ cast = nullptr,
                                                      int64_t n = 0) {
  if (kind == 1)
    pool_body<IO, 0, W, 256, Cast>(k, lay, nullptr, chunk_sums, L, D, KMEAN_CHUNK, nchunk, 0, bx, bh, cast + n);
  else
    pool_body<IO, 1, W, 256, Cast>(q, lay, nullptr, pq, L, D, BLKQ, nblkq, tiled, bx, bh, cast);
}

// One thread per 4 bytes of a block's columns while the first pass of the wide form would not put a wave on every SIMD.
static inline bool narrow_pools(int dtype, int BH, int L, int D) {
  return (int64_t)BH * cdiv(L, KMEAN_CHUNK) * D * elem_bytes(dtype) / 16 < 1024 * 64;
}

// Column mean of K, levels 2 and 3 of the summation order: one workgroup of NT threads per (head, slab of COLMEAN_SLAB
// columns), thread (gi, c) = (tid / COLMEAN_SLAB, tid % COLMEAN_SLAB) forms group sums gi, gi + NT / COLMEAN_SLAB, ...
// of its column; the first COLMEAN_SLAB threads then add the groups in ascending order.  (256 threads where it is a launch of its
// own or shares one with v's scales, 512 beside the slices' partial states.)
constexpr int COLMEAN_SLAB = 16;
constexpr int COLMEAN_MAX_GROUPS = 256;
template <typename IO, int NT>
static __device__ __forceinline__ void colmean_body(const float* __restrict__ chunk_sums, typename IO::raw* __restrict__ colmean,
                                                    int nchunk, int ngroup, int D, int L, int slab, int bh, float* gs) {
  const int tid = threadIdx.x;
  const int c = tid % COLMEAN_SLAB, d = slab * COLMEAN_SLAB + c;
  for (int g = tid / COLMEAN_SLAB; g < ngroup; g += NT / COLMEAN_SLAB) {
    const int c0 = g * KMEAN_GROUP;
    const int n = min(KMEAN_GROUP, nchunk - c0);
    // (a group's loads all in flight, then added in order: mask builder of 16 heads x 6001 x 64 25.3 -> 23.2 us, of 40 x 75600 x 128 656 -> 652)
    const float* p = chunk_sums + ((size_t)bh * nchunk + c0) * D + d;
    float x[KMEAN_GROUP];
#pragma unroll
    for (int i = 0; i < KMEAN_GROUP; ++i) x[i] = p[(size_t)min(i, n - 1) * D];
    __builtin_amdgcn_sched_barrier(0);
    float acc = 0.f;
#pragma unroll
    for (int i = 0; i < KMEAN_GROUP; ++i)
      if (i < n) acc = acc + x[i];
    gs[g * COLMEAN_SLAB + c] = acc;
  }
  __syncthreads();
  if (tid < COLMEAN_SLAB) {
    float acc = 0.f;
    for (int g = 0; g < ngroup; ++g) acc = acc + gs[g * COLMEAN_SLAB + tid];
    colmean[(size_t)bh * D + d] = IO::st(acc / (float)L);
  }
}

// The same mean by one workgroup of NT threads for every column of a head, into LDS: for a launch whose workgroups each want it and
// may not wait for a launch that forms it.  gs: COLMEAN_LDS_GROUPS * D words of LDS; `out`: D numbers of LDS, in place behind a barrier.
constexpr int COLMEAN_LDS_GROUPS = 8;
template <typename IO, int D, int NT>
static __device__ __forceinline__ void colmean_all_body(const float* __restrict__ chunk_sums, int nchunk, int L, int bh, float* gs,
                                                        typename IO::raw* out) {
  const int d = threadIdx.x % D, ngroup = (nchunk + KMEAN_GROUP - 1) / KMEAN_GROUP;
  float total = 0.f;
  for (int g0 = 0; g0 < ngroup; g0 += COLMEAN_LDS_GROUPS) {
    if (g0) __syncthreads();
    for (int g = (int)threadIdx.x / D; g < COLMEAN_LDS_GROUPS && g0 + g < ngroup; g += NT / D) {
      const int c0 = (g0 + g) * KMEAN_GROUP;
      const int n = min(KMEAN_GROUP, nchunk - c0);
      const float* p = chunk_sums + ((size_t)bh * nchunk + c0) * D + d;
      float x[KMEAN_GROUP];
#pragma unroll
      for (int i = 0; i < KMEAN_GROUP; ++i) x[i] = p[(size_t)min(i, n - 1) * D];
      __builtin_amdgcn_sched_barrier(0);
      float acc = 0.f;
#pragma unroll
      for (int i = 0; i < KMEAN_GROUP; ++i)
        if (i < n) acc = acc + x[i];
      gs[g * D + d] = acc;
    }
    __syncthreads();
    if (threadIdx.x < D)
      for (int g = 0; g < COLMEAN_LDS_GROUPS && g0 + g < ngroup; ++g) total = total + gs[g * D + d];
  }
  if (threadIdx.x < D) out[d] = IO::st(total / (float)L);
  __syncthreads();
}

}  // namespace sla
