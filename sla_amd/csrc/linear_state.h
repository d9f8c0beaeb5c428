// phi(K)^T V and sum phi(K) state kernels of the linear branch (used by forward and backward).
#pragma once
#include "linear_common.h"

namespace sla {

// ---- kernel 1: partial states -----------------------------------------------------------
// grid (nsplit, BH).  Thread t moves 16-byte chunk (t%CPR) of rows t/CPR + i*RPP.
// A slice is a chain of tiles, each a memory latency, the feature map and the products' reads of LDS: two tiles are in flight in
// registers beside the one in LDS, and eight waves share a tile (head dim 128: 64 rows, two 32 x 32 parts of the state per wave;
// head dim 64: 128 rows, one part per wave and half of the rows, the halves added at the end).  Against four waves per 64 rows
// with one tile in flight, each row's sums through LDS: 8 heads x 4096 x 128, softmax map 19.8 -> 14.3 us, 16 heads x 6001 x 64
// 13.6 -> 11.8, 12 heads x 32760 x 128 beside the mask builder 79.5 -> 76.5.
// OUT16 (one tile of 64 rows per workgroup): four waves.
// OUT16: the D x D partial is written rounded to 16 bit (per-key-block states of the complement mode).
// ZW: zweight holds one fp32 per row of the head, (BH, L), and the z partial becomes sum_rows zweight * phi(k)
// instead of sum_rows phi(k) (used by the complement backward, where "k" is q and "v" a row gradient).
// VMAX: the largest |v| of every column over the slice goes to vmax_part[bh][split][D] (what the FP8 quantiser of v
// needs of v before it can start: v is streamed here anyway).
// IDENT: phi is the identity (the projection's gradients: d(out)^T y, with the sum of d(out) as z).
template <int D, bool OUT16>
struct StateTile {
  static constexpr int NTH = OUT16 ? 256 : 512;                    // threads
  static constexpr int GROUPS = D == 64 && !OUT16 ? 2 : 1;         // groups of 64 rows, each with its own waves
  static constexpr int TR = 64 * GROUPS;                           // rows per LDS tile
  static constexpr int DEPTH = OUT16 ? 1 : 2;                      // tiles in flight in registers
  static constexpr int STR = D + 16;                               // LDS row stride: transposed reads of 4 rows hit disjoint banks
  static constexpr int LDS = 2 * TR * STR * 2;                     // bytes; the final sums reuse it
};
template <typename Tag, int D, bool OUT16, bool ZW, bool VMAX, bool IDENT = false>
static __device__ __forceinline__ void state_partial_body(const uint16_t* __restrict__ k, const uint16_t* __restrict__ v,
                                                          const RowLayout lay, void* __restrict__ kv_part_,
                                                          float* __restrict__ z_part, int L, int rows_per_split, int fmap,
                                                          const float* __restrict__ zweight, float* __restrict__ vmax_part,
                                                          int split, int bh, int nsplit, char* smem) {
  using E = Elem<Tag>;
  using T = StateTile<D, OUT16>;
  constexpr int TR = T::TR, STR = T::STR, NTH = T::NTH, DEPTH = T::DEPTH;
  constexpr int CPR = D / 8;             // 16-byte chunks per row
  constexpr int RPP = NTH / CPR;         // rows covered by one pass of the workgroup
  constexpr int NP = TR / RPP;           // passes per tile
  constexpr int DT = D / 32;             // 32-wide parts of the state along either dimension
  constexpr int NWG = NTH / 64 / T::GROUPS;    // waves per group of rows
  constexpr int WPT = (DT * DT) / NWG;   // parts per wave
  static_assert(DT * DT % NWG == 0, "the parts of the state must divide among the waves");

  uint16_t* const sK = reinterpret_cast<uint16_t*>(smem);
  uint16_t* const sV = sK + TR * STR;
  float (*sZ)[D] = reinterpret_cast<float (*)[D]>(smem);
  static_assert(RPP * D * 4 <= T::LDS && (T::GROUPS == 1 || NWG * 64 * 16 * 4 <= T::LDS), "the final sums do not fit the tiles");

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int g = lane >> 5;
  const int row_begin = split * rows_per_split;
  const int row_end = min(L, row_begin + rows_per_split);
  // (slices are whole tiles but for the last of a head: rows past it lie outside the descriptors and read as zero)
  const __amdgpu_buffer_rsrc_t k_rs = make_rsrc(k + lay.head(bh), lay.head_range_bytes(L, D));
  const __amdgpu_buffer_rsrc_t v_rs = make_rsrc(v + lay.head(bh), lay.head_range_bytes(L, D));
  const __amdgpu_buffer_rsrc_t w_rs = make_rsrc(ZW ? zweight + (size_t)bh * L : nullptr, ZW ? (uint32_t)L * 4u : 0u);
  const uint32_t pitch_b = (uint32_t)lay.sl * 2u;

  const int lrow = tid / CPR, lcol = (tid % CPR) * 8;

  // wave w of its group owns parts w*WPT .. w*WPT+WPT-1; part = d1part*DT + d2part
  const int gw = wave % NWG, group = wave / NWG;
  f32x16_t acc[WPT];
#pragma unroll
  for (int t = 0; t < WPT; ++t)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[t][i] = 0.f;
  float zacc[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) zacc[e] = 0.f;
  // |v| of this thread's eight columns as 16-bit patterns without their sign bits: for bf16 and f16 alike the larger
  // magnitude has the larger pattern, so a packed unsigned maximum keeps two columns per register
  typedef unsigned short u16x2_t __attribute__((ext_vector_type(2)));
  u16x2_t vmx[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) vmx[j] = u16x2_t{0, 0};

  const int tr_row = (lane & 15) >> 2;
  const int tr_col = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);

  // rows of the next tiles are fetched into registers while the current tile is multiplied
  i16x8_t kreg[DEPTH][NP], vreg[DEPTH][NP];
  float wreg[DEPTH][NP];
  auto fetch = [&](int r0, int s) __attribute__((always_inline)) {
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const uint32_t grow = (uint32_t)(r0 + lrow + p * RPP);
      kreg[s][p] = buf_load_b128(k_rs, grow * pitch_b + 2u * (uint32_t)lcol);
      vreg[s][p] = buf_load_b128(v_rs, grow * pitch_b + 2u * (uint32_t)lcol);
      wreg[s][p] = ZW ? __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(w_rs, (int)(grow * 4u), 0, 0)) : 1.0f;
    }
  };
  if (row_begin < row_end)
#pragma unroll
    for (int s = 0; s < DEPTH; ++s) fetch(row_begin + s * TR, s);
  const auto tile = [&](int r0, int s) __attribute__((always_inline)) {
    lds_barrier();
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const int row = lrow + p * RPP;
      const int grow = r0 + row;
      const i16x8_t kk = kreg[s][p], vv = vreg[s][p];
      const bool ok = grow < row_end;
      float f[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) f[e] = E::to_float((uint16_t)kk[e]);
      if constexpr (IDENT) {
      } else if (fmap == SLA_FMAP_SOFTMAX) {
        // the CPR lanes that share this row are adjacent: reduce max and sum across them
        float mx = f[0];
#pragma unroll
        for (int e = 1; e < 8; ++e) mx = fmaxf(mx, f[e]);
        mx = over_lanes<CPR>(mx, [](float a, float b) { return fmaxf(a, b); });
        float sum = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          f[e] = __expf(f[e] - mx);
          sum += f[e];
        }
        sum = over_lanes<CPR>(sum, [](float a, float b) { return a + b; });
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
      i16x8_t fk;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        if (!ok) f[e] = 0.f;              // rows past the end take no part (phi(0) is not 0 for elu/softmax)
        zacc[e] += ZW ? wreg[s][p] * f[e] : f[e];
        fk[e] = (short)E::from_float(f[e]);
      }
      *reinterpret_cast<i16x8_t*>(&sK[row * STR + lcol]) = fk;
      *reinterpret_cast<i16x8_t*>(&sV[row * STR + lcol]) = vv;
      if (VMAX) {                          // (rows past the end were fetched as zeros)
        const i32x4_t vw = __builtin_bit_cast(i32x4_t, vv);
#pragma unroll
        for (int j = 0; j < 4; ++j)
          vmx[j] = __builtin_elementwise_max(vmx[j], __builtin_bit_cast(u16x2_t, vw[j] & 0x7fff7fff));
      }
    }
    lds_barrier();
    if (r0 + DEPTH * TR < row_end) fetch(r0 + DEPTH * TR, s);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int l0 = 64 * group + 16 * c + 8 * g + tr_row;
#pragma unroll
      for (int t = 0; t < WPT; ++t) {
        const int d1t = (gw * WPT + t) / DT, d2t = (gw * WPT + t) % DT;
        const uint16_t* pa = &sK[l0 * STR + 32 * d1t + tr_col];
        const uint16_t* pb = &sV[l0 * STR + 32 * d2t + tr_col];
        const i16x8_t a = concat4(lds_read_tr16(pa), lds_read_tr16(pa + 4 * STR));
        const i16x8_t b = concat4(lds_read_tr16(pb), lds_read_tr16(pb + 4 * STR));
        acc[t] = E::mfma32(a, b, acc[t]);
      }
    }
  };
  for (int r0 = row_begin; r0 < row_end; r0 += DEPTH * TR)
#pragma unroll
    for (int s = 0; s < DEPTH; ++s)
      if (s == 0 || r0 + s * TR < row_end) tile(r0 + s * TR, s);

  lds_barrier();             // (the tiles are free)
  if constexpr (T::GROUPS == 2) {
    static_assert(WPT == 1, "one part per wave");
    f32x16_t* const other = reinterpret_cast<f32x16_t*>(smem) + (size_t)gw * 64 + lane;
    if (group) *other = acc[0];
    lds_barrier();
    if (!group) acc[0] += *other;
    lds_barrier();
  }
  // partial KV, stored transposed: kv_part[bh][split][d2][d1]
  const size_t part_off = ((size_t)bh * nsplit + split) * D * D;
  // (16 bit: through LDS, so that whole lines leave; a lane's pieces are 8 bytes of 32 rows.  States of 256 blocks of 12 heads x 128:
  //  kernel 53 -> 36.5 us; forward and backward of the branch there 494 -> 468 us, 12 x 9000 x 128 318 -> 301, 24 x 10000 x 64 224.6 ->
  //  222.9.  fp32 leaves in pieces of 32 bytes, where LDS gains nothing: 16 x 5003 x 64, quantised, 74.3 -> 74.9)
  constexpr int OSTR = D + 8;
  uint16_t* const sOut = reinterpret_cast<uint16_t*>(smem);
  static_assert(!OUT16 || (D * OSTR * 2 <= T::LDS && T::GROUPS == 1 && D * D % (8 * NTH) == 0), "the state does not fit the tiles");
#pragma unroll
  for (int t = 0; t < WPT; ++t) {
    if (group) break;
    const int d1t = (gw * WPT + t) / DT, d2t = (gw * WPT + t) % DT;
    const int d2 = 32 * d2t + (lane & 31);
#pragma unroll
    for (int i4 = 0; i4 < 4; ++i4) {
      const size_t o = part_off + (size_t)d2 * D + 32 * d1t + 8 * i4 + 4 * g;
      if (OUT16) {
        i32x2_t w;
        w[0] = (int)E::pack2(acc[t][4 * i4], acc[t][4 * i4 + 1]);
        w[1] = (int)E::pack2(acc[t][4 * i4 + 2], acc[t][4 * i4 + 3]);
        *reinterpret_cast<i32x2_t*>(&sOut[d2 * OSTR + 32 * d1t + 8 * i4 + 4 * g]) = w;
      } else {
        f32x4_t w = {acc[t][4 * i4], acc[t][4 * i4 + 1], acc[t][4 * i4 + 2], acc[t][4 * i4 + 3]};
        *reinterpret_cast<f32x4_t*>(reinterpret_cast<float*>(kv_part_) + o) = w;
      }
    }
  }
  if constexpr (OUT16) {
    lds_barrier();
#pragma unroll
    for (int p = 0; p < D * D / 8 / NTH; ++p) {
      const int idx = (tid + NTH * p) * 8;
      *reinterpret_cast<i16x8_t*>(reinterpret_cast<uint16_t*>(kv_part_) + part_off + idx) =
          *reinterpret_cast<const i16x8_t*>(&sOut[idx / D * OSTR + idx % D]);
    }
    lds_barrier();
  }
  // partial z: reduce the RPP row groups through LDS
#pragma unroll
  for (int x = 0; x < 2; ++x)
    *reinterpret_cast<f32x4_t*>(&sZ[lrow][lcol + 4 * x]) = f32x4_t{zacc[4 * x], zacc[4 * x + 1], zacc[4 * x + 2], zacc[4 * x + 3]};
  lds_barrier();
  if (tid < D) {
    float s = 0.f;
#pragma unroll
    for (int r = 0; r < RPP; ++r) s += sZ[r][tid];
    z_part[((size_t)bh * nsplit + split) * D + tid] = s;
  }
  if (VMAX) {
    lds_barrier();
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      sZ[lrow][lcol + 2 * j] = E::to_float(vmx[j][0]);
      sZ[lrow][lcol + 2 * j + 1] = E::to_float(vmx[j][1]);
    }
    lds_barrier();
    if (tid < D) {
      float a = 0.f;
#pragma unroll
      for (int r = 0; r < RPP; ++r) a = fmaxf(a, sZ[r][tid]);
      vmax_part[((size_t)bh * nsplit + split) * D + tid] = a;
    }
  }
}

template <typename Tag, int D, bool OUT16 = false, bool ZW = false, bool VMAX = false, bool IDENT = false>
__global__ __launch_bounds__((StateTile<D, OUT16>::NTH)) __attribute__((amdgpu_waves_per_eu(OUT16 ? 3 : 4, OUT16 ? 3 : 4))) void linear_state_partial_kernel(
    const uint16_t* __restrict__ k, const uint16_t* __restrict__ v, const RowLayout lay, void* __restrict__ kv_part,
    float* __restrict__ z_part, int L, int rows_per_split, int fmap, const float* __restrict__ zweight = nullptr,
    float* __restrict__ vmax_part = nullptr) {
  __shared__ __attribute__((aligned(16))) char smem[StateTile<D, OUT16>::LDS];
  state_partial_body<Tag, D, OUT16, ZW, VMAX, IDENT>(k, v, lay, kv_part, z_part, L, rows_per_split, fmap, zweight, vmax_part,
                                                     blockIdx.x, blockIdx.y, gridDim.x, smem);
}

// 16-bit copy of the projection weight as the A operand of dY^T = W^T G^T, in the order in which a wave reads it: 32 rows d x 16
// columns e after one another, a lane's eight columns together.  One thread per element.
template <typename Tag>
__global__ void linear_prep_weight_kernel(const float* __restrict__ weight, uint16_t* __restrict__ wt, int D) {
  using E = Elem<Tag>;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= D * D) return;
  const int e = i / D, d = i % D;
  const uint16_t h = E::from_float(weight[i]);
  wt[(((d >> 5) * (D / 16) + (e >> 4)) * 64 + 32 * (e >> 3 & 1) + (d & 31)) * 8 + (e & 7)] = h;
}

// ---- kernel 2 (forward, and a backward that has to rebuild the states): finish the states ----------------------------
// From the slices' partial states of a head: their sums in ascending slice order, rounded to 16 bit (kvt, the transposed
// state; z), and with the projection folded in
//   kvwt[bh][e][d1] = round16( sum_d2 round16(W[e][d2]) * KVT[d2][d1] ), fp32 accumulation:
// (phi(Q) KV / den) W^T = (phi(Q) (KV W^T)) / den, so the output kernel needs one product per query tile.  kvw[d1][e] is that
// matrix for the backward, from the sums before their rounding (fp32 products): dq's relative error against 64 bits 4.13e-3
// where twice rounded sums leave 4.66e-3 (softmax map, 4 heads x 6001 x 64 in bf16).
// One workgroup of 512 threads per head and 16 columns d1 (neighbouring workgroups on one XCD, so that the two halves of a
// 128-byte line meet in its L2): the two halves of the workgroup sum one half of the slices each, over every row d2, and meet
// in LDS; holding all a row of kvwt needs of the state, the workgroup then multiplies by W on the matrix cores.  Bound by
// latency: the loads of eight slices and the workgroup's rows of W are in flight at once.
// Against a summing and a folding kernel (the latter on the vector ALU), B1 H12 L9360 D128: 16.3 against 10.1 + 8.5 us and one
// launch less; state build of 40 heads x 32760 x 128: 159 against 172 us, of 16 heads x 6001 x 64: 17.5 against 20.9.
template <int NV, int BATCH = 8>
static __device__ __forceinline__ void sum_slices(const float* __restrict__ p, int n, size_t slice_stride, size_t vec_stride,
                                                  f32x4_t (&acc)[NV]) {
  // acc[i] += the 16 bytes at p + i vec_stride of n slices, in ascending order, BATCH slices' loads in flight
  int sp = 0;
  for (; sp + BATCH <= n; sp += BATCH) {
    f32x4_t b[BATCH][NV];
#pragma unroll
    for (int x = 0; x < BATCH; ++x)
#pragma unroll
      for (int i = 0; i < NV; ++i) b[x][i] = *reinterpret_cast<const f32x4_t*>(p + (size_t)(sp + x) * slice_stride + i * vec_stride);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int x = 0; x < BATCH; ++x)
#pragma unroll
      for (int i = 0; i < NV; ++i) acc[i] += b[x][i];
  }
  if (sp < n) {                      // the rest: the last slice again where there is none, not added
    f32x4_t b[BATCH][NV];
#pragma unroll
    for (int x = 0; x < BATCH; ++x)
#pragma unroll
      for (int i = 0; i < NV; ++i)
        b[x][i] = *reinterpret_cast<const f32x4_t*>(p + (size_t)min(sp + x, n - 1) * slice_stride + i * vec_stride);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int x = 0; x < BATCH; ++x)
      if (sp + x < n) {
#pragma unroll
        for (int i = 0; i < NV; ++i) acc[i] += b[x][i];
      }
  }
}

// The same sums in a launch of their own, left in the place of every head's first slice, with the same bits.  The kernel
// below has D / 16 workgroups per head: few heads with many slices leave it reading on a few compute units.  Here a workgroup
// of 512 threads takes 256 elements, its halves one half of the slices each, 32 loads in flight; the last one of a head takes z,
// another one behind it (the backward's sums have one) a second vector.
// Bound by latency.  State build in us without this launch and with it: 1 head x 75600 x 128 (256 slices) 72.0 / 29.6, 2 heads x
// 75600 x 128 (128) 54.8 / 35.6, 4 heads x 32760 x 128 (64) 39.6 / 32.7, 8 heads x 16384 x 64 (32) 18.7 / 17.8, 12 heads x 24576 x
// 128 (21) 52.3 / 51.6, 16 heads x 16384 x 128 (16) 45.7 / 48.4.  Among the other launches of a forward the line lies between 36 and
// 50 slices; whole forward without / with: 128 columns 6 heads x 14000 (37) 106.8 / 101.7, 8 x 14000 (32) 120.8 / 121.8, 8 x 20000
// (32) 136.1 / 137.3; 64 columns 5 x 17000 (45) 70.2 / 72.1, 3 x 12000 (47) 49.6 / 51.2, 4 x 14000 (55) 53.8 / 52.3; quantised 6 x
// 10000 x 128 (40) 85.5 / 89.3, 6 x 12000 x 128 (38) 117.3 / 113.5, 5 x 25000 x 64 (49) 112.4 / 109.4.
template <int D>
__global__ __launch_bounds__(512) void linear_state_presum_kernel(float* __restrict__ kv_part, float* __restrict__ z_part,
                                                                  float* __restrict__ z2_part, int nsplit) {
  constexpr int DD = D * D, BATCH = 32;
  __shared__ float s_half[256];
  const int bh = blockIdx.y, tid = threadIdx.x & 255, half = threadIdx.x >> 8;
  const auto sum = [](const float* p, int n, size_t stride) __attribute__((always_inline)) {
    float acc = 0.f;
    for (int sp = 0; sp < n; sp += BATCH) {
      float x[BATCH];
#pragma unroll
      for (int i = 0; i < BATCH; ++i) x[i] = p[(size_t)min(sp + i, n - 1) * stride];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < BATCH; ++i)
        if (sp + i < n) acc += x[i];
    }
    return acc;
  };
  if (blockIdx.x >= DD / 256) {
    float* p = (blockIdx.x == DD / 256 ? z_part : z2_part) + (size_t)bh * nsplit * D + threadIdx.x;
    if (threadIdx.x < D) *p = sum(p, nsplit, D);
    return;
  }
  float* p = kv_part + (size_t)bh * nsplit * DD + blockIdx.x * 256 + tid;
  const int n0 = (nsplit + 1) >> 1;
  const float acc = half ? sum(p + (size_t)n0 * DD, nsplit - n0, DD) : sum(p, n0, DD);
  if (half) s_half[tid] = acc;
  __syncthreads();
  if (!half) *p = acc + s_half[tid];
}

// (nsum: the slices to add up, all nsplit of a head or the first one alone, which then holds the sums)
struct StateFinish {
  const float *kv_part, *z_part, *weight;
  uint16_t *kvt, *kvw, *kvwt, *z;
  int nsplit, nsum, total;                 // total = heads x D / 16 workgroups
};
template <int D>
constexpr int state_finish_lds() { return D / 64 * 256 * 16 + 16 * (D + 4) * 4 + 16 * (D + 8) * 2; }       // bytes
template <typename Tag, int D>
static __device__ __forceinline__ void state_finish_body(const StateFinish& job, int logical, char* smem) {
  const float *kv_part = job.kv_part, *z_part = job.z_part, *weight = job.weight;
  uint16_t *kvt = job.kvt, *kvw = job.kvw, *kvwt = job.kvwt, *z = job.z;
  const int nsplit = job.nsplit, nsum = job.nsum;
  using E = Elem<Tag>;
  constexpr int DD = D * D;
  constexpr int STR = D + 8;               // row pitch of the strip in LDS
  constexpr int NR = D / 64;               // rows d2 per thread
  constexpr int STR32 = D + 4;
  float* const s_half = reinterpret_cast<float*>(smem);                   // sums of the upper half of the slices
  float* const s_kv32 = s_half + NR * 256 * 4;                            // [d1][d2] before rounding
  uint16_t* const s_kv = reinterpret_cast<uint16_t*>(s_kv32 + 16 * STR32); // [d1][d2]
  const int bh = logical / (D / 16), d1_0 = 16 * (logical % (D / 16));
  const int tid = threadIdx.x & 255, half = threadIdx.x >> 8, lane = tid & 63, wave = threadIdx.x >> 6;
  const int l = lane & 15, h = lane >> 4;
  const int tile = wave < D / 16 ? wave : 0;         // 16 rows e per wave (head dim 64: four of the eight waves)

  // B operand of (KV W^T)^T = KV^T-strip x W^T: column e = 16 tile + l, rows d2 = 32 c + 8 h ..
  f32x4_t wraw[D / 32][2];
#pragma unroll
  for (int c = 0; c < D / 32; ++c)
#pragma unroll
    for (int x = 0; x < 2; ++x)
      wraw[c][x] = *reinterpret_cast<const f32x4_t*>(weight + (size_t)(16 * tile + l) * D + 32 * c + 8 * h + 4 * x);

  const int dr = tid >> 2, dc = 4 * (tid & 3);      // rows dr (+ 64), columns d1_0 + dc .. + 3
  f32x4_t acc[NR];
#pragma unroll
  for (int i = 0; i < NR; ++i) acc[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const int n0 = (nsum + 1) >> 1, first = half ? n0 : 0, n = half ? nsum - n0 : n0;
  sum_slices<NR>(kv_part + ((size_t)bh * nsplit + first) * DD + (size_t)dr * D + d1_0 + dc, n, DD, (size_t)64 * D, acc);
  if (half) {
#pragma unroll
    for (int i = 0; i < NR; ++i) *reinterpret_cast<f32x4_t*>(s_half + (i * 256 + tid) * 4) = acc[i];
    if (tid < 16) {
      const float* pz = z_part + (size_t)bh * nsplit * D + d1_0 + tid;
      float sum = 0.f;
#pragma unroll 8
      for (int sp = 0; sp < nsum; ++sp) sum += pz[(size_t)sp * D];
      z[(size_t)bh * D + d1_0 + tid] = E::from_float(sum);
    }
  }
  __syncthreads();
  if (!half) {
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const int d2 = dr + 64 * i;
      acc[i] += *reinterpret_cast<const f32x4_t*>(s_half + (i * 256 + tid) * 4);
      i32x2_t w;
      w[0] = (int)E::pack2(acc[i][0], acc[i][1]);
      w[1] = (int)E::pack2(acc[i][2], acc[i][3]);
      *reinterpret_cast<i32x2_t*>(kvt + (size_t)bh * DD + (size_t)d2 * D + d1_0 + dc) = w;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        s_kv[(dc + j) * STR + d2] = (uint16_t)((uint32_t)w[j >> 1] >> (16 * (j & 1)));
        s_kv32[(dc + j) * STR32 + d2] = acc[i][j];
      }
    }
  }
  __syncthreads();
  if (wave >= D / 16) return;
  f32x4_t o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int c = 0; c < D / 32; ++c) {
    i32x4_t w;
#pragma unroll
    for (int x = 0; x < 4; ++x) w[x] = (int)E::pack2(wraw[c][x >> 1][2 * (x & 1)], wraw[c][x >> 1][2 * (x & 1) + 1]);
    o = E::mfma16(*reinterpret_cast<const i16x8_t*>(s_kv + l * STR + 32 * c + 8 * h), __builtin_bit_cast(i16x8_t, w), o);
  }
  // rows d1 = 4 h + i, column e
  i32x2_t w;
  w[0] = (int)E::pack2(o[0], o[1]);
  w[1] = (int)E::pack2(o[2], o[3]);
  *reinterpret_cast<i32x2_t*>(kvwt + (size_t)bh * DD + (size_t)(16 * tile + l) * D + d1_0 + 4 * h) = w;
  f32x4_t p = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int c = 0; c < D / 32; ++c)
#pragma unroll
    for (int x = 0; x < 2; ++x) {
      const f32x4_t a = *reinterpret_cast<const f32x4_t*>(s_kv32 + l * STR32 + 32 * c + 8 * h + 4 * x);
#pragma unroll
      for (int j = 0; j < 4; ++j) p = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j], round16<Tag>(wraw[c][x][j]), p, 0, 0, 0);
    }
#pragma unroll
  for (int i = 0; i < 4; ++i) kvw[(size_t)bh * DD + (size_t)(d1_0 + 4 * h + i) * D + 16 * tile + l] = E::from_float(p[i]);
}

// ---- workspace layout of the state build -----------------------------------------------------
// The finished states (kvt .. z) come first: `states_end` bytes that a caller may copy aside after the
// forward and put back at the start of the backward's workspace instead of having them rebuilt.
struct LinWs {
  int nsplit, rows_per_split;
  size_t kvt, kvw, kvwt, z, states_end, kv_part, z_part, vmax_part, total;
};

static inline LinWs lin_ws(int BH, int L, int D) {
  LinWs w;
  // One workgroup per compute unit (256 slots): more, shorter slices only add partial states to write and to add up again by few
  // workgroups (module forward, two per unit / one: 12 heads x 14000 x 128 225.6 / 222.6 us, 24 x 2500 x 128 66.5 / 60.4, 32 x 1500 x
  // 128 60.3 / 57.3, 36 x 2500 x 128 90.4 / 86.5, 48 x 2500 x 64 60.3 / 58.9, 80 x 1500 x 128 100.5 / 97.6).  Two (512 slots)
  // - where the whole slices of all heads leave more than three of sixteen units without one (one per unit / two: 129 heads x 2000 x 128
  //   230 / 186, 130 x 6000 x 64 329 / 296, 96 x 2500 x 64 94.0 / 91.1, 100 x 2500 x 128 183.0 / 179.3; with 210 of 256 or more, 72 x 2500
  //   x 128 139.9 / 139.7, 112 x 2500 x 128 195 / 204, 128 x 2500 x 128 219 / 236);
  // - above 64 Mi elements, where the sums are a small part: 40 heads x 32760 x 128, quantised 2153 / 2141.
  // Short sequences: at most sixteen slices, or slices of 256
  // rows; more only lengthen the chain that adds them up (state build of 8 heads x 4096 rows x 128: 64 slices 34.6 us, 16
  // slices 23.8; 4 heads x 7813 x 64: 123 slices 23.5, 31 slices 15.3; with 1024 rows 16 slices of 64 rows 14.7, 4 of 256 19.4).
  const int min_rows = L >= 4096 ? 256 : cdiv(L, 16);
  const int slots = (int64_t)BH * L * D <= (64ll << 20) && BH * (256 / BH) >= 208 ? 256 : 512;
  const int tr = D == 64 ? StateTile<64, false>::TR : StateTile<128, false>::TR;
  const LinSplit sp = lin_split(BH, L, slots, tr, min_rows);
  w.nsplit = sp.nsplit;
  w.rows_per_split = sp.rows_per_split;
  size_t off = 0;
  w.kvt = off;     off += align_up((int64_t)BH * D * D * 2, 256);
  w.kvw = off;     off += align_up((int64_t)BH * D * D * 2, 256);
  w.kvwt = off;    off += align_up((int64_t)BH * D * D * 2, 256);
  w.z = off;       off += align_up((int64_t)BH * D * 2, 256);
  w.states_end = off;
  w.kv_part = off; off += align_up((int64_t)BH * w.nsplit * D * D * 4, 256);
  w.z_part = off;  off += align_up((int64_t)BH * w.nsplit * D * 4, 256);
  w.vmax_part = off; off += align_up((int64_t)BH * w.nsplit * D * 4, 256);      // (filled on request: column maxima of |v| per slice)
  w.total = off;
  return w;
}


template <typename Tag, int D>
__global__ __launch_bounds__(512) void linear_state_finish_kernel(const StateFinish job) {
  __shared__ __attribute__((aligned(16))) char smem[state_finish_lds<D>()];
  const int logical = xcd_remap(blockIdx.x, gridDim.x, job.total);
  if (logical >= 0) state_finish_body<Tag, D>(job, logical, smem);
}

constexpr int PRESUM_MIN_SLICES = 40;       // (both sides measured at linear_state_presum_kernel; the backward's at linear_bwd_finish_kernel)

// What is left to do behind the partial states (and, with many slices, behind the launch that adds them up first).  ws: where
// the states go; parts: where the slices' partial sums lie, the offsets of `w` past states_end.
template <int D>
static inline StateFinish state_finish_job(const float* weight, int BH, char* ws, char* parts, const LinWs& w) {
  return StateFinish{(const float*)(parts + (w.kv_part - w.states_end)), (const float*)(parts + (w.z_part - w.states_end)), weight,
                     (uint16_t*)(ws + w.kvt), (uint16_t*)(ws + w.kvw), (uint16_t*)(ws + w.kvwt), (uint16_t*)(ws + w.z), w.nsplit,
                     w.nsplit >= PRESUM_MIN_SLICES ? 1 : w.nsplit, BH * (D / 16)};
}
template <int D>
static inline void launch_state_presum(int BH, char* parts, const LinWs& w, hipStream_t st) {
  if (w.nsplit >= PRESUM_MIN_SLICES)
    hipLaunchKernelGGL((linear_state_presum_kernel<D>), dim3(D * D / 256 + 1, BH), dim3(512), 0, st,
                       (float*)(parts + (w.kv_part - w.states_end)), (float*)(parts + (w.z_part - w.states_end)), nullptr, w.nsplit);
}
template <typename Tag, int D>
static inline void launch_state_finish(const float* weight, int BH, char* ws, char* parts, const LinWs& w, hipStream_t st) {
  launch_state_presum<D>(BH, parts, w, st);
  const StateFinish job = state_finish_job<D>(weight, BH, ws, parts, w);
  hipLaunchKernelGGL((linear_state_finish_kernel<Tag, D>), dim3(xcd_grid(job.total)), dim3(512), 0, st, job);
}

// Streams K and V once and leaves the finished states.
template <typename Tag, int D>
static inline void launch_state_build(const void* k, const void* v, const RowLayout& lay, const float* weight, int fmap,
                                      int BH, int L, char* ws, char* parts, const LinWs& w, hipStream_t st) {
  hipLaunchKernelGGL((linear_state_partial_kernel<Tag, D>), dim3(w.nsplit, BH), dim3(StateTile<D, false>::NTH), 0, st, (const uint16_t*)k,
                     (const uint16_t*)v, lay, (void*)(parts + (w.kv_part - w.states_end)),
                     (float*)(parts + (w.z_part - w.states_end)), L, w.rows_per_split, fmap);
  launch_state_finish<Tag, D>(weight, BH, ws, parts, w, st);
}

}  // namespace sla
