// Linear branch's backward, key side, for a wave's tiles of 16 keys: dv = c dS, dc = v dS^T + dz, dk = phi'(k) dc with
// c = phi(k) (core.py:90-99 of the reference through autograd).  KeyTiles is what the attention's dK/dV kernel, which has a key
// block's gradients at hand when it ends, does for its rows.  The kernel that walks k and v for it (linear_bwd_keys_kernel in
// linear_bwd_stream.h: a tile per step, the matrices in LDS) takes only the swizzle from here and forms the same sums by steps of
// its own: which of the two runs follows from the size of the call and must not show in the bits, so a change to the arithmetic
// of one is a change to both.
#pragma once
#include "linear_common.h"

namespace sla {

// LDS tiles of 256-byte rows without padding: 16-byte piece p of row r sits at piece slot p ^ swz(r).  Row-wise
// 16-byte / 8-byte reads by 16 consecutive rows and transposing reads of 4 rows x 4 pieces both touch every bank once.
// Rows of 128 bytes (head dim 64): a line of all banks holds two of them, so the swizzle counts pairs of rows.
template <int D>
static __device__ __forceinline__ int lbs_swz(int row) {
  return D == 128 ? ((row & 3) << 2) | ((row >> 2) & 3) : ((row & 2) << 1) | ((row >> 2) & 3);
}
template <int D>
static __device__ __forceinline__ uint32_t lbs_off(int row, int col) {
  return (uint32_t)row * (2u * D) + (uint32_t)(((col >> 3) ^ lbs_swz<D>(row & 15)) << 4) + (uint32_t)(col & 7) * 2u;
}

// What the attention's dK/dV kernel needs of the linear branch: dS [head][d1][d2] and its transpose (16 bit), dz [head][D].
struct LinearKeys {
  const uint16_t *ds, *dst;
  const float* dz;
  int fmap;
};

// Key rows and value rows lie in the wave-private tiles (tile t: keys at tiles + 2 t KEY_TILE bytes, values behind them,
// swizzled); they are replaced by dv and dk.  dz: in LDS.  The matrices are read where they lie in memory, in operand order (16
// rows x 64 bytes per load), every fragment serving the products of all tiles: those of dS^T, asked for by fetch_transposed()
// long before, for dv, and each strip's registers then take the strip of dS.  (With two strips in flight the wave waits for
// each of them: 9 to 11 us per key block, now 5 to 6: the feature map 1.6, the products 1.3 and 1.1, its derivative 1.0.)
// The sums run as in linear_bwd_keys_kernel: the same bits.
template <int D>
constexpr int KEY_TILE = 16 * D * 2;             // bytes
template <typename Tag, int D, int NTILE>
struct KeyTiles {
  using E = Elem<Tag>;
  static constexpr int NT = D / 16, NC = D / 32, WT = KEY_TILE<D>;
  i16x8_t a[NT][NC];                             // rows 16 T + l of the matrix, columns 32 c + 8 h ..; l = lane % 16, h = lane / 16
  __device__ __forceinline__ void fetch(__amdgpu_buffer_rsrc_t m, int T, int lane) {
    const uint32_t off = (uint32_t)(lane & 15) * (2 * D) + 16u * (lane >> 4);
#pragma unroll
    for (int c = 0; c < NC; ++c) a[T][c] = __builtin_bit_cast(i16x8_t, __builtin_amdgcn_raw_buffer_load_b128(m, (int)(off + 64 * c), T * (32 * D), 0));
  }
  __device__ __forceinline__ void fetch_transposed(__amdgpu_buffer_rsrc_t dst, int lane) {
#pragma unroll
    for (int T = 0; T < NT; ++T) fetch(dst, T, lane);
  }
  template <int FMAP>
  __device__ __forceinline__ void run(char* tiles, __amdgpu_buffer_rsrc_t ds, const float* dz, int lane) {
    // lane = (key l of the tile's 16, quarter h): d = 16 T + 4 h + j
    const int l = lane & 15, h = lane >> 4;
    const uint32_t acc_off0 = lbs_off<D>(l, 4 * h), b_off0 = lbs_off<D>(l, 8 * h);       // pieces of a row are exclusive-ored
    const auto acc_off = [&](int T) __attribute__((always_inline)) { return acc_off0 ^ (uint32_t)(T * 32); };
    const auto b_off = [&](int c) __attribute__((always_inline)) { return b_off0 ^ (uint32_t)(c * 64); };
    i16x4_t xraw[NTILE][NT];
    float mx[NTILE], inv[NTILE];
#pragma unroll
    for (int t = 0; t < NTILE; ++t) {
      char* const tK = tiles + 2 * t * WT;
      i32x2_t apk[NT];
#pragma unroll
      for (int T = 0; T < NT; ++T) xraw[t][T] = *reinterpret_cast<const i16x4_t*>(tK + acc_off(T));
      mx[t] = 0.f;
      inv[t] = 1.f;
      phi_quarters<Tag, FMAP, NT>(xraw[t], apk, mx[t], inv[t]);
#pragma unroll
      for (int T = 0; T < NT; ++T) *reinterpret_cast<i32x2_t*>(tK + acc_off(T)) = apk[T];
    }
    wave_lds_fence();
    // dv^T = dS^T c^T
    {
      i16x8_t cf[NTILE][NC];
#pragma unroll
      for (int t = 0; t < NTILE; ++t)
#pragma unroll
        for (int c = 0; c < NC; ++c) cf[t][c] = *reinterpret_cast<const i16x8_t*>(tiles + 2 * t * WT + b_off(c));
      i32x2_t wv[NTILE][NT];
#pragma unroll
      for (int T = 0; T < NT; ++T) {
        f32x4_t acc[NTILE];
#pragma unroll
        for (int t = 0; t < NTILE; ++t) acc[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
          for (int t = 0; t < NTILE; ++t) acc[t] = E::mfma16(a[T][c], cf[t][c], acc[t]);
        fetch(ds, T, lane);
#pragma unroll
        for (int t = 0; t < NTILE; ++t) {
          wv[t][T][0] = (int)E::pack2(acc[t][0], acc[t][1]);
          wv[t][T][1] = (int)E::pack2(acc[t][2], acc[t][3]);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      // (phi(k) makes room for dv; v still stands in its own tile)
#pragma unroll
      for (int t = 0; t < NTILE; ++t)
#pragma unroll
        for (int T = 0; T < NT; ++T) *reinterpret_cast<i32x2_t*>(tiles + 2 * t * WT + acc_off(T)) = wv[t][T];
    }
    // dc^T = dS v^T + dz ; dk = phi'(k) dc
    i16x8_t vf[NTILE][NC];
    f32x4_t dca[NTILE][NT];
#pragma unroll
    for (int t = 0; t < NTILE; ++t)
#pragma unroll
      for (int c = 0; c < NC; ++c) vf[t][c] = *reinterpret_cast<const i16x8_t*>(tiles + (2 * t + 1) * WT + b_off(c));
    wave_lds_fence();
#pragma unroll
    for (int T = 0; T < NT; ++T) {
#pragma unroll
      for (int t = 0; t < NTILE; ++t) dca[t][T] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int t = 0; t < NTILE; ++t) dca[t][T] = E::mfma16(a[T][c], vf[t][c], dca[t][T]);
    }
#pragma unroll
    for (int t = 0; t < NTILE; ++t) {
#pragma unroll
      for (int T = 0; T < NT; ++T) {
        const f32x4_t zz = *reinterpret_cast<const f32x4_t*>(dz + 16 * T + 4 * h);
#pragma unroll
        for (int j = 0; j < 4; ++j) dca[t][T][j] += zz[j];
      }
      phi_quarters_backward<Tag, FMAP, NT>(xraw[t], mx[t], inv[t], dca[t]);
#pragma unroll
      for (int T = 0; T < NT; ++T) {
        i32x2_t wk;
        wk[0] = (int)E::pack2(dca[t][T][0], dca[t][T][1]);
        wk[1] = (int)E::pack2(dca[t][T][2], dca[t][T][3]);
        *reinterpret_cast<i32x2_t*>(tiles + (2 * t + 1) * WT + acc_off(T)) = wk;
      }
    }
    wave_lds_fence();
  }
};

}  // namespace sla
