// Short jobs of the backward that ride in other kernels' launches: the per-key-block lists of the map, the work items of the
// dK/dV kernel, and the sum of the heads' weight gradients.  Each is a few workgroups bound by latency; a launch of its own
// costs what it computes once more (10 + 6 + 5 us of a 207 us forward and backward of 8 heads x 4096 x 128).
#pragma once
#include "common.h"

namespace sla {

// ---- per-key-block lists ------------------------------------------------------------------
// One workgroup of COL_NW wavefronts per strip of 64 key blocks.  Every wavefront takes its own chunk of
// 64 map rows (query blocks): it reads them with coalesced 16-byte loads (a row starts at any byte) and transposes them through its
// private LDS tile; lane c counts the ones of column c in that chunk.  After a barrier every wave knows
// how many entries the chunks before its own contribute to each column and writes its matches at that
// offset, walking the chunk in row order, so list[bh][n][0..count) holds the selecting query blocks in
// ascending order.  Capacity Mblk per list (only `count` entries are ever touched).
// Bound by the latency of a round's loads.  With single bytes where rows are not multiples of 16 bytes, 2 heads of 1182 x 1182 blocks
// took 48 us, now 26 (they stand before dQ).
constexpr int COL_NW = 8;
typedef i32x4_t __attribute__((aligned(1))) i32x4_any_t;
constexpr int COL_TILE = 64 * 80;                                    // bytes of a wave's tile
constexpr int COL_LDS = COL_NW * (COL_TILE + 64 * 4);
static __device__ __forceinline__ int further_segments(int count, int seg) {      // of a list, behind its first
  return count <= seg ? 0 : (count + seg - 1) / seg - 1;
}
struct ColLists {
  const int8_t* map;
  int *list, *count, *done;                                            // done: cleared here where not null
  i32x2_t* cuts;                                                       // where not null: per strip, {segments of `seg` entries behind the
  int seg;                                                             // lists' first ones, lists that have any}
  int Mblk, Nblk, strips, wgs;                                         // wgs = strips of 64 key blocks x heads; 0: nothing to do
};
static inline ColLists col_lists_job(const int8_t* map, int* list, int* count, int* done, i32x2_t* cuts, int seg,
                                     int BH, int Mblk, int Nblk) {
  const int strips = cdiv(Nblk, 64);
  return ColLists{map, list, count, done, cuts, seg, Mblk, Nblk, strips, strips * BH};
}
// (64 * COL_NW threads; smem: COL_LDS bytes, 16-byte aligned)
static __device__ __forceinline__ void col_lists_body(const ColLists& j, int wg, char* smem) {
  int8_t (*tile)[64][80] = reinterpret_cast<int8_t (*)[64][80]>(smem);
  int (*cnt)[64] = reinterpret_cast<int (*)[64]>(smem + COL_NW * COL_TILE);
  const int Mblk = j.Mblk, Nblk = j.Nblk;
  const int bh = wg / j.strips;
  const int n0 = (wg - bh * j.strips) * 64;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int n = n0 + lane;
  const int8_t* base = j.map + (size_t)bh * Mblk * Nblk;
  int* out = j.list + ((size_t)bh * Nblk + (n < Nblk ? n : 0)) * Mblk;
  // lane -> (row lr + 16j, 16-byte chunk lc) of the tile
  const int lr = lane >> 2, lc = (lane & 3) * 16;
  int done = 0;              // entries of column `lane` written by earlier rounds
  for (int r0 = 0; r0 < Mblk; r0 += 64 * COL_NW) {
    const int m0 = r0 + 64 * wave;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int m = m0 + lr + 16 * i;
      i32x4_t x = {0, 0, 0, 0};
      if (m < Mblk) {
        // (past the row's end: the last 16 bytes of the row, moved down)
        const int over = max(n0 + lc + 16 - Nblk, 0);
        if (Nblk >= 16) {
          if (over < 16)
            x = __builtin_bit_cast(i32x4_t, __builtin_bit_cast(unsigned __int128, *reinterpret_cast<const i32x4_any_t*>(
                                                                                      base + (size_t)m * Nblk + n0 + lc - over)) >>
                                                (8 * over));
        } else {
          int8_t* b = reinterpret_cast<int8_t*>(&x);
          for (int e = 0; e < 16; ++e)
            if (n0 + lc + e < Nblk) b[e] = base[(size_t)m * Nblk + n0 + lc + e];
        }
      }
      *reinterpret_cast<i32x4_t*>(&tile[wave][lr + 16 * i][lc]) = x;
    }
    wave_lds_fence();
    int mine = 0;
#pragma unroll 16
    for (int r = 0; r < 64; ++r) mine += tile[wave][r][lane] == 1;
    cnt[wave][lane] = mine;
    __syncthreads();
    int before = 0, all = 0;
#pragma unroll
    for (int w = 0; w < COL_NW; ++w) {
      const int cw = cnt[w][lane];
      before += w < wave ? cw : 0;
      all += cw;
    }
    if (n < Nblk) {
      int c = done + before;
#pragma unroll 16
      for (int r = 0; r < 64; ++r)
        if (tile[wave][r][lane] == 1) out[c++] = m0 + r;
    }
    done += all;
    __syncthreads();         // cnt and the tiles are rewritten by the next round
  }
  if (wave == 0 && n < Nblk) {
    j.count[(size_t)bh * Nblk + n] = done;
    if (j.done) j.done[(size_t)bh * Nblk + n] = 0;
  }
  if (wave == 0 && j.cuts) {
    const int mine = n < Nblk ? further_segments(done, j.seg) : 0;
    const int lists = __builtin_popcountll(__ballot(mine > 0));
    int all = mine;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) all += __shfl_xor(all, o);
    if (lane == 0) j.cuts[wg] = i32x2_t{all, lists};
  }
}

// ---- delta = rowsum(dO * O) ------------------------------------------------------------------
// (reference kernel.py:282-286, the preprocess step.)  Three kernels form it: this job, bwd_delta_kernel, and the stream dQ kernel for its own
// rows.  All add eight columns' products with delta_sum8, then meet the neighbours at distance 1, 2, 4 (8): the same bits.

// The products of eight columns, added in order: bf16 one by one with fused multiply-adds, half precision two by two with v_dot2_f32_f16.
// Said here, because the compiler, left to itself, takes either for half precision, in one kernel not what it takes in another, and their
// sums differ in the last place.  Of the two the dot product stands nearer to 64 bits: delta of 16 heads x 6001 x 64 6.15e-8 of its norm off,
// 6.55e-8 one by one, of 12 x 9360 x 128 6.76e-8 and 7.10e-8.
template <typename Tag>
static __device__ __forceinline__ float delta_sum8(const i16x8_t& o, const i16x8_t& d_o) {
#pragma clang fp contract(off)
  float s = 0.f;
  if constexpr (__is_same(Tag, f16_tag)) {
    const f16x8_t a = __builtin_bit_cast(f16x8_t, o), b = __builtin_bit_cast(f16x8_t, d_o);
#pragma unroll
    for (int e = 0; e < 8; e += 2) s = __builtin_amdgcn_fdot2(f16x2_t{a[e], a[e + 1]}, f16x2_t{b[e], b[e + 1]}, s, false);
  } else {
    using E = Elem<Tag>;
#pragma unroll
    for (int e = 0; e < 8; ++e) s = __builtin_fmaf(E::to_float((uint16_t)o[e]), E::to_float((uint16_t)d_o[e]), s);
  }
  return s;
}

// 512 threads take four strips of 4096 / D rows, whose loads are all in flight together.
struct DeltaRows {
  const uint16_t *o, *d_o;                                             // o contiguous (B, H, L, D)
  RowLayout ldo;
  float* delta;
  int L, chunks, wgs;                                                  // chunks of a head's rows; wgs = chunks x heads; 0: nothing to do
};
constexpr int DELTA_STRIPS = 4;
static inline DeltaRows delta_rows_job(const void* o, const void* d_o, const RowLayout& ldo, float* delta, int BH, int L, int D) {
  const int chunks = cdiv(L, DELTA_STRIPS * 4096 / D);
  return DeltaRows{(const uint16_t*)o, (const uint16_t*)d_o, ldo, delta, L, chunks, chunks * BH};
}
template <typename Tag, int D>
static __device__ __forceinline__ void delta_rows_body(const DeltaRows& j, int wg) {
  constexpr int CPR = D / 8, ROWS = 512 / CPR;
  const int bh = wg / j.chunks, row0 = (wg - bh * j.chunks) * (DELTA_STRIPS * ROWS) + (int)threadIdx.x / CPR;
  const int col = ((int)threadIdx.x % CPR) * 8;
  const uint16_t* const o = j.o + (size_t)bh * j.L * D + col;
  const uint16_t* const d_o = j.d_o + j.ldo.head(bh) + col;
  i16x8_t a[DELTA_STRIPS], b[DELTA_STRIPS];
#pragma unroll
  for (int i = 0; i < DELTA_STRIPS; ++i) {
    const size_t row = min(row0 + ROWS * i, j.L - 1);
    a[i] = *reinterpret_cast<const i16x8_t*>(o + row * D);
    b[i] = *reinterpret_cast<const i16x8_t*>(d_o + row * (size_t)j.ldo.sl);
  }
#pragma unroll
  for (int i = 0; i < DELTA_STRIPS; ++i) {
    float s = delta_sum8<Tag>(a[i], b[i]);
#pragma unroll
    for (int sh = 1; sh < CPR; sh <<= 1) s += __shfl_xor(s, sh);
    const int row = row0 + ROWS * i;
    if (col == 0 && row < j.L) j.delta[(size_t)bh * j.L + row] = s;
  }
}

// ---- work items of the dK/dV kernel --------------------------------------------------------
// A key block that very many query blocks selected (an attention "sink") would make one workgroup walk a list
// many times the average length.  Lists longer than `seg` entries are therefore cut into segments of `seg`; every
// segment is one work item.  item = {bh, key block, segment, slot}: slot < 0 for a key block with a single segment
// (the workgroup writes dK / dV itself), otherwise the index of the fp32 partial this segment writes; the partials
// of a key block occupy consecutive slots and are added in segment order.
// A map whose rows hold more ones than the topk the workspace was sized for: the tables have room for every key block's first
// segment and `room` further ones, in the order of the key blocks; what exceeds that is left out, and the lists end there.  (Each
// of the room's segments belongs to at most two slots, of which there are two for each.)
// One wave per 512 (head, key block) pairs: it counts the items of all pairs before its own (no other wave is waited for),
// then numbers its own, 64 adjacent pairs at a time.  (One workgroup for all pairs, with eight adjacent ones per thread and
// therefore scattered stores, took 38 us for 32 heads x 512.)
constexpr int SEG_PAIRS = 512;
struct Segments {
  const int* count;
  int *nseg, *slot0, *done;                                            // done: segments finished so far, cleared here
  i32x4_t* items;
  int* totals;
  int nblocks, Nblk, seg, room, wgs;                                   // nblocks = heads x key blocks; wgs 0: nothing to do
};
static __device__ __forceinline__ void segments_body(const Segments& s, int wg) {
  const int lane = threadIdx.x & 63;
  const int first = wg * SEG_PAIRS;
  const auto further = [&](int c) { return further_segments(c, s.seg); };
  int extra0 = 0, slot = 0;
  for (int i = lane; i < first; i += SEG_PAIRS) {
    int c[SEG_PAIRS / 64];
#pragma unroll
    for (int x = 0; x < SEG_PAIRS / 64; ++x) c[x] = s.count[i + 64 * x];
#pragma unroll
    for (int x = 0; x < SEG_PAIRS / 64; ++x) {
      const int n = further(c[x]);
      extra0 += n;
      slot += n > 0 ? n + 1 : 0;
    }
  }
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    extra0 += __shfl_xor(extra0, o);
    slot += __shfl_xor(slot, o);
  }
  int c[SEG_PAIRS / 64];
#pragma unroll
  for (int x = 0; x < SEG_PAIRS / 64; ++x) {
    const int i = first + 64 * x + lane;
    c[x] = i < s.nblocks ? s.count[i] : 0;
  }
#pragma unroll
  for (int x = 0; x < SEG_PAIRS / 64; ++x) {
    const int i = first + 64 * x + lane;
    const int n = further(c[x]), m = n > 0 ? n + 1 : 0;
    int a = n, b = m;                          // inclusive scans
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int ta = __shfl_up(a, o), tb = __shfl_up(b, o);
      if (lane >= o) {
        a += ta;
        b += tb;
      }
    }
    if (i < s.nblocks) {
      const int e0 = min(extra0 + a - n, s.room), kept = 1 + min(extra0 + a, s.room) - e0;
      const int fi = i + e0, fs = slot + b - m;
      s.nseg[i] = kept;
      s.slot0[i] = fs;
      s.done[i] = 0;
      const int bh = i / s.Nblk, nb = i - bh * s.Nblk;
      for (int sg = 0; sg < kept; ++sg) s.items[fi + sg] = i32x4_t{bh, nb, sg, kept > 1 ? fs + sg : -1};
    }
    extra0 += __shfl(a, 63);
    slot += __shfl(b, 63);
  }
  if (first + SEG_PAIRS >= s.nblocks && lane == 0) s.totals[0] = s.nblocks + min(extra0, s.room);
}

// ---- the heads' weight gradients added up, in ascending head order ----------------------------
// dw_head [head][d][e], db_head [head][e] (fp32) -> d_weight [e][d], d_bias [e].  One wave per 256 elements.
struct HeadSums {
  const float *dw_head, *db_head;
  float *d_weight, *d_bias;
  int BH, D, wgs;                                                       // wgs = D * D / 256; 0: nothing to do
};
static __device__ __forceinline__ void head_sums_body(const HeadSums& s, int wg) {
  const int lane = threadIdx.x & 63, DD = s.D * s.D;
  const int i = wg * 256 + lane * 4;
  f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
  for (int h = 0; h < s.BH; ++h) acc += *reinterpret_cast<const f32x4_t*>(s.dw_head + (size_t)h * DD + i);
  const int d = i / s.D, e = i % s.D;
#pragma unroll
  for (int j = 0; j < 4; ++j) s.d_weight[(e + j) * s.D + d] = acc[j];
  if (wg == 0)
    for (int x = lane; x < s.D; x += 64) {
      float b = 0.f;
#pragma unroll 8
      for (int h = 0; h < s.BH; ++h) b += s.db_head[(size_t)h * s.D + x];
      s.d_bias[x] = b;
    }
}

}  // namespace sla
