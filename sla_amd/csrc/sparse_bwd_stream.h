// dK / dV of the block-sparse attention backward for 64-row query blocks: one workgroup of two waves per key block (or
// per segment of a key block's list), one wave per SIMD at head dim 128, two at head dim 64 (where everything a wave
// keeps is half as large).
//
// Stands in for _attn_bwd_dkdv of the reference (sparse_linear_attention/kernel.py:160-237) like bwd_dkdv_kernel,
// whose work items, lists and arithmetic it shares.  What differs:
//   * a wave owns 32 keys and the whole head dimension: K^T and V^T fragments (B operands of S = Q K^T and
//     dP = dO V^T) and the dK^T / dV^T accumulators (D x 32 keys each) stay in its registers, P and dS leave
//     the accumulators in the B-operand layout of dV^T += dO^T P and dK^T += Q^T dS.  Nothing is handed from wave
//     to wave, and there is one barrier per 32 query rows;
//   * Q and dO rows go from memory straight into LDS (buffer loads with the LDS bit), 32 rows at a time, into a
//     ring of four generations; a generation is requested two units of 32 rows before it is first read.  The
//     16-byte pieces of a row are XOR-swizzled so that both the row-wise reads (A operands of S and dP) and the
//     transposing reads (A operands of the second products) are free of bank conflicts;
//   * the loop is rotated: the exponentials and the rest of the vector arithmetic of unit u run beside the first
//     products of unit u + 1, then come the second products of unit u;
//   * a lone wave issues one instruction per four cycles at best, so instructions are what is saved: V^T is kept
//     negated and the accumulators of -dP start from delta (no subtraction per element; dK comes out negated and is
//     turned at the end), four requests share one M0, LDS offsets are instruction immediates: 225 instructions per
//     unit of 32 products (1024 cycles of the matrix pipe) where 300 were needed without all that.  The barrier stands
//     where the fragments of a unit have all been read, so that the first reads of the next unit and the requests for
//     the unit after next run beside products.  Measured, before and after: B1 H12 L32760 with 25 key blocks per row
//     840 -> 758 us (matrix pipe busy 44 -> 52 % of the cycles, at 1.7 to 1.9 GHz, where the power limit holds it), B2 H16
//     L32760 with 128-row query blocks 2272 -> 2065 us, B2 H4 L4096 48.5 -> 43.0 us.  Head dim 64 against
//     bwd_dkdv_kernel: B2 H8 L6001 with 9 key blocks per row 57.6 -> 44.2 us.
#pragma once
#include <type_traits>

#include "linear_keys.h"

namespace sla {

template <int N>
using I = std::integral_constant<int, N>;

// One of four requests of 16 bytes per lane, memory -> LDS (lane l's piece lands 16 l bytes on), REQ_PITCH bytes apart in
// LDS.  The instruction offset counts for both addresses: off is the memory offset less J * REQ_PITCH (never negative:
// REQ_SLACK bytes are part of it and of a descriptor that starts as many bytes early).  The first of a group sets M0.
// (Between a scalar write of M0 and a memory -> LDS load that reads it the hardware wants one wait state; the compiler
// adds it to its own code and does not look into these instructions.)
constexpr int REQ_PITCH = 1040;                // 4 rows of 256 bytes (8 of 128) + 16 bytes of padding
constexpr int REQ_SLACK = 64;
template <int J, bool SET = J == 0>
static __device__ __forceinline__ void lds_dma_row4(__amdgpu_buffer_rsrc_t rsrc, uint32_t off, uint32_t lds) {
  if constexpr (SET)
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen offset:%3 lds" ::"s"(lds), "v"(off), "s"(rsrc),
                 "n"(J * REQ_PITCH)
                 : "memory");
  else
    asm volatile("buffer_load_dwordx4 %0, %1, 0 offen offset:%2 lds" ::"v"(off), "s"(rsrc), "n"(J * REQ_PITCH) : "memory");
}
// Where the 16-byte pieces of 32 rows lie: request j holds rows RPR j .., piece p of a row in slot p ^ swz(row).  For one piece
// the 16 rows of a row-wise read hit 16 different slots of the 256 bytes LDS serves at a time, and so do the 4 rows x 4 pieces
// of a transposing read.  (256-byte rows: row % 4 picks the group of four slots, the padding of a request the slot in it.
// 128-byte rows: row % 2 and row / 2 % 2 pick the group, row / 4 % 2 a pair in it and the padding the slot of the pair.)
template <int D>
struct BwdTile {
  static constexpr int ROWB = D * 2, RPR = 1024 / ROWB, NREQ = 32 / RPR, BYTES = NREQ * REQ_PITCH;
  static __device__ __forceinline__ int swz(int row) { return D == 128 ? 4 * (row & 3) : 4 * ((row >> 1) & 1) + 2 * ((row >> 2) & 1); }
  static __device__ __forceinline__ int piece_at(int row, int piece) {        // byte offset inside the tile
    return row * ROWB + row / RPR * 16 + (piece ^ swz(row)) * 16;
  }
};
// 4 bytes per lane: lane l's word lands at lds_base + lds_off + 4 l
static __device__ __forceinline__ void lds_dma_b32(__amdgpu_buffer_rsrc_t rsrc, uint32_t byte_off, uint32_t lds_base,
                                                   uint32_t lds_off) {
  asm volatile("s_add_u32 m0, %0, %3\n\ts_nop 0\n\tbuffer_load_dword %1, %2, 0 offen lds" ::"s"(lds_base), "v"(byte_off), "s"(rsrc),
               "s"(lds_off)
               : "memory", "scc");
}

constexpr int DKDV_STREAM_MAX_SEG = 1024;      // list entries one work item may have (they are copied into LDS)

template <int D>
constexpr int DKDV_LDS = 4 * (2 * BwdTile<D>::BYTES + 512);    // four generations: Q rows, dO rows, log-sum-exps, deltas (32 of 64 words used)

// One work item: key block `nb` of head `bh`, entries sg * seg .. of its list; slot: where its partial sums go, if the list is cut
// (into `ns` segments), or < 0.  smem: DKDV_LDS bytes, entries: DKDV_STREAM_MAX_SEG words of LDS.
template <typename Tag, int D, bool LINEAR>
static __device__ __forceinline__ void dkdv_stream_body(
    const uint16_t* q, const uint16_t* k, const uint16_t* v,
    const uint16_t* d_o, const float* lse, const float* delta,
    const int* list, const int* count, float* part, int seg, uint16_t* dk,
    uint16_t* dv, const RowLayout lin, const RowLayout ldo, int L, int Mblk, int Nblk, float qk_scale, int wide,
    int add, int* done, const LinearKeys& keys, uint8_t* const smem, int* const entries, const int bh, const int nb,
    const int sg, const int slot, const int ns) {
  // (wide = 1: the lists name 128-row query blocks; an entry is then walked as its two 64-row halves.  add: the gradients are
  //  added, rounded, to what dk and dv hold.  LINEAR: to the linear branch's gradients of the same rows, which are formed here,
  //  in 16 bit: the same sums)
  using E = Elem<Tag>;
  using T32 = BwdTile<D>;
  constexpr int DC = D / 16, DT = D / 32;
  constexpr int TILE = T32::BYTES;          // 32 rows of Q or of dO
  constexpr int GEN = 2 * TILE + 512;       // one generation: Q rows, dO rows, log-sum-exps, deltas (32 of 64 words used)
  constexpr int NG = 4;
  constexpr int NR = T32::NREQ / 2;         // requests per wave (16 rows) and tile
  constexpr int NREQ = 2 * NR + 1;          // requests per wave and unit: Q, dO, 1 x lse or delta
  constexpr int NGRP = 2 * DT;              // groups (16 query rows x 32 d) of two second products
  constexpr int ROWS8 = 8 / T32::RPR * REQ_PITCH;              // 8 rows further on in a tile
  static_assert(NG * GEN == DKDV_LDS<D>, "the generations");
  // (`entries`: this work item's list entries.  Read from memory inside the loop they would be vector loads - the inline assembly
  // keeps the compiler from using the scalar path - and waiting for a vector load means waiting for every memory ->
  // LDS request issued before it.)
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);         // keys 32w .. 32w+31 of the block
  const int g = lane >> 5, r = lane & 31;
  const float c_log2e = qk_scale * 1.4426950408889634f;

  const size_t head_off = first_lane64(lin.head(bh)), head_do = first_lane64(ldo.head(bh));
  const uint32_t pitch = (uint32_t)lin.sl, pitch_do = (uint32_t)ldo.sl;
  const __amdgpu_buffer_rsrc_t qh = make_rsrc(q + head_off - REQ_SLACK / 2, lin.head_range_bytes(L, D) + REQ_SLACK);
  const __amdgpu_buffer_rsrc_t doh = make_rsrc(d_o + head_do - REQ_SLACK / 2, ldo.head_range_bytes(L, D) + REQ_SLACK);
  const __amdgpu_buffer_rsrc_t kb = make_rsrc(k + head_off, lin.head_range_bytes(L, D));
  const __amdgpu_buffer_rsrc_t vb = make_rsrc(v + head_off, lin.head_range_bytes(L, D));
  // wave 0 fetches the log-sum-exps of a unit, wave 1 its deltas
  const __amdgpu_buffer_rsrc_t ldh = make_rsrc((w ? delta : lse) + (size_t)bh * L, (uint32_t)L * 4);

  // The length of this key block's list and the first 128 entries of this work item's part of it are asked for before
  // the fragments below (loads come back in the order they were issued, and the first requests for Q and dO hang on
  // the entries); entries past the end of the list are read from inside its row of Mblk words and never used.
  const int* mylist = list + ((size_t)bh * Nblk + nb) * Mblk;
  const int e0 = sg * seg;
  const int count_lane = count[(size_t)bh * Nblk + nb];
  const int first_entry = mylist[min(e0 + (tid >> wide), Mblk - 1)];
  // K^T and -V^T fragments (B operands): this lane's key column, 8 adjacent d per chunk; parked in accumulation registers
  const int krow = nb * 64 + w * 32 + r;
  const bool kok = krow < L;
  i16x8_t kf[DC], vf[DC];
#pragma unroll
  for (int c = 0; c < DC; ++c) {
    kf[c] = buf_load_b128(kb, ((uint32_t)krow * pitch + 16 * c + 8 * g) * 2);     // rows past L read as zero
    vf[c] = buf_load_b128(vb, ((uint32_t)krow * pitch + 16 * c + 8 * g) * 2);
  }
  // Rows past L are never written into LDS (they lie outside the buffers), and what LDS holds in their place must
  // be finite: their probabilities are exactly 0 (log-sum-exp +inf), and 0 times a finite number adds nothing.
#pragma unroll
  for (int i = 0; i < (NG * GEN / 16 + 127) / 128; ++i)
    if (i * 128 + tid < NG * GEN / 16) reinterpret_cast<i32x4_t*>(smem)[i * 128 + tid] = i32x4_t{0, 0, 0, 0};

  // what the gradients are added to, asked for before the last unit's arithmetic: what dk and dv hold; LINEAR: rows of k and
  // v as they are, and what becomes of them
  const int krow0 = nb * 64 + w * 32;
  TileRows<D> rows[2];
  KeyTiles<Tag, D, 2> key_work;
  const __amdgpu_buffer_rsrc_t ds_rs = make_rsrc(keys.ds + (size_t)bh * (D * D), 2 * D * D),
                               dst_rs = make_rsrc(keys.dst + (size_t)bh * (D * D), 2 * D * D);
  float dz_lane[D / 64];
  const auto fetch_rows = [&]() __attribute__((always_inline)) {
    if constexpr (!LINEAR) {
      if (!add) return;
      rows[0].fetch(dk + head_off + (size_t)krow0 * pitch, L - krow0, lane, pitch);
      rows[1].fetch(dv + head_off + (size_t)krow0 * pitch, L - krow0, lane, pitch);
      return;
    }
#pragma unroll
    for (int i = 0; i < TileRows<D>::N; ++i) {                   // (rows past L read as zero)
      const uint32_t at = (uint32_t)(krow0 + lane / (D / 8) + 512 / D * i) * (pitch * 2) + (uint32_t)(lane % (D / 8)) * 16;
      rows[0].x[i] = buf_load_b128(kb, at);
      rows[1].x[i] = buf_load_b128(vb, at);
    }
#pragma unroll
    for (int i = 0; i < D / 64; ++i) dz_lane[i] = keys.dz[(size_t)bh * D + 64 * i + lane];
    key_work.fetch_transposed(dst_rs, lane);
  };
  char* const key_tiles = reinterpret_cast<char*>(smem) + w * (4 * KEY_TILE<D>);         // (over the generations)
  // piece i of a lane: where TileRows has it; which: 0 k, then dv, 1 v, then dk
  const auto key_piece = [&](int which, int i) __attribute__((always_inline)) {
    const int row = lane / (D / 8) + 512 / D * i;
    return key_tiles + (2 * (row >> 4) + which) * KEY_TILE<D> + lbs_off<D>(row & 15, 8 * (lane % (D / 8)));
  };
  const auto linear_gradients = [&]() __attribute__((always_inline)) {
    int lane = threadIdx.x & 63;
    asm volatile("" : "+v"(lane));               // (nothing of this is worth keeping through the loop)
#pragma unroll
    for (int which = 0; which < 2; ++which)
#pragma unroll
      for (int i = 0; i < TileRows<D>::N; ++i) *reinterpret_cast<i16x8_t*>(key_piece(which, i)) = rows[which].x[i];
    float* const dz = reinterpret_cast<float*>(smem + 8 * KEY_TILE<D> + 4 * 32 * TileRows<D>::SSTR * 2) + w * D;
#pragma unroll
    for (int i = 0; i < D / 64; ++i) dz[64 * i + lane] = dz_lane[i];
    wave_lds_fence();
    if (keys.fmap == SLA_FMAP_ELU) key_work.template run<SLA_FMAP_ELU>(key_tiles, ds_rs, dz, lane);
    else if (keys.fmap == SLA_FMAP_RELU) key_work.template run<SLA_FMAP_RELU>(key_tiles, ds_rs, dz, lane);
    else key_work.template run<SLA_FMAP_SOFTMAX>(key_tiles, ds_rs, dz, lane);
  };
  static_assert(8 * KEY_TILE<D> + 4 * 32 * TileRows<D>::SSTR * 2 + 2 * D * 4 <= NG * GEN, "tiles, staging rows and dz fit the generations");

  f32x16_t dkacc[DT], dvacc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      dkacc[dt][i] = 0.f;
      dvacc[dt][i] = 0.f;
    }

  // this work item's part of the list, in units of 32 query rows (two per listed query block)
  const int e1 = min(__builtin_amdgcn_readfirstlane(count_lane), (sg + 1) * seg);
  const int nent = (e1 - e0) << wide;               // 64-row blocks this work item walks
  const int row_none = (L + 63) & ~63;              // past every head: such requests touch neither memory nor LDS
  auto entry_row0 = [&](int e) __attribute__((always_inline)) -> int {
    const int row0 = __builtin_amdgcn_readfirstlane(entries[min(e, nent - 1)]) * 64;
    return e < nent ? row0 : row_none;
  };
  if (tid < (seg << wide)) entries[tid] = (first_entry << wide) + (tid & wide);
  for (int i = 128 + tid; i < nent; i += 128) entries[i] = (mylist[e0 + (i >> wide)] << wide) + (i & wide);

  // ---- addressing ----
  // A request moves RPR rows (64 lanes x 16 bytes): lane -> row RPR j + lane / (D / 8) of this wave's 16 rows, 16-byte slot
  // lane % (D / 8), which receives piece (slot ^ swz(row)) of that row.
  const uint32_t smem_addr = (uint32_t)(size_t)smem;
  const int lrow = lane / (D / 8), lslot = lane % (D / 8);
  uint32_t qoff[NR], dooff[NR];
#pragma unroll
  for (int j = 0; j < NR; ++j) {
    const uint32_t row = 16 * w + T32::RPR * j + lrow;         // row of the unit
    const uint32_t piece = (uint32_t)(lslot ^ T32::swz(lrow)) * 16 + REQ_SLACK - j * REQ_PITCH;
    qoff[j] = row * pitch * 2 + piece;
    dooff[j] = row * pitch_do * 2 + piece;
  }
  // LDS addresses of this wave's 16 rows inside a tile and of its words (log-sum-exps or deltas) behind the tiles
  const uint32_t rows_base = __builtin_amdgcn_readfirstlane(smem_addr + (uint32_t)(NR * w) * REQ_PITCH);
  const uint32_t ld_base = __builtin_amdgcn_readfirstlane(smem_addr + (uint32_t)w * 256);
  const uint32_t lane4 = (uint32_t)lane * 4;
#define SLA_DKDV_REQUEST_Q(J, ROW0, GENERATION) \
  lds_dma_row4<J>(qh, qoff[J] + (uint32_t)(ROW0) * (pitch * 2), rows_base + (uint32_t)(GENERATION) * GEN)
#define SLA_DKDV_REQUEST_DO(J, ROW0, GENERATION) \
  lds_dma_row4<J>(doh, dooff[J] + (uint32_t)(ROW0) * (pitch_do * 2), rows_base + (uint32_t)(GENERATION) * GEN + TILE)
#define SLA_DKDV_REQUEST_LD(ROW0, GENERATION) \
  lds_dma_b32(ldh, lane4 + (uint32_t)(ROW0) * 4, ld_base, (uint32_t)(GENERATION) * GEN + 2 * TILE)
  // fragments: row-wise, row r, piece 2c + g: four bases; transposed (16 query rows x 32 d), rows 16 c2 + 4 g +
  // (lane % 16) / 4 and 8 further on, 8 bytes at element 4 (lane % 4) of the 16-column strip 2 dt + (lane / 16) % 2: one
  // base per dt
  const uint8_t* rfp[4];
  const uint8_t* tfp[DT];
  const uint8_t* const ldp = smem + 2 * TILE + 16 * g;       // log-sum-exps of rows 4g .. 4g + 3; deltas 256 bytes on
  const int tr_row = 4 * g + ((lane & 15) >> 2);
#pragma unroll
  for (int i = 0; i < 4; ++i) rfp[i] = smem + T32::piece_at(r, 2 * (i * DC / 4) + g);
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
    tfp[dt] = smem + T32::piece_at(tr_row, 4 * dt + 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1)) + (lane & 1) * 8;
  constexpr int TRS = D == 128 ? 5 : 4;
  i16x8_t af[3], bf[3];              // row-wise Q and dO fragments, two chunks ahead
  i16x8_t trd[TRS], trq[TRS];        // transposed dO / Q fragments of group grp in slot grp % TRS, four groups ahead
  f32x4_t l4[4];                     // log-sum-exps of the unit whose elements come next: accumulator register
                                     // 4 i4 + j of S / dP is query row 8 i4 + 4 g + j of the unit, this lane's column its key
  auto row_frags = [&](int at, int c) __attribute__((always_inline)) {
    const uint8_t* p = rfp[c * 4 / DC] + at + (D == 128 ? (c & 1) * 32 : 0);
    af[c % 3] = *reinterpret_cast<const i16x8_t*>(p);
    bf[c % 3] = *reinterpret_cast<const i16x8_t*>(p + TILE);
  };
  auto tr_frags = [&](int at, int grp) __attribute__((always_inline)) {
    const uint8_t* t0 = tfp[grp % DT] + at + grp / DT * 2 * ROWS8;
    trd[grp % TRS] = concat4(lds_read_tr16(reinterpret_cast<const uint16_t*>(t0 + TILE)),
                             lds_read_tr16(reinterpret_cast<const uint16_t*>(t0 + TILE + ROWS8)));
    trq[grp % TRS] = concat4(lds_read_tr16(reinterpret_cast<const uint16_t*>(t0)),
                             lds_read_tr16(reinterpret_cast<const uint16_t*>(t0 + ROWS8)));
  };
  auto read_lse = [&](int at, int i4) __attribute__((always_inline)) {
    l4[i4] = *reinterpret_cast<const f32x4_t*>(ldp + at + i4 * 32);
  };
  auto read_delta = [&](int at, f32x16_t& dp, int i4) __attribute__((always_inline)) {      // what the chain of -dP starts from
    const f32x4_t d4 = *reinterpret_cast<const f32x4_t*>(ldp + at + 256 + i4 * 32);
#pragma unroll
    for (int j = 0; j < 4; ++j) dp[4 * i4 + j] = d4[j];
  };
  // product 2 c + {0, 1} of the first sixteen: S, -dP + delta, chunk c of the head dimension
  auto score_product = [&](f32x16_t& s, f32x16_t& dp, int c, int which) __attribute__((always_inline)) {
    if (which) mfma_scores<Tag>(dp, bf[c % 3], vf[c]);
    else if (c == 0) mfma_scores_first<Tag>(s, af[0], kf[0]);
    else mfma_scores<Tag>(s, af[c % 3], kf[c]);
  };
  i32x4_t pw[2], dw[2];
  // element i of a unit: P = exp2(S c - lse), then -dS = P (delta - dP); packed in pairs
  auto prob = [&](f32x16_t& s, int i) __attribute__((always_inline)) {
    float p = fast_exp2(__builtin_fmaf(s[i], c_log2e, -l4[i >> 2][i & 3]));
    asm volatile("" : "+v"(p));
    s[i] = p;
  };
  auto grad = [&](f32x16_t& s, f32x16_t& dp, int i) __attribute__((always_inline)) {
    float ds = s[i] * dp[i];
    asm volatile("" : "+v"(ds));
    dp[i] = ds;
    if (i & 1) {
      uint32_t a = E::pack2(s[i - 1], s[i]), b = E::pack2(dp[i - 1], dp[i]);
      asm volatile("" : "+v"(a), "+v"(b));
      pw[i >> 3][(i >> 1) & 3] = (int)a;
      dw[i >> 3][(i >> 1) & 3] = (int)b;
    }
  };
  auto second_products = [&](int grp) __attribute__((always_inline)) {
    const int c2 = grp / DT, dt = grp % DT;
    dvacc[dt] = E::mfma32(trd[grp % TRS], __builtin_bit_cast(i16x8_t, pw[c2]), dvacc[dt]);
    dkacc[dt] = E::mfma32(trq[grp % TRS], __builtin_bit_cast(i16x8_t, dw[c2]), dkacc[dt]);
  };
  auto mask_rows = [&](int row0) __attribute__((always_inline)) {      // rows past L: +inf makes every probability exactly 0
#pragma unroll
    for (int i4 = 0; i4 < 4; ++i4)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (row0 + 8 * i4 + 4 * g + j >= L) l4[i4][j] = INFINITY;
  };

  // One iteration = unit u in generation GU = u % 4, D / 4 products:
  //   first half   S and dP of unit u + 1 (two chains)        beside: P and dS of unit u, the transposed fragments of its first
  //                                                            four groups, the requests for dO and scalars of unit u + 3
  //   second half  dV^T += dO^T P, dK^T += Q^T dS of unit u   beside: the other transposed fragments; then, from the barrier on,
  //                                                            the requests for Q of unit u + 4 (into unit u's generation) and
  //                                                            what the next iteration wants first from LDS
  // The barrier stands where this wave has read all of unit u's generation and its part of unit u + 2 has landed (only
  // the requests for unit u + 3 may be out): behind it everyone's has, and the generation may be overwritten.
  // At head dim 64 a unit has half the products for the same vector arithmetic: two elements per product, the last four
  // beside the first second products, which need the first eight only.
  // (A key row past L only ever feeds its own, never stored, column of dK^T / dV^T: no masking needed.)
  f32x16_t s_a, dp_a, s_b, dp_b;
  auto iteration = [&](auto gu, f32x16_t& s_cur, f32x16_t& dp_cur, f32x16_t& s_nxt, f32x16_t& dp_nxt, int row0_u, int row0_u3,
                       int row0_u4) __attribute__((always_inline)) {
    constexpr int EA = D == 128 ? 16 : 12;                     // elements beside the first half
    constexpr int GU = decltype(gu)::value, AT0 = GU * GEN, AT1 = ((GU + 1) & 3) * GEN, AT2 = ((GU + 2) & 3) * GEN;
    if (__builtin_expect(row0_u + 32 > L, 0)) mask_rows(row0_u);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < DC; ++c) {
#pragma unroll
      for (int which = 0; which < 2; ++which) {
        const int sl = 2 * c + which;
        score_product(s_nxt, dp_nxt, c, which);
#pragma unroll
        for (int i = sl * EA / (2 * DC); i < (sl + 1) * EA / (2 * DC); ++i) {
          prob(s_cur, i);
          if (i > 0) grad(s_cur, dp_cur, i - 1);
        }
        if (which == 0 && c + 2 < DC) row_frags(AT1, c + 2);
        if (sl == 1) SLA_DKDV_REQUEST_DO(0, row0_u3, (GU + 3) & 3);
        if (sl == 2) SLA_DKDV_REQUEST_DO(1, row0_u3, (GU + 3) & 3);
        if constexpr (NR == 4) {
          if (sl == 3) SLA_DKDV_REQUEST_DO(NR - 2, row0_u3, (GU + 3) & 3);
          if (sl == 4) SLA_DKDV_REQUEST_DO(NR - 1, row0_u3, (GU + 3) & 3);
        }
        if (sl == NR + 1) SLA_DKDV_REQUEST_LD(row0_u3, (GU + 3) & 3);
        if (D == 128 ? (sl >= 9 && (sl & 1)) : sl >= 4) tr_frags(AT0, D == 128 ? (sl - 9) >> 1 : sl - 4);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if (EA == 16) grad(s_cur, dp_cur, 15);
#pragma unroll
    for (int grp = 0; grp < NGRP; ++grp) {
      constexpr int BAR = D == 128 ? 5 : 2;                    // the group before which the barrier stands
      if (grp + 4 < NGRP) tr_frags(AT0, grp + 4);
      if (grp == BAR) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(NREQ) : "memory");
      if (EA < 16 && grp == DT) grad(s_cur, dp_cur, 15);
      second_products(grp);
      if (EA < 16 && grp < DT) {
        constexpr int PER = (16 - EA) / DT;
#pragma unroll
        for (int i = EA + grp * PER; i < EA + (grp + 1) * PER; ++i) {
          prob(s_cur, i);
          grad(s_cur, dp_cur, i - 1);
        }
      }
      if (grp == BAR) {
        SLA_DKDV_REQUEST_Q(0, row0_u4, GU);
        row_frags(AT2, 0);
      }
      if (grp == BAR + 1) {
        SLA_DKDV_REQUEST_Q(1, row0_u4, GU);
#pragma unroll
        for (int i4 = 0; i4 < 4; ++i4) read_delta(AT2, dp_cur, i4);
      }
      if (grp == NGRP - 1) {
        if constexpr (NR == 4) {
          SLA_DKDV_REQUEST_Q(NR - 2, row0_u4, GU);
          SLA_DKDV_REQUEST_Q(NR - 1, row0_u4, GU);
        }
        row_frags(AT2, 1);
      }
      if (D == 128 ? grp >= 3 && grp < 7 : grp >= 2) {
        read_lse(AT1, D == 128 ? grp - 3 : 2 * grp - 4);
        if (D == 64) read_lse(AT1, 2 * grp - 3);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  __syncthreads();                                             // the zeros and the entries are in place before anything is requested
  const auto request_q = [&](int row0, int gen) __attribute__((always_inline)) {
    SLA_DKDV_REQUEST_Q(0, row0, gen);
    SLA_DKDV_REQUEST_Q(1, row0, gen);
    if constexpr (NR == 4) {
      SLA_DKDV_REQUEST_Q(NR - 2, row0, gen);
      SLA_DKDV_REQUEST_Q(NR - 1, row0, gen);
    }
  };
  const auto request_unit = [&](int row0, int gen) __attribute__((always_inline)) {
    request_q(row0, gen);
    SLA_DKDV_REQUEST_DO(0, row0, gen);
    SLA_DKDV_REQUEST_DO(1, row0, gen);
    if constexpr (NR == 4) {
      SLA_DKDV_REQUEST_DO(NR - 2, row0, gen);
      SLA_DKDV_REQUEST_DO(NR - 1, row0, gen);
    }
    SLA_DKDV_REQUEST_LD(row0, gen);
  };
  // first query rows of the listed blocks: E0 = of the entry of units u and u + 1, E1 = of the next one, E2 = of the one after
  int E0 = 0, E1 = 0, E2 = 0;
  if (nent > 0) {
    E0 = entry_row0(0);
    E1 = entry_row0(1);
    E2 = entry_row0(2);
    request_unit(E0, 0);
    request_unit(E0 + 32, 1);
    request_unit(E1, 2);
  }
  // (the wait for the K^T and V^T fragments comes here, behind the first requests, which only needed the list)
#pragma unroll
  for (int c = 0; c < DC; ++c) {
    vf[c] ^= (short)0x8000;                                    // -V
    asm volatile("" : "+a"(kf[c]), "+a"(vf[c]));
  }
  if (nent > 0) {
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(2 * NREQ) : "memory");
    row_frags(0, 0);
    row_frags(0, 1);
#pragma unroll
    for (int i4 = 0; i4 < 4; ++i4) {
      read_delta(0, dp_a, i4);
      read_lse(0, i4);
    }
#pragma unroll
    for (int c = 0; c < DC; ++c) {
      score_product(s_a, dp_a, c, 0);
      score_product(s_a, dp_a, c, 1);
      if (c + 2 < DC) row_frags(0, c + 2);
    }
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");         // (the vector ALU reads these results next)
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(NREQ) : "memory");
    request_q(E1 + 32, 3);
    row_frags(GEN, 0);
    row_frags(GEN, 1);
#pragma unroll
    for (int i4 = 0; i4 < 4; ++i4) read_delta(GEN, dp_b, i4);
    int last_at;                                               // where the last unit lies (an odd one: generation 1 or 3)
    for (int b = 0;; b += 2) {
      int E3 = entry_row0(b + 3);                              // (looked up now, used two units from now)
      iteration(I<0>{}, s_a, dp_a, s_b, dp_b, E0, E1 + 32, E2);
      last_at = GEN;
      if (b + 1 >= nent) break;
      iteration(I<1>{}, s_b, dp_b, s_a, dp_a, E0 + 32, E2, E2 + 32);
      E0 = E1;
      E1 = E2;
      E2 = E3;
      E3 = entry_row0(b + 4);
      iteration(I<2>{}, s_a, dp_a, s_b, dp_b, E0, E1 + 32, E2);
      last_at = 3 * GEN;
      if (b + 2 >= nent) break;
      iteration(I<3>{}, s_b, dp_b, s_a, dp_a, E0 + 32, E2, E2 + 32);
      E0 = E1;
      E1 = E2;
      E2 = E3;
    }
    // the last unit: no scores left to form beside its arithmetic
    if (slot < 0) fetch_rows();
    if (__builtin_expect(E0 + 64 > L, 0)) mask_rows(E0 + 32);
#pragma unroll
    for (int grp = 0; grp < 4; ++grp) tr_frags(last_at, grp);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      prob(s_b, i);
      grad(s_b, dp_b, i);
    }
#pragma unroll
    for (int grp = 0; grp < NGRP; ++grp) {
      if (grp + 4 < NGRP) tr_frags(last_at, grp + 4);
      second_products(grp);
    }
  }
  if (slot < 0 && nent <= 0) fetch_rows();
#undef SLA_DKDV_REQUEST_Q
#undef SLA_DKDV_REQUEST_DO
#undef SLA_DKDV_REQUEST_LD
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");    // (nothing of this workgroup is in flight when it ends)

  const auto turned = [&](float x) __attribute__((always_inline)) { return __builtin_fmaf(x, -qk_scale, 0.f); };   // (+0 for an empty sum)
  // [dk | dv][wave][32 rows]
  uint16_t* const stage = reinterpret_cast<uint16_t*>(smem + (LINEAR ? 8 * KEY_TILE<D> : 0)) + w * (32 * TileRows<D>::SSTR);
  if (slot >= 0) {
    // One segment of a long list: fp32 partial [dk | dv][64][D].  The workgroup that finishes a key block's last segment adds
    // all of them up, in segment order: its count is raised only when a workgroup's whole partial is visible to the others.
    // (One thread releases, behind the barrier, for both waves, and only the last workgroup of a key block acquires: a release
    // writes an XCD's modified lines back.  With both fences in every thread of every segment, and the sums four values of a thread
    // at a time, this kernel took 437 us at 2 heads x 75600 x 64 and 718 at 2 x 75600 x 128, now 372 and 658; with the sums in a
    // launch of their own 356 + 14 and 612 + 24, and 4 to 5 us more where no list is cut.)
    float* pk = part + (size_t)slot * (2 * 64 * D) + (size_t)(w * 32 + r) * D;
    float* pv = pk + 64 * D;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int i4 = 0; i4 < 4; ++i4) {
        const int d0 = 32 * dt + 8 * i4 + 4 * g;
        *reinterpret_cast<f32x4_t*>(pk + d0) = f32x4_t{turned(dkacc[dt][4 * i4 + 0]), turned(dkacc[dt][4 * i4 + 1]),
                                                       turned(dkacc[dt][4 * i4 + 2]), turned(dkacc[dt][4 * i4 + 3])};
        *reinterpret_cast<f32x4_t*>(pv + d0) =
            f32x4_t{dvacc[dt][4 * i4 + 0], dvacc[dt][4 * i4 + 1], dvacc[dt][4 * i4 + 2], dvacc[dt][4 * i4 + 3]};
      }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // (the barrier alone does not wait for a wave's stores)
    __syncthreads();
    if (tid == 0) {
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
      entries[0] = atomicAdd(&done[(size_t)bh * Nblk + nb], 1);
    }
    __syncthreads();
    if (__builtin_amdgcn_readfirstlane(entries[0]) != ns - 1) return;
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    if (LINEAR) fetch_rows();
  } else {
    // The rounded rows go through LDS (both waves are done with the generations) and leave as whole rows in streaming
    // stores: they are not read again here, and what does not stay behind as modified lines in L2 need not be written
    // back when the kernel ends.
    __syncthreads();
#pragma unroll
    for (int which = 0; which < 2; ++which)
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int i4 = 0; i4 < 4; ++i4) {
          i32x2_t wv;
          if (which == 0) {
            wv[0] = (int)E::pack2(turned(dkacc[dt][4 * i4 + 0]), turned(dkacc[dt][4 * i4 + 1]));
            wv[1] = (int)E::pack2(turned(dkacc[dt][4 * i4 + 2]), turned(dkacc[dt][4 * i4 + 3]));
          } else {
            wv[0] = (int)E::pack2(dvacc[dt][4 * i4 + 0], dvacc[dt][4 * i4 + 1]);
            wv[1] = (int)E::pack2(dvacc[dt][4 * i4 + 2], dvacc[dt][4 * i4 + 3]);
          }
          *reinterpret_cast<i32x2_t*>(&stage[which * (64 * TileRows<D>::SSTR) + r * TileRows<D>::SSTR + 32 * dt + 8 * i4 + 4 * g]) = wv;
        }
    wave_lds_fence();
  }
  if constexpr (LINEAR) linear_gradients();
  if (slot >= 0) {
    if (LINEAR) __syncthreads();
    const float* p0 = part + (size_t)(slot - sg) * (2 * 64 * D);
    // (all of a thread's loads of a segment's dK or dV in flight at once)
    constexpr int NV = 64 * D / 4 / 128;
#pragma unroll
    for (int which = 0; which < 2; ++which) {
      f32x4_t acc[NV];
#pragma unroll
      for (int i = 0; i < NV; ++i) acc[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      const float* p = p0 + which * (64 * D) + tid * 4;
      for (int x = 0; x < ns; ++x, p += 2 * 64 * D) {
        f32x4_t b[NV];
#pragma unroll
        for (int i = 0; i < NV; ++i) b[i] = *reinterpret_cast<const f32x4_t*>(p + i * 512);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < NV; ++i) acc[i] += b[i];
      }
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        const int idx = tid * 4 + i * 512, r64 = idx / D, row = nb * 64 + r64;
        uint16_t* const dst = (which ? dv : dk) + head_off + (size_t)row * pitch + idx % D;
        const void* old = add ? dst : nullptr;
        if constexpr (LINEAR)
          old = smem + (4 * (r64 >> 5) + 2 * ((r64 >> 4) & 1) + 1 - which) * KEY_TILE<D> +
                lbs_off<D>(r64 & 15, idx % D);
        if (row < L) store_4<E>(dst, acc[i][0], acc[i][1], acc[i][2], acc[i][3], reinterpret_cast<const i32x2_t*>(old));
      }
    }
    return;
  }
#pragma unroll
  for (int which = 0; which < 2; ++which) {
    TileRows<D> t;
    t.unpark(stage + which * (64 * TileRows<D>::SSTR), lane);
    if constexpr (LINEAR)
#pragma unroll
      for (int i = 0; i < TileRows<D>::N; ++i) rows[which].x[i] = *reinterpret_cast<const i16x8_t*>(key_piece(1 - which, i));
    if (LINEAR || add) t.template add<E>(rows[which]);
    t.store_streaming((which == 0 ? dk : dv) + head_off + (size_t)krow0 * pitch, L - krow0, lane, pitch);
  }
}


template <typename Tag, int D>
__global__ __launch_bounds__(128) __attribute__((amdgpu_waves_per_eu(D == 64 ? 2 : 1, D == 64 ? 2 : 1))) void bwd_dkdv_stream_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ k, const uint16_t* __restrict__ v,
    const uint16_t* __restrict__ d_o, const float* __restrict__ lse, const float* __restrict__ delta,
    const int* __restrict__ list, const int* __restrict__ count, const i32x4_t* __restrict__ items,
    const int* __restrict__ totals, float* __restrict__ part, int seg, uint16_t* __restrict__ dk, uint16_t* __restrict__ dv,
    const RowLayout lin, const RowLayout ldo, int L, int Mblk, int Nblk, float qk_scale, int wide, int add,
    const int* __restrict__ nseg, int* __restrict__ done) {
  __shared__ __attribute__((aligned(16))) uint8_t smem[DKDV_LDS<D>];
  __shared__ int entries[DKDV_STREAM_MAX_SEG];
  // work item (see bwd_dkdv_kernel)
  const int total = totals[0];
  const int per_xcd = (total + 7) >> 3;
  if ((int)(blockIdx.x >> 3) >= per_xcd) return;
  const int logical = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  if (logical >= total) return;
  const i32x4_t item = items[logical];
  const int bh = __builtin_amdgcn_readfirstlane(item[0]), nb = __builtin_amdgcn_readfirstlane(item[1]);
  const int sg = __builtin_amdgcn_readfirstlane(item[2]), slot = __builtin_amdgcn_readfirstlane(item[3]);
  const int ns = slot < 0 ? 1 : nseg[(size_t)bh * Nblk + nb];
  dkdv_stream_body<Tag, D, false>(q, k, v, d_o, lse, delta, list, count, part, seg, dk, dv, lin, ldo, L, Mblk, Nblk, qk_scale, wide,
                                   add, done, LinearKeys{}, smem, entries, bh, nb, sg, slot, ns);
}

// ---- dQ ------------------------------------------------------------------------------------------------------------
// dQ of the block-sparse attention backward for 64-row query blocks: one wave per query block, one wave per SIMD, no
// barriers.
//
// Stands in for _attn_bwd_dq of the reference (sparse_linear_attention/kernel.py:95-157) like bwd_dq_kernel, whose
// arithmetic it shares (S^T = K Q^T and dP^T = V dO^T, so that the log-sum-exp and delta of a query are per-lane
// scalars and dS^T leaves the accumulator as the B operand of dQ^T += K^T dS^T).  What differs:
//   * the wave owns all 64 query rows (two tiles of 32): Q^T and dO^T fragments and the dQ^T accumulators fill the
//     accumulation registers, and every K or V fragment read from LDS feeds the products of both tiles;
//   * K and V go from memory straight into LDS, 32 keys at a time, two generations each, swizzled; a generation takes the
//     32 keys after next as soon as its fragments have been read (the transposed K fragments wait in registers);
//   * the loop is rotated: S and dP of both tiles of unit u + 1 (32 products) run beside the vector arithmetic of unit u,
//     then come dQ of unit u (16 products) beside the requests and the transposed fragments of unit u + 1.
// A lone wave issues one instruction per four cycles at best, and every one of them takes its turn with the 48 products
// (1536 cycles) of a unit, so instructions are what is saved: the accumulators of dP start from -delta instead of zero
// (no subtraction per element), four requests share one M0, every LDS offset but eight is an instruction immediate: 272
// instructions per unit where reading the row-wise fragments once per tile took 367.  Measured, that version against this:
// B1 H12 L32760 with 25 key blocks per row 551 -> 485 us (matrix pipe busy 49 -> 59 % of the cycles, at a clock that the
// power limit holds near 1.7 GHz), B2 H16 L32760 with 128-row blocks 1428 -> 1224 us, B2 H4 L4096 37.9 -> 33.2 us.
// Head dim 64 has dq_pair_body.
constexpr int DQ_STREAM_MAX_T = 2048;          // look-up rows longer than this take bwd_dq_kernel

template <int D>
constexpr int DQ_LDS = 4 * BwdTile<D>::BYTES;  // K generation 0, 1; V generation 0, 1

// The 64 query rows `logical`, by one wave.  smem: DQ_LDS bytes, entries: DQ_STREAM_MAX_T numbers of LDS, the wave's own.  DELTA: delta of
// these rows is formed here and written out; else it is read.
template <typename Tag, int D, bool DELTA>
static __device__ __forceinline__ void dq_stream_body(
    const uint16_t* q, const uint16_t* k, const uint16_t* v,
    const uint16_t* d_o, const uint16_t* o, const float* lse, float* delta,
    const void* lut, int lut64, uint16_t* dq, const RowLayout lin, const RowLayout ldo, int L,
    int Mblk, int topk, float qk_scale, int wide, int add, uint8_t* const smem, uint16_t* const entries, const int logical) {
  // (Mblk: 64-row blocks per head.  wide = 1: the look-up table has one row per 128-row block, which both halves follow.  add:
  //  dQ is added, rounded, to what dq holds.)
  using E = Elem<Tag>;
  using T32 = BwdTile<D>;
  static_assert(D == 128, "elements and requests are laid beside the products of head dim 128");
  constexpr int DC = D / 16, DT = D / 32;
  constexpr int TILE = T32::BYTES;                // 32 rows of K or V
  constexpr int NR = T32::NREQ;                   // requests per tile
  constexpr int ROWS8 = 8 / T32::RPR * REQ_PITCH; // 8 rows further on in a tile
  const int bh = logical / Mblk;
  const int mb = logical - bh * Mblk;
  const int lane = threadIdx.x & 63;
  const int g = lane >> 5, r = lane & 31;
  const float c_log2e = qk_scale * 1.4426950408889634f;

  const size_t head_off = lin.head(bh);
  const uint32_t pitch = (uint32_t)lin.sl, pitch_do = (uint32_t)ldo.sl;
  const uint32_t row_bytes = pitch * 2;
  const __amdgpu_buffer_rsrc_t qh = make_rsrc(q + head_off, lin.head_range_bytes(L, D));
  const __amdgpu_buffer_rsrc_t doh = make_rsrc(d_o + ldo.head(bh), ldo.head_range_bytes(L, D));
  const __amdgpu_buffer_rsrc_t kh = make_rsrc(k + head_off - REQ_SLACK / 2, lin.head_range_bytes(L, D) + REQ_SLACK);
  const __amdgpu_buffer_rsrc_t vh = make_rsrc(v + head_off - REQ_SLACK / 2, lin.head_range_bytes(L, D) + REQ_SLACK);
  const int qrow0 = mb * 64;

  // The first 64 entries of the look-up row are asked for before anything else: the first requests for K and V hang on
  // them, and loads come back in the order they were issued (the low word of a 64-bit entry is the entry).
  const size_t lut_row = wide ? ((size_t)bh * ((Mblk + 1) >> 1) + (mb >> 1)) * topk : ((size_t)bh * Mblk + mb) * topk;
  auto lut_at = [&](size_t i) __attribute__((always_inline)) -> int { return reinterpret_cast<const int*>(lut)[lut64 ? 2 * i : i]; };
  int first_entries = 0;
  if (topk > 0) first_entries = lut_at(lut_row + min(lane, topk - 1));      // (an empty table may be a null pointer)
  // Q^T and dO^T fragments (B operands; rows past L read as zero), per-lane scalars of the two query tiles
  // The rows of the forward's output come the same way: delta = rowsum(dO * O) (reference kernel.py:282-286, the
  // preprocess step) is formed here, for this block's rows, and written out for the dK/dV kernel.
  i16x8_t qf[2][DC], dof[2][DC], of[2][DC];
  float lse_q[2], delta_q[2];
  f32x16_t neg_delta[2];                          // sixteen copies of -delta: what the accumulators of dP start from
  const __amdgpu_buffer_rsrc_t oh = make_rsrc(o + (size_t)bh * L * D, (uint32_t)L * D * 2);      // (contiguous (B, H, L, D))
#pragma unroll
  for (int qt = 0; qt < 2; ++qt) {
    const int qrow = qrow0 + 32 * qt + r;
#pragma unroll
    for (int c = 0; c < DC; ++c) {
      qf[qt][c] = buf_load_b128(qh, ((uint32_t)qrow * pitch + 16 * c + 8 * g) * 2);
      dof[qt][c] = buf_load_b128(doh, ((uint32_t)qrow * pitch_do + 16 * c + 8 * g) * 2);
      if (DELTA) of[qt][c] = buf_load_b128(oh, ((uint32_t)qrow * D + 16 * c + 8 * g) * 2);       // rows past L: 0, delta 0
    }
    if (!DELTA) delta_q[qt] = qrow < L ? delta[(size_t)bh * L + qrow] : 0.f;
    // rows past L: lse = +inf makes every probability exactly 0 (the reference loads `other=inf`)
    lse_q[qt] = qrow < L ? lse[(size_t)bh * L + qrow] : INFINITY;
  }
  if (lane < topk) entries[lane] = (uint16_t)first_entries;
  for (int i = 64 + lane; i < topk; i += 64) entries[i] = (uint16_t)lut_at(lut_row + i);
  // key rows past L are never written into LDS: what LDS holds in their place has to be finite (their probabilities
  // are masked to exactly 0 below)
#pragma unroll
  for (int i = 0; i < (4 * TILE / 16 + 63) / 64; ++i)
    if (i * 64 + lane < 4 * TILE / 16) reinterpret_cast<i32x4_t*>(smem)[i * 64 + lane] = i32x4_t{0, 0, 0, 0};
  wave_lds_fence();

  // what dq holds, asked for before the last unit's arithmetic
  TileRows<D> old[2];
  const auto fetch_old = [&]() __attribute__((always_inline)) {
    if (!add) return;
#pragma unroll
    for (int qt = 0; qt < 2; ++qt)
      old[qt].fetch(dq + head_off + (size_t)(qrow0 + 32 * qt) * pitch, L - qrow0 - 32 * qt, lane, pitch);
  };

  f32x16_t dqacc[DT][2];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int qt = 0; qt < 2; ++qt)
#pragma unroll
      for (int i = 0; i < 16; ++i) dqacc[dt][qt][i] = 0.f;

  // ---- addressing ----
  // A request moves RPR rows (64 lanes x 16 bytes): lane -> row RPR j + lane / (D / 8), 16-byte slot lane % (D / 8), which
  // receives piece (slot ^ swz(row)) of that row.
  const uint32_t smem_addr = __builtin_amdgcn_readfirstlane((uint32_t)(size_t)smem);
  const int lrow = lane / (D / 8), lslot = lane % (D / 8);
  uint32_t koff[4];                  // requests 0 .. 3; sixteen rows more for requests 4 .. 7
#pragma unroll
  for (int j = 0; j < 4; ++j)
    koff[j] = (uint32_t)(T32::RPR * j + lrow) * row_bytes + (uint32_t)(lslot ^ T32::swz(lrow)) * 16 + REQ_SLACK - j * REQ_PITCH;
  const uint32_t half_bytes = 16 * row_bytes;
  const int row_none = (L + 63) & ~63;            // past every head: such requests touch neither memory nor LDS
  auto entry_row0 = [&](int e) __attribute__((always_inline)) -> int {
    const int row0 = __builtin_amdgcn_readfirstlane((int)entries[min(e, topk - 1)]) * 64;
    return e < topk ? row0 : row_none;
  };
  // request J (rows RPR J ..) of the 32 rows from key0 on, into the tile at LDS address `tile`; SET: the first of its group
#define SLA_DQ_REQUEST(RSRC, J, SET, KEY0, TILE_AT)                                                                  \
  lds_dma_row4<(J) & 3, SET>(RSRC, koff[(J) & 3] + ((uint32_t)(KEY0) * row_bytes + ((J) >= 4 ? half_bytes : 0u)),     \
                             smem_addr + (uint32_t)(TILE_AT) + ((J) >> 2) * 4 * REQ_PITCH)
  // the first (H = 0) or second sixteen rows of a tile, request i of them
  auto request_half = [&](const __amdgpu_buffer_rsrc_t& rsrc, auto h, auto i, int key0, int tile_at) __attribute__((always_inline)) {
    constexpr int J = decltype(h)::value * (NR / 2) + decltype(i)::value;
    SLA_DQ_REQUEST(rsrc, J, decltype(i)::value == 0, key0, tile_at);
  };
  auto request_rows = [&](const __amdgpu_buffer_rsrc_t& rsrc, auto h, int key0, int tile_at) __attribute__((always_inline)) {
    request_half(rsrc, h, I<0>{}, key0, tile_at);
    request_half(rsrc, h, I<1>{}, key0, tile_at);
    request_half(rsrc, h, I<2>{}, key0, tile_at);
    request_half(rsrc, h, I<3>{}, key0, tile_at);
  };
  // fragments: row-wise, row r, piece 2 c + g: four bases; transposed, rows tr_row and tr_row + 8 (and 16 further for the
  // second half), 8 bytes at element 4 (lane % 4) of the 16-column strip 2 dt + (lane / 16) % 2: one base per dt
  const uint8_t* rfp[4];
  const uint8_t* tfp[DT];
  const int tr_row = 4 * g + ((lane & 15) >> 2);
#pragma unroll
  for (int i = 0; i < 4; ++i) rfp[i] = smem + T32::piece_at(r, 2 * (i * DC / 4) + g);
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
    tfp[dt] = smem + T32::piece_at(tr_row, 4 * dt + 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1)) + (lane & 1) * 8;
  i16x8_t af[3], bf[3];              // row-wise K and V fragments, two chunks ahead
  i16x8_t trk[2][DT];                // transposed K fragments of the unit whose dQ products come next
  auto row_frags = [&](int GEN, int c) __attribute__((always_inline)) {
    const uint8_t* p = rfp[c * 4 / DC] + GEN * TILE + (c & 1) * 32;
    af[c % 3] = *reinterpret_cast<const i16x8_t*>(p);
    bf[c % 3] = *reinterpret_cast<const i16x8_t*>(p + 2 * TILE);
  };
  auto tr_frag = [&](int GEN, int c2, int dt) __attribute__((always_inline)) {
    const uint8_t* t0 = tfp[dt] + GEN * TILE + 2 * c2 * ROWS8;
    trk[c2][dt] = concat4(lds_read_tr16(reinterpret_cast<const uint16_t*>(t0)),
                          lds_read_tr16(reinterpret_cast<const uint16_t*>(t0 + ROWS8)));
  };

  struct Tiles {
    f32x16_t s[2], dp[2];            // S^T and dP^T - delta of the two query tiles
  };
  Tiles ta, tb;
  i32x4_t dsw[2][2];                 // dS^T of the two query tiles, packed: B operands of the dQ products
  // element i of tile qt: P = exp2(S c - lse), then dS = P (dP - delta), two per packed word
  auto prob = [&](Tiles& t, int qt, int i) __attribute__((always_inline)) {
    float p = fast_exp2(__builtin_fmaf(t.s[qt][i], c_log2e, -lse_q[qt]));
    asm volatile("" : "+v"(p));
    t.s[qt][i] = p;
  };
  auto grad = [&](Tiles& t, int qt, int i) __attribute__((always_inline)) {
    float ds = t.s[qt][i] * t.dp[qt][i];
    asm volatile("" : "+v"(ds));
    t.dp[qt][i] = ds;
    if (i & 1) {
      uint32_t a = E::pack2(t.dp[qt][i - 1], t.dp[qt][i]);
      asm volatile("" : "+v"(a));
      dsw[qt][i >> 3][(i >> 1) & 3] = (int)a;
    }
  };
  // element e of the unit's 32 in the order the dQ products want them: the first eight registers of both tiles, then the others
  auto element = [&](Tiles& t, int e) __attribute__((always_inline)) {
    const auto qt = [](int n) __attribute__((always_inline)) { return (n >> 3) & 1; };
    const auto at = [](int n) __attribute__((always_inline)) { return (n >> 4) * 8 + (n & 7); };
    if (e < 32) prob(t, qt(e), at(e));
    if (e > 0) grad(t, qt(e - 1), at(e - 1));
  };
  // product 4 c + {0, 1, 2, 3} of the first ones: S and dP of tile 0, then of tile 1, chunk c of the head dimension
  auto score_product = [&](Tiles& t, int c, int which) __attribute__((always_inline)) {
    const int qt = which >> 1;
    if (which & 1) {
      if (c == 0) mfma_scores_first<Tag>(t.dp[qt], bf[0], dof[qt][0], neg_delta[qt]);
      else mfma_scores<Tag>(t.dp[qt], bf[c % 3], dof[qt][c]);
    } else {
      if (c == 0) mfma_scores_first<Tag>(t.s[qt], af[0], qf[qt][0]);
      else mfma_scores<Tag>(t.s[qt], af[c % 3], qf[qt][c]);
    }
  };
  auto mask_tail = [&](Tiles& t, int valid) __attribute__((always_inline)) {   // key index of register i is 8 (i / 4) + i % 4 + 4 g
    const int lim = valid - 4 * g;
#pragma unroll
    for (int qt = 0; qt < 2; ++qt)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        float x = 8 * (i >> 2) + (i & 3) >= lim ? -INFINITY : t.s[qt][i];
        asm volatile("" : "+v"(x));              // (in place, one after the other: no second copy of the tile)
        t.s[qt][i] = x;
      }
  };

  // One iteration = unit u (generation GU = u % 2), 3 D / 8 products:
  //   first two thirds  S and dP of unit u + 1 into `nxt`     beside: P and dS of unit u (in `cur`), K rows 16.. of unit u + 2
  //   last third        dQ += K^T dS of unit u                 beside: V and K rows 0..15 of unit u + 3, and from unit u + 1
  //                                                            the transposed K fragments, from u + 2 the first row-wise ones
  // Requests are answered in order.  When the row-wise fragments of unit u + 2 are first read, only the requests for V of
  // unit u + 3 may be out; a tile half is requested again only behind a product that waited for LDS reads issued after
  // the last read of that half (LDS reads return in order).
  auto iteration = [&](auto gu, Tiles& cur, Tiles& nxt, int key_u, int key_u2, int key_u3) __attribute__((always_inline)) {
    constexpr int GU = decltype(gu)::value, GN = GU ^ 1;
    if (__builtin_expect(L - key_u < 32, 0)) mask_tail(cur, L - key_u);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < DC; ++c) {
#pragma unroll
      for (int which = 0; which < 4; ++which) {
        const int sl = 4 * c + which;
        score_product(nxt, c, which);
#pragma unroll
        for (int e = sl * 32 / (4 * DC); e < (sl + 1) * 32 / (4 * DC); ++e) element(cur, e);
        if (which == 1 && c + 2 < DC) row_frags(GN, c + 2);
        if (sl == 12) request_half(kh, I<1>{}, I<0>{}, key_u2, GU * TILE);
        if (sl == 15) request_half(kh, I<1>{}, I<1>{}, key_u2, GU * TILE);
        if (sl == 18) request_half(kh, I<1>{}, I<2>{}, key_u2, GU * TILE);
        if (sl == 21) request_half(kh, I<1>{}, I<3>{}, key_u2, GU * TILE);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    element(cur, 32);
#pragma unroll
    for (int sl = 0; sl < 4 * DT; ++sl) {
      const int c2 = sl / (2 * DT), dt = (sl >> 1) % DT, qt = sl & 1;
      dqacc[dt][qt] = E::mfma32(trk[c2][dt], __builtin_bit_cast(i16x8_t, dsw[qt][c2]), dqacc[dt][qt]);
      if (sl == 0) request_half(vh, I<0>{}, I<0>{}, key_u3, (2 + GN) * TILE);
      if (sl == 1) request_half(vh, I<0>{}, I<1>{}, key_u3, (2 + GN) * TILE);
      if (sl == 2) request_half(vh, I<0>{}, I<2>{}, key_u3, (2 + GN) * TILE);
      if (sl == 3) request_half(vh, I<0>{}, I<3>{}, key_u3, (2 + GN) * TILE);
      if (sl == 4) request_half(vh, I<1>{}, I<0>{}, key_u3, (2 + GN) * TILE);
      if (sl == 5) request_half(vh, I<1>{}, I<1>{}, key_u3, (2 + GN) * TILE);
      if (sl == 6) request_half(vh, I<1>{}, I<2>{}, key_u3, (2 + GN) * TILE);
      if (sl == 7) request_half(vh, I<1>{}, I<3>{}, key_u3, (2 + GN) * TILE);
      if (qt == 1) tr_frag(GN, c2, dt);
      constexpr int W = 9;                                     // unit u + 2 has landed from here on
      if (sl == W) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NR) : "memory");
      if (sl == W + 1) row_frags(GU, 0);
      if (sl == 12) {
        row_frags(GU, 1);
        asm volatile("s_waitcnt lgkmcnt(4)" ::: "memory");     // (K rows 0..15 of unit u + 1 have been read: six or more reads came after)
        request_half(kh, I<0>{}, I<0>{}, key_u3, GN * TILE);
      }
      if (sl == 13) request_half(kh, I<0>{}, I<1>{}, key_u3, GN * TILE);
      if (sl == 14) request_half(kh, I<0>{}, I<2>{}, key_u3, GN * TILE);
      if (sl == 15) request_half(kh, I<0>{}, I<3>{}, key_u3, GN * TILE);
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // first key rows of the listed blocks: E0 of the entry of units u and u + 1, E1 of the next one, E2 of the one after
  int E0 = 0, E1 = 0, E2 = 0;
  if (topk > 0) {
    E0 = entry_row0(0);
    E1 = entry_row0(1);
    E2 = entry_row0(2);
    request_rows(kh, I<0>{}, E0, 0);
    request_rows(kh, I<1>{}, E0, 0);
    request_rows(vh, I<0>{}, E0, 2 * TILE);
    request_rows(vh, I<1>{}, E0, 2 * TILE);
    request_rows(kh, I<0>{}, E0 + 32, TILE);
    request_rows(kh, I<1>{}, E0 + 32, TILE);
    request_rows(vh, I<0>{}, E0 + 32, 3 * TILE);
    request_rows(vh, I<1>{}, E0 + 32, 3 * TILE);
  }
  // delta of this lane's two rows.  The sum runs in the order of bwd_delta_kernel, whose thread t adds the eight products
  // of columns 8t .. 8t+7 (delta_sum8) and then meets threads t^1, t^2, t^4, t^8: here t = 2c + g, so the first
  // meeting is the one with lane^32 and the other three are between this lane's own chunks.
#pragma unroll
  for (int qt = 0; qt < 2; ++qt) {
    if constexpr (!DELTA) {
#pragma unroll
      for (int i = 0; i < 16; ++i) neg_delta[qt][i] = -delta_q[qt];
      asm volatile("" : "+v"(neg_delta[qt]));
      continue;
    }
    float part[DC];
#pragma unroll
    for (int c = 0; c < DC; ++c) {
      const float acc = delta_sum8<Tag>(of[qt][c], dof[qt][c]);
      part[c] = acc + __shfl_xor(acc, 32);
    }
#pragma unroll
    for (int sh = 1; sh < DC; sh <<= 1)
#pragma unroll
      for (int c = 0; c < DC; c += 2 * sh) part[c] = part[c] + part[c + sh];
#pragma unroll
    for (int i = 0; i < 16; ++i) neg_delta[qt][i] = -part[0];
    asm volatile("" : "+v"(neg_delta[qt]));
    const int qrow = qrow0 + 32 * qt + r;
    if (g == 0 && qrow < L) delta[(size_t)bh * L + qrow] = part[0];
  }
  // Q^T and dO^T are only ever MFMA operands and are parked in the accumulation registers (the wait for them comes
  // here, behind the first requests for K and V, which only needed the look-up row)
#pragma unroll
  for (int qt = 0; qt < 2; ++qt)
#pragma unroll
    for (int c = 0; c < DC; ++c) asm volatile("" : "+a"(qf[qt][c]), "+a"(dof[qt][c]));
  if (topk > 0) {
    // (the two rows of delta written above count as memory operations too: two more may be out)
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * NR) : "memory");
    row_frags(0, 0);
    row_frags(0, 1);
#pragma unroll
    for (int c = 0; c < DC; ++c) {
#pragma unroll
      for (int which = 0; which < 4; ++which) score_product(ta, c, which);
      if (c + 2 < DC) row_frags(0, c + 2);
    }
#pragma unroll
    for (int c2 = 0; c2 < 2; ++c2)
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) tr_frag(0, c2, dt);
    // (the vector ALU reads the products' results next; every fragment of unit 0 has been read)
    asm volatile("s_nop 15\n\ts_nop 15\n\ts_waitcnt lgkmcnt(0)" ::: "memory");
    request_rows(vh, I<0>{}, E1, 2 * TILE);
    request_rows(vh, I<1>{}, E1, 2 * TILE);
    request_rows(kh, I<0>{}, E1, 0);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NR + NR / 2) : "memory");
    row_frags(1, 0);
    row_frags(1, 1);
    for (int b = 0;; ++b) {
      const int E3 = entry_row0(b + 3);                       // (looked up now, used two units from now)
      iteration(I<0>{}, ta, tb, E0, E1, E1 + 32);                  // unit 2 b
      if (b + 1 >= topk) break;
      iteration(I<1>{}, tb, ta, E0 + 32, E1 + 32, E2);             // unit 2 b + 1
      E0 = E1;
      E1 = E2;
      E2 = E3;
    }
    // the last unit: no scores left to form beside its arithmetic
    fetch_old();
    if (__builtin_expect(L - (E0 + 32) < 32, 0)) mask_tail(tb, L - (E0 + 32));
#pragma unroll
    for (int e = 0; e <= 32; ++e) element(tb, e);
#pragma unroll
    for (int sl = 0; sl < 4 * DT; ++sl) {
      const int c2 = sl / (2 * DT), dt = (sl >> 1) % DT, qt = sl & 1;
      dqacc[dt][qt] = E::mfma32(trk[c2][dt], __builtin_bit_cast(i16x8_t, dsw[qt][c2]), dqacc[dt][qt]);
    }
  }
  if (topk <= 0) fetch_old();
#undef SLA_DQ_REQUEST
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // (nothing of this workgroup is in flight when it ends)

  // The rounded rows go through LDS (the rings are free now) and leave as whole rows in streaming stores: they are not
  // read again here, and what does not stay behind as modified lines in L2 need not be written back when the kernel ends.
  uint16_t* const stage = reinterpret_cast<uint16_t*>(smem);
#pragma unroll
  for (int qt = 0; qt < 2; ++qt) {
    constexpr int SSTR = TileRows<D>::SSTR;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int i4 = 0; i4 < 4; ++i4) {
        i32x2_t wv;
        wv[0] = (int)E::pack2(dqacc[dt][qt][4 * i4 + 0] * qk_scale, dqacc[dt][qt][4 * i4 + 1] * qk_scale);
        wv[1] = (int)E::pack2(dqacc[dt][qt][4 * i4 + 2] * qk_scale, dqacc[dt][qt][4 * i4 + 3] * qk_scale);
        *reinterpret_cast<i32x2_t*>(&stage[r * SSTR + 32 * dt + 8 * i4 + 4 * g]) = wv;
      }
    wave_lds_fence();
    TileRows<D> t;
    t.unpark(stage, lane);
    if (add) t.template add<E>(old[qt]);
    t.store_streaming(dq + head_off + (size_t)(qrow0 + 32 * qt) * pitch, L - qrow0 - 32 * qt, lane, pitch);
    wave_lds_fence();
  }
}

template <typename Tag, int D>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(1, 1))) void bwd_dq_stream_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ k, const uint16_t* __restrict__ v,
    const uint16_t* __restrict__ d_o, const uint16_t* __restrict__ o, const float* __restrict__ lse, float* __restrict__ delta,
    const void* __restrict__ lut, int lut64, uint16_t* __restrict__ dq, const RowLayout lin, const RowLayout ldo, int L,
    int Mblk, int topk, float qk_scale, int total, int wide, int add, int first_wg, const Segments segs, const HeadSums heads) {
  // (The first `first_wg` workgroups, a multiple of eight, take the short jobs along that dK/dV and the caller wait for: they are
  //  done long before the rest.)
  __shared__ __attribute__((aligned(16))) uint8_t smem[DQ_LDS<D>];
  __shared__ uint16_t entries[DQ_STREAM_MAX_T];                        // this block's look-up row
  if ((int)blockIdx.x < first_wg) {
    const int job = blockIdx.x;
    if (job < segs.wgs) segments_body(segs, job);
    else if (job < segs.wgs + heads.wgs) head_sums_body(heads, job - segs.wgs);
    return;
  }
  const int logical = xcd_remap((int)blockIdx.x - first_wg, (int)gridDim.x - first_wg, total);
  if (logical < 0) return;
  dq_stream_body<Tag, D, true>(q, k, v, d_o, o, lse, delta, lut, lut64, dq, lin, ldo, L, Mblk, topk, qk_scale, wide, add, smem, entries,
                               logical);
}

// The 64 query rows `logical` by two waves of 32 rows each, for a launch whose waves share a SIMD in twos (head dim 64): half the
// registers of a wave with all 64 (364, which dK/dV's waves cannot share a SIMD with), K and V in rings of four generations of 32 keys that both waves request and read, one barrier
// per generation, delta read.  Order of the products, arithmetic and roundings follow dq_stream_body's scheme, which has head dim 128.
// smem: DQ_PAIR_LDS bytes, entries: DQ_STREAM_MAX_T numbers of LDS.
template <int D>
constexpr int DQ_PAIR_LDS = 8 * BwdTile<D>::BYTES;      // four generations: 32 rows of K and of V

template <typename Tag, int D>
static __device__ __forceinline__ void dq_pair_body(const uint16_t* q, const uint16_t* k, const uint16_t* v, const uint16_t* d_o,
                                                    const float* lse, const float* delta, const void* lut, int lut64, uint16_t* dq,
                                                    const RowLayout lin, const RowLayout ldo, int L, int Mblk, int topk,
                                                    float qk_scale, int wide, int add, uint8_t* const smem, uint16_t* const entries,
                                                    const int logical) {
  using E = Elem<Tag>;
  using T32 = BwdTile<D>;
  static_assert(D == 64, "elements and requests are laid beside the products of head dim 64");
  constexpr int DC = D / 16, DT = D / 32;
  constexpr int TILE = T32::BYTES, GEN = 2 * TILE;
  constexpr int NR = T32::NREQ / 2, NREQ = 2 * NR;             // requests per wave and tile, and unit
  constexpr int ROWS8 = 8 / T32::RPR * REQ_PITCH;
  const int bh = logical / Mblk, mb = logical - bh * Mblk;
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 5, r = lane & 31;
  const float c_log2e = qk_scale * 1.4426950408889634f;

  const size_t head_off = first_lane64(lin.head(bh)), head_do = first_lane64(ldo.head(bh));
  const uint32_t pitch = (uint32_t)lin.sl, pitch_do = (uint32_t)ldo.sl, row_bytes = pitch * 2;
  const __amdgpu_buffer_rsrc_t qh = make_rsrc(q + head_off, lin.head_range_bytes(L, D));
  const __amdgpu_buffer_rsrc_t doh = make_rsrc(d_o + head_do, ldo.head_range_bytes(L, D));
  const __amdgpu_buffer_rsrc_t kh = make_rsrc(k + head_off - REQ_SLACK / 2, lin.head_range_bytes(L, D) + REQ_SLACK);
  const __amdgpu_buffer_rsrc_t vh = make_rsrc(v + head_off - REQ_SLACK / 2, lin.head_range_bytes(L, D) + REQ_SLACK);

  // (the look-up row first, as in dq_stream_body)
  const size_t lut_row = wide ? ((size_t)bh * ((Mblk + 1) >> 1) + (mb >> 1)) * topk : ((size_t)bh * Mblk + mb) * topk;
  const auto lut_at = [&](size_t i) __attribute__((always_inline)) -> int { return reinterpret_cast<const int*>(lut)[lut64 ? 2 * i : i]; };
  int first_entries = 0;
  if (topk > 0) first_entries = lut_at(lut_row + min(tid, topk - 1));       // (an empty table may be a null pointer)
  const int qrow0 = mb * 64 + 32 * w, qrow = qrow0 + r;
  i16x8_t qf[DC], dof[DC];                                                    // rows past L read as zero
#pragma unroll
  for (int c = 0; c < DC; ++c) {
    qf[c] = buf_load_b128(qh, ((uint32_t)qrow * pitch + 16 * c + 8 * g) * 2);
    dof[c] = buf_load_b128(doh, ((uint32_t)qrow * pitch_do + 16 * c + 8 * g) * 2);
  }
  const float lse_q = qrow < L ? lse[(size_t)bh * L + qrow] : INFINITY;     // (+inf: every probability exactly 0)
  const float delta_q = qrow < L ? delta[(size_t)bh * L + qrow] : 0.f;
  if (tid < topk) entries[tid] = (uint16_t)first_entries;
  for (int i = 128 + tid; i < topk; i += 128) entries[i] = (uint16_t)lut_at(lut_row + i);
  // (key rows past L are never written into LDS: what it holds in their place has to be finite)
#pragma unroll
  for (int i = 0; i < (4 * GEN / 16 + 127) / 128; ++i)
    if (i * 128 + tid < 4 * GEN / 16) reinterpret_cast<i32x4_t*>(smem)[i * 128 + tid] = i32x4_t{0, 0, 0, 0};

  TileRows<D> old;
  const auto fetch_old = [&]() __attribute__((always_inline)) {
    if (add) old.fetch(dq + head_off + (size_t)qrow0 * pitch, L - qrow0, lane, pitch);
  };
  f32x16_t dqacc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) dqacc[dt][i] = 0.f;

  // ---- addressing (as in dkdv_stream_body: a wave requests 16 rows of a tile) ----
  const uint32_t smem_addr = (uint32_t)(size_t)smem;
  const int lrow = lane / (D / 8), lslot = lane % (D / 8);
  uint32_t koff[NR];
#pragma unroll
  for (int j = 0; j < NR; ++j)
    koff[j] = (uint32_t)(16 * w + T32::RPR * j + lrow) * row_bytes + (uint32_t)(lslot ^ T32::swz(lrow)) * 16 + REQ_SLACK - j * REQ_PITCH;
  const uint32_t rows_base = __builtin_amdgcn_readfirstlane(smem_addr + (uint32_t)(NR * w) * REQ_PITCH);
  const int row_none = (L + 63) & ~63;
  const auto entry_row0 = [&](int e) __attribute__((always_inline)) -> int {
    const int row0 = __builtin_amdgcn_readfirstlane((int)entries[min(e, topk - 1)]) * 64;
    return e < topk ? row0 : row_none;
  };
#define SLA_DQ_REQUEST(RSRC, J, KEY0, AT) lds_dma_row4<J>(RSRC, koff[J] + (uint32_t)(KEY0) * row_bytes, rows_base + (uint32_t)(AT))
  const uint8_t* rfp[4];
  const uint8_t* tfp[DT];
  const int tr_row = 4 * g + ((lane & 15) >> 2);
#pragma unroll
  for (int i = 0; i < 4; ++i) rfp[i] = smem + T32::piece_at(r, 2 * (i * DC / 4) + g);
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
    tfp[dt] = smem + T32::piece_at(tr_row, 4 * dt + 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1)) + (lane & 1) * 8;
  i16x8_t af[3], bf[3];              // row-wise K and V fragments, two chunks ahead
  i16x8_t trk[2][DT];                // transposed K fragments
  const auto row_frags = [&](int at, int c) __attribute__((always_inline)) {
    const uint8_t* p = rfp[c * 4 / DC] + at;
    af[c % 3] = *reinterpret_cast<const i16x8_t*>(p);
    bf[c % 3] = *reinterpret_cast<const i16x8_t*>(p + TILE);
  };
  const auto tr_frag = [&](int at, int c2, int dt) __attribute__((always_inline)) {
    const uint8_t* t0 = tfp[dt] + at + 2 * c2 * ROWS8;
    trk[c2][dt] = concat4(lds_read_tr16(reinterpret_cast<const uint16_t*>(t0)),
                          lds_read_tr16(reinterpret_cast<const uint16_t*>(t0 + ROWS8)));
  };
  f32x16_t neg_delta, s_a, dp_a, s_b, dp_b;      // S^T and dP^T - delta of two units
  i32x4_t dsw[2];
  const auto prob = [&](f32x16_t& s, int i) __attribute__((always_inline)) {
    float p = fast_exp2(__builtin_fmaf(s[i], c_log2e, -lse_q));
    asm volatile("" : "+v"(p));
    s[i] = p;
  };
  const auto grad = [&](f32x16_t& s, f32x16_t& dp, int i) __attribute__((always_inline)) {
    float ds = s[i] * dp[i];
    asm volatile("" : "+v"(ds));
    dp[i] = ds;
    if (i & 1) {
      uint32_t a = E::pack2(dp[i - 1], dp[i]);
      asm volatile("" : "+v"(a));
      dsw[i >> 3][(i >> 1) & 3] = (int)a;
    }
  };
  const auto score_product = [&](f32x16_t& s, f32x16_t& dp, int c, int which) __attribute__((always_inline)) {
    if (which) {
      if (c == 0) mfma_scores_first<Tag>(dp, bf[0], dof[0], neg_delta);
      else mfma_scores<Tag>(dp, bf[c % 3], dof[c]);
    } else {
      if (c == 0) mfma_scores_first<Tag>(s, af[0], qf[0]);
      else mfma_scores<Tag>(s, af[c % 3], qf[c]);
    }
  };
  const auto mask_tail = [&](f32x16_t& s, int valid) __attribute__((always_inline)) {
    const int lim = valid - 4 * g;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      float x = 8 * (i >> 2) + (i & 3) >= lim ? -INFINITY : s[i];
      asm volatile("" : "+v"(x));
      s[i] = x;
    }
  };
  const auto dq_product = [&](int n) __attribute__((always_inline)) {
    const int c2 = n / DT, dt = n % DT;
    dqacc[dt] = E::mfma32(trk[c2][dt], __builtin_bit_cast(i16x8_t, dsw[c2]), dqacc[dt]);
  };

  // One iteration = unit u in generation GU = u % 4: S and dP of unit u + 1 beside the arithmetic of unit u and its transposed
  // fragments, then dQ += K^T dS of unit u.  The barrier stands where this wave has read all of unit u's generation and its part of
  // unit u + 2 has landed (only the requests for unit u + 3 may be out); behind it unit u + 4 is requested into unit u's place.
  const auto iteration = [&](auto gu, f32x16_t& s_cur, f32x16_t& dp_cur, f32x16_t& s_nxt, f32x16_t& dp_nxt, int key_u,
                             int key_u4) __attribute__((always_inline)) {
    constexpr int EA = 12;                                       // elements beside the first products
    constexpr int GU = decltype(gu)::value, AT0 = GU * GEN, AT1 = ((GU + 1) & 3) * GEN, AT2 = ((GU + 2) & 3) * GEN;
    if (__builtin_expect(L - key_u < 32, 0)) mask_tail(s_cur, L - key_u);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < DC; ++c)
#pragma unroll
      for (int which = 0; which < 2; ++which) {
        const int sl = 2 * c + which;
        score_product(s_nxt, dp_nxt, c, which);
#pragma unroll
        for (int i = sl * EA / (2 * DC); i < (sl + 1) * EA / (2 * DC); ++i) {
          prob(s_cur, i);
          if (i > 0) grad(s_cur, dp_cur, i - 1);
        }
        if (which == 0 && c + 2 < DC) row_frags(AT1, c + 2);
        if (sl >= 2 && sl < 6) tr_frag(AT0, (sl - 2) / DT, (sl - 2) % DT);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
    for (int n = 0; n < 2 * DT; ++n) {
      if (n == 1) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(NREQ) : "memory");
      if (n == DT) grad(s_cur, dp_cur, 15);
      dq_product(n);
      if (n < DT) {
        constexpr int PER = (16 - EA) / DT;
#pragma unroll
        for (int i = EA + n * PER; i < EA + (n + 1) * PER; ++i) {
          prob(s_cur, i);
          grad(s_cur, dp_cur, i - 1);
        }
      }
      if (n == 1) {
        SLA_DQ_REQUEST(kh, 0, key_u4, AT0);
        SLA_DQ_REQUEST(kh, 1, key_u4, AT0);
        row_frags(AT2, 0);
      }
      if (n == 2) {
        SLA_DQ_REQUEST(vh, 0, key_u4, AT0 + TILE);
        SLA_DQ_REQUEST(vh, 1, key_u4, AT0 + TILE);
        row_frags(AT2, 1);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  __syncthreads();                                               // the zeros and the entries are in place before anything is requested
  int E0 = 0, E1 = 0, E2 = 0;
  if (topk > 0) {
    const auto request_unit = [&](int key0, int gen) __attribute__((always_inline)) {
      SLA_DQ_REQUEST(kh, 0, key0, gen * GEN);
      SLA_DQ_REQUEST(kh, 1, key0, gen * GEN);
      SLA_DQ_REQUEST(vh, 0, key0, gen * GEN + TILE);
      SLA_DQ_REQUEST(vh, 1, key0, gen * GEN + TILE);
    };
    E0 = entry_row0(0);
    E1 = entry_row0(1);
    E2 = entry_row0(2);
    request_unit(E0, 0);
    request_unit(E0 + 32, 1);
    request_unit(E1, 2);
    request_unit(E1 + 32, 3);
  }
  // (the wait for the rows' loads comes here, behind the first requests)
#pragma unroll
  for (int i = 0; i < 16; ++i) neg_delta[i] = -delta_q;
  asm volatile("" : "+v"(neg_delta));
#pragma unroll
  for (int c = 0; c < DC; ++c) asm volatile("" : "+a"(qf[c]), "+a"(dof[c]));
  if (topk > 0) {
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(3 * NREQ) : "memory");
    row_frags(0, 0);
    row_frags(0, 1);
#pragma unroll
    for (int c = 0; c < DC; ++c) {
      score_product(s_a, dp_a, c, 0);
      score_product(s_a, dp_a, c, 1);
      if (c + 2 < DC) row_frags(0, c + 2);
    }
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");          // (the vector ALU reads these results next)
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(2 * NREQ) : "memory");
    row_frags(GEN, 0);
    row_frags(GEN, 1);
    int last_at;                                                 // where the last unit lies
    for (int b = 0;; b += 2) {
      int E3 = entry_row0(b + 3);
      iteration(I<0>{}, s_a, dp_a, s_b, dp_b, E0, E2);
      last_at = GEN;
      if (b + 1 >= topk) break;
      iteration(I<1>{}, s_b, dp_b, s_a, dp_a, E0 + 32, E2 + 32);
      E0 = E1;
      E1 = E2;
      E2 = E3;
      E3 = entry_row0(b + 4);
      iteration(I<2>{}, s_a, dp_a, s_b, dp_b, E0, E2);
      last_at = 3 * GEN;
      if (b + 2 >= topk) break;
      iteration(I<3>{}, s_b, dp_b, s_a, dp_a, E0 + 32, E2 + 32);
      E0 = E1;
      E1 = E2;
      E2 = E3;
    }
    // the last unit: no scores left to form beside its arithmetic
    fetch_old();
    if (__builtin_expect(L - (E0 + 32) < 32, 0)) mask_tail(s_b, L - (E0 + 32));
#pragma unroll
    for (int n = 0; n < 2 * DT; ++n) tr_frag(last_at, n / DT, n % DT);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      prob(s_b, i);
      grad(s_b, dp_b, i);
    }
#pragma unroll
    for (int n = 0; n < 2 * DT; ++n) dq_product(n);
  } else {
    fetch_old();
  }
#undef SLA_DQ_REQUEST
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");              // (nothing of this workgroup is in flight when it ends)
  __syncthreads();                                               // (both waves are done with the generations)
  uint16_t* const stage = reinterpret_cast<uint16_t*>(smem) + w * (32 * TileRows<D>::SSTR);
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int i4 = 0; i4 < 4; ++i4) {
      i32x2_t wv;
      wv[0] = (int)E::pack2(dqacc[dt][4 * i4 + 0] * qk_scale, dqacc[dt][4 * i4 + 1] * qk_scale);
      wv[1] = (int)E::pack2(dqacc[dt][4 * i4 + 2] * qk_scale, dqacc[dt][4 * i4 + 3] * qk_scale);
      *reinterpret_cast<i32x2_t*>(&stage[r * TileRows<D>::SSTR + 32 * dt + 8 * i4 + 4 * g]) = wv;
    }
  wave_lds_fence();
  TileRows<D> t;
  t.unpark(stage, lane);
  if (add) t.template add<E>(old);
  t.store_streaming(dq + head_off + (size_t)qrow0 * pitch, L - qrow0, lane, pitch);
}

// ---- both in one launch ------------------------------------------------------------------------------------------------
// dK/dV and dQ: with delta formed beforehand the two need nothing of each other, and what either leaves idle of the machine the other
// takes.  First come the key blocks, whose lists differ in length, then the query blocks (at head dim 128 two per workgroup), all equally
// long, which fill the places that short lists leave early.  Kernels in us, apart and together: 8 heads x 4096 x 128, 12 of 64 key blocks
// 35.5 + 51.0 / 67.6; 12 x 9360 x 128, 14 of 147, 128-row blocks 96 + 128 / 204; 16 x 6001 x 64, 9 of 94 41.9 + 52.7 / 71.6; 12 x 16380 x 128,
// 12 of 256 145 + 172 / 285.
struct BwdBoth {
  const uint16_t *q, *k, *v, *d_o;
  const float *lse, *delta;
  const int *list, *count;
  const i32x2_t* cuts;
  float* part;
  uint16_t *dq, *dk, *dv;
  int* done;
  const void* lut;
  RowLayout lin, ldo;
  int lut64, seg, room, nblocks, L, Mblk, Mblk64, Nblk, topk, wide, add, total_q;
  int head_wgs, key_wgs, cut_wgs;             // workgroups of the sums over the heads, of the key blocks, of cut lists' further segments
  float qk_scale;
};
// Work item i, as segments_body numbers them, but with the key blocks' first segments ahead of all further ones: i < nblocks is key
// block i, nblocks + x the x-th further segment.  Only a cut list wants sums over the counts before its own, which a wave then
// forms for itself: over the strips' sums, then inside the strip.  False: there is no such item.
static __device__ __forceinline__ bool both_item(const BwdBoth& a, int i, int& bh, int& nb, int& sg, int& slot, int& ns) {
  const int lane = threadIdx.x & 63;
  sg = 0;
  slot = -1;
  ns = 1;
  if (i < a.nblocks) {
    bh = i / a.Nblk;
    nb = i - bh * a.Nblk;
    if (further_segments(a.count[i], a.seg) == 0) return true;
  }
  const int x = i - a.nblocks, strips = (a.Nblk + 63) >> 6, all = a.nblocks / a.Nblk * strips;
  const int mine = x < 0 ? bh * strips + (nb >> 6) : -1;                 // this key block's strip
  const auto scan = [&](int n) {                                         // over the lanes, inclusive
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int t = __shfl_up(n, o);
      if (lane >= o) n += t;
    }
    return n;
  };
  int strip = -1, extra0 = 0, cuts0 = 0;                                  // further segments and cut lists before it
  for (int first = 0; first < all && strip < 0; first += 64) {
    const int at = first + lane;
    const i32x2_t c = at < all ? a.cuts[at] : i32x2_t{0, 0};
    const int upto = scan(c[0]), lists = scan(c[1]), before = extra0 + upto - c[0];
    const uint64_t found = __ballot(x < 0 ? at == mine : x >= before && x < before + c[0]);
    const int from = found ? __builtin_ctzll(found) : 63;
    if (found) {
      strip = first + from;
      extra0 = __shfl(before, from);
      cuts0 += __shfl(lists - c[1], from);
    } else {
      extra0 += __shfl(upto, 63);
      cuts0 += __shfl(lists, 63);
    }
  }
  if (strip < 0) return false;
  bh = strip / strips;
  const int n0 = (strip - bh * strips) * 64;
  const int n = n0 + lane < a.Nblk ? further_segments(a.count[bh * a.Nblk + n0 + lane], a.seg) : 0;
  const int upto = scan(n), lists = scan(n > 0), before = extra0 + upto - n;
  const int from = __builtin_ctzll(__ballot(x < 0 ? n0 + lane == nb : x >= before && x < before + n));
  const int e0 = min(__shfl(before, from), a.room), e1 = min(__shfl(before + n, from), a.room);
  nb = __builtin_amdgcn_readfirstlane(n0 + from);
  bh = __builtin_amdgcn_readfirstlane(bh);
  ns = __builtin_amdgcn_readfirstlane(1 + e1 - e0);
  sg = __builtin_amdgcn_readfirstlane(x < 0 ? 0 : x - e0 + 1);
  if (ns > 1) slot = __builtin_amdgcn_readfirstlane(__shfl(before + cuts0 + lists - (n > 0), from) + sg);
  return sg < ns;
}

template <typename Tag, int D, bool LINEAR>
__global__ __launch_bounds__(128) __attribute__((amdgpu_waves_per_eu(D == 64 ? 2 : 1, D == 64 ? 2 : 1))) void bwd_both_stream_kernel(
    const BwdBoth a, const LinearKeys keys, const HeadSums heads) {
  constexpr int DQ_WAVE = DQ_LDS<D> + DQ_STREAM_MAX_T * 2, DQ_ALL = D == 64 ? DQ_PAIR_LDS<D> + DQ_STREAM_MAX_T * 2 : 2 * DQ_WAVE;
  constexpr int KEYS_ALL = DKDV_LDS<D> + DKDV_STREAM_MAX_SEG * 4;
  __shared__ __attribute__((aligned(16))) uint8_t smem[DQ_ALL > KEYS_ALL ? DQ_ALL : KEYS_ALL];
  int wg = blockIdx.x;
  if (wg < a.key_wgs + a.cut_wgs) {
    const int i = wg < a.key_wgs ? xcd_remap(wg, a.key_wgs, a.nblocks) : a.nblocks + wg - a.key_wgs;
    if (i < 0) return;
    int bh, nb, sg, slot, ns;
    if (!both_item(a, i, bh, nb, sg, slot, ns)) return;
    dkdv_stream_body<Tag, D, LINEAR>(a.q, a.k, a.v, a.d_o, a.lse, a.delta, a.list, a.count, a.part, a.seg, a.dk, a.dv, a.lin, a.ldo, a.L,
                                     a.Mblk, a.Nblk, a.qk_scale, a.wide, a.add, a.done, keys, smem,
                                     reinterpret_cast<int*>(smem + DKDV_LDS<D>), bh, nb, sg, slot, ns);
    return;
  }
  wg -= a.key_wgs + a.cut_wgs;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (wg < a.head_wgs) {
    if (2 * wg + wave < heads.wgs) head_sums_body(heads, 2 * wg + wave);
    return;
  }
  wg -= a.head_wgs;
  const int wgs = (int)gridDim.x - a.key_wgs - a.cut_wgs - a.head_wgs;
  if constexpr (D == 64) {
    const int logical = xcd_remap(wg, wgs, a.total_q);
    if (logical < 0) return;
    dq_pair_body<Tag, D>(a.q, a.k, a.v, a.d_o, a.lse, a.delta, a.lut, a.lut64, a.dq, a.lin, a.ldo, a.L, a.Mblk64, a.topk, a.qk_scale,
                         a.wide, a.add, smem, reinterpret_cast<uint16_t*>(smem + DQ_PAIR_LDS<D>), logical);
  } else {
    const int pair = xcd_remap(wg, wgs, (a.total_q + 1) >> 1);
    if (pair < 0 || 2 * pair + wave >= a.total_q) return;
    uint8_t* const own = smem + wave * DQ_WAVE;
    dq_stream_body<Tag, D, false>(a.q, a.k, a.v, a.d_o, nullptr, a.lse, const_cast<float*>(a.delta), a.lut, a.lut64, a.dq, a.lin, a.ldo,
                                  a.L, a.Mblk64, a.topk, a.qk_scale, a.wide, a.add, own,
                                  reinterpret_cast<uint16_t*>(own + DQ_LDS<D>), 2 * pair + wave);
  }
}

}  // namespace sla
