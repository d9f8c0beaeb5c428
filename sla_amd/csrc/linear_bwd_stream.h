// Backward of the linear-attention branch + projection, query side: one pass over q and G = d(out).
//
// With a = phi(q), S = phi(k)^T v, z = sum phi(k), den = 1e-5 + a.z, P = S W^T (the folded state of the forward,
// core.py:90-99 of the reference) the branch is out = a P / den + b, so per query row
//   t    = G P^T                         (the only product that needs the row's G)
//   dden = -(a.t) / den^2
//   da   = t / den + dden z ;  dq = phi'(q) da
// and the sums over the rows reduce to ONE D x D matrix and two vectors:
//   M  = sum_l a_l^T G_l / den_l         ->  dS = M W,  dW = M^T S     (small products per head, formed afterwards)
//   dz = sum_l dden_l a_l ;  db = sum_l G_l
// No row-wise temporary goes to memory: q and G are read once, dq is read (when accumulating) and written once.
//
//   stream   : grid (slices of L, heads), 8 waves.  Per 128 rows: every wave takes 16 rows through t, dden, da, dq
//              (16x16x32 products, the row spread over 4 lanes), leaves the weighted rows and dq in LDS; then the workgroup
//              adds the tile's product to M (both operands read transposed from LDS), dz and db on the vector ALU, and
//              writes the dq rows whole.
//   The factor 1/den goes, with one rounding to 16 bit, to a at head dim 128 and to G at head dim 64, where a stays the 16-bit
//   value it is.  In half precision G / den leaves the format's range: a row whose phi(q) is zero (relu map, padding) has
//   den = 1e-5, and 0 times an infinite G / den is no number; small gradients over long sequences lose their bits (3 % of d_weight
//   for G of 1e-4 over 6001 rows).  There G takes a factor between 1/2 and 1 only and a the power of two that is
//   left: exact, and in range, since a_d / den <= 1 / z_d.  Both are relative to the power of two below the mean of z,
//   which the partial sums lose again: the sums' bits are those of G / den wherever that is in range.
//   finish   : fixed-order sums of the slices' partials -> M^T (fp32), dz, db per head, and from them
//              dS = M W (16 bit, both orientations) and this head's dW = M^T S (fp32)
#pragma once
#include "bwd_lists.h"
#include "linear_keys.h"
#include "linear_state.h"

namespace sla {

constexpr int LBS_TR = 128;   // rows per step of the stream kernel

// Head dim 64 keeps half the registers and 60 KB of LDS, so two workgroups share a compute unit.  Against kernels with
// row-wise temporaries (dn, y, dden) in memory, the backward of 16 heads x 6001 x 64, softmax map in half precision: rows 20.8 +
// states 16.3 + sums 14.1 + heads 5.4 + keys 21.2 us; now stream 19.8 + finish 5.8 + keys 12.8.
// Bound by the vector ALU in the row phase (30 instructions per element) with one workgroup per compute unit in step between
// barriers: 12 heads x 32760 x 128, elu map: 137 us with the floats of a row carried along (the compiler then spills what was
// fetched ahead, waiting for it) and each product waiting for its fragment, now 112.
// (At head dim 64 the compiler keeps 3 to 8 of a lane's registers in scratch, 11 with the softmax map in bf16 when accumulating.
// Half precision's two factors: forward and backward of 16 heads x 6001 x 64 188.5 -> 189.1 us, runs of one side differ by 0.3 %.)
template <typename Tag, int D, int FMAP, bool ACC>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(D == 128 ? 2 : 4, D == 128 ? 2 : 4))) void linear_bwd_stream_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ gout, const uint16_t* __restrict__ kvw,
    const uint16_t* __restrict__ z, uint16_t* __restrict__ dq, const RowLayout lin, const RowLayout ldo,
    float* __restrict__ m_part, float* __restrict__ dz_part, float* __restrict__ db_part, int L, int rows_per_split) {
  // (the feature map is a template argument: as a run-time value every element's phi sits behind its own branch; ACC: dq is
  //  added to what the tensor holds)
  using E = Elem<Tag>;
  constexpr int TR = LBS_TR;
  constexpr int TILE = TR * D * 2;               // bytes of one swizzled tile of rows
  constexpr int CPR = D / 8;                     // 16-byte pieces per row
  constexpr int RPP = 512 / CPR, NP = TR / RPP;  // rows per pass of the workgroup, passes per tile
  constexpr int NF = CPR / 4;                    // passes of a wave over its own 16 rows
  constexpr int NT = D / 16, NC = D / 32;        // 16-column tiles of a row, 32-column fragments
  constexpr bool WEIGHT_G = D == 64;             // 1 / den goes to G, not to a
  constexpr bool SPLIT = WEIGHT_G && __is_same(Tag, f16_tag);      // its power of two to a
  constexpr int PSTR = D * 2 + 16;               // row pitch of sP: 16 rows x 16 bytes of a row-wise read cover every bank
  __shared__ __attribute__((aligned(16))) char smem[3 * TILE + D * PSTR + D * 4 + D * 2 + TR * 4 + (SPLIT ? 16 : 0)];
  char* const sQ = smem;                         // raw q rows, then a (/ den) of the same rows
  char* const sG = smem + TILE;                  // G rows (then G / den)
  char* const sO = smem + 2 * TILE;              // dq rows of this step (16 bit)
  char* const sP = smem + 3 * TILE;              // folded state, P[d1][e]
  float* const sZ = reinterpret_cast<float*>(smem + 3 * TILE + D * PSTR);   // z[d1]
  uint16_t* const sZ16 = reinterpret_cast<uint16_t*>(sZ + D);               // the same, as stored
  float* const sDD = reinterpret_cast<float*>(sZ16 + D);                    // weight in dz of the row that sQ then holds
  float* const sUnit = sDD + TR;                 // SPLIT: the power of two below the mean of z
  float (*sRed)[8][D] = reinterpret_cast<float (*)[8][D]>(smem);            // final sums over the waves (over the tiles)

  const int split = blockIdx.x, bh = blockIdx.y, nsplit = gridDim.x;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int row_begin = split * rows_per_split;
  const int row_end = min(L, row_begin + rows_per_split);
  // loader layout: thread = (row lrow + RPP p, 16-byte piece lp); + 8 KiB per p in a tile
  const int lrow = tid / CPR, lp = tid % CPR;
  const uint32_t ld_off = lbs_off<D>(lrow, 8 * lp);
  // row phase: lane = (row l of the wave's 16, quarter h): d1 = 16 T + 4 h + j
  const int l = lane & 15, h = lane >> 4;

  const __amdgpu_buffer_rsrc_t q_rs = make_rsrc(q + lin.head(bh), lin.head_range_bytes(L, D));
  const __amdgpu_buffer_rsrc_t g_rs = make_rsrc(gout + ldo.head(bh), ldo.head_range_bytes(L, D));
  const __amdgpu_buffer_rsrc_t dq_rs = make_rsrc(dq + lin.head(bh), lin.head_range_bytes(L, D));
  uint16_t* const dqh = dq + lin.head(bh);
  const size_t pitch = (size_t)lin.sl;
  const uint32_t pitch_b = (uint32_t)lin.sl * 2u, pitch_gb = (uint32_t)ldo.sl * 2u;

  // (rows past L lie outside the descriptors and read as zero: phi(0) meets G = 0 there and adds nothing)
  i16x8_t rq[NP], rg[NP];
  auto fetch_qg = [&](int r0) __attribute__((always_inline)) {
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const uint32_t grow = (uint32_t)(r0 + lrow + RPP * p);
      rq[p] = buf_load_b128(q_rs, grow * pitch_b + 16 * lp);
      rg[p] = buf_load_b128(g_rs, grow * pitch_gb + 16 * lp);
    }
  };

  fetch_qg(row_begin);      // (on their way while the state is staged)
  {
    const uint16_t* src = kvw + (size_t)bh * D * D;
#pragma unroll
    for (int p = 0; p < D / RPP; ++p)
      *reinterpret_cast<i16x8_t*>(sP + (lrow + RPP * p) * PSTR + 16 * lp) =
          *reinterpret_cast<const i16x8_t*>(src + (size_t)(lrow + RPP * p) * D + 8 * lp);
    if (tid < D) {
      const uint16_t zz = z[(size_t)bh * D + tid];
      sZ[tid] = E::to_float(zz);
      sZ16[tid] = zz;
      if constexpr (SPLIT) {                     // (the D threads are one wave)
        float sum = E::to_float(zz);
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) sum += __shfl_xor(sum, o);
        if (tid == 0) *sUnit = __uint_as_float(__float_as_uint(fminf(fmaxf(sum / D, 0x1p-14f), 0x1p15f)) & 0x7f800000u);
      }
    }
    // (the first step's barrier stands before the first read of either)
  }

  // M tiles of this wave, MW x MW: rows d1 = MW mt .., columns e = MW nt0 .. and MW (nt0 + 1) .. (32x32x16 products at head dim
  // 128, 16x16x32 at 64)
  constexpr int MW = D / 4, MR = MW * MW / 64;
  typedef __attribute__((__vector_size__(MR * sizeof(float)))) float macc_t;
  const int mt = wave >> 1, nt0 = 2 * (wave & 1);
  macc_t macc[2];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int i = 0; i < MR; ++i) macc[t][i] = 0.f;
  float zacc[8], bacc[8];                        // dz and db of the loader's eight columns
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    zacc[e] = 0.f;
    bacc[e] = 0.f;
  }

  const int prow = 16 * wave + l;
  // (prow, 16 T + 4 h) in a row tile, and (prow, 32 c + 8 h), G in B-operand order: pieces of a row are exclusive-ored
  const uint32_t acc_off0 = lbs_off<D>(prow, 4 * h), g_off0 = lbs_off<D>(prow, 8 * h);
  const auto acc_off = [&](int T) __attribute__((always_inline)) { return acc_off0 ^ (uint32_t)(T * 32); };
  const auto g_off = [&](int c) __attribute__((always_inline)) { return g_off0 ^ (uint32_t)(c * 64); };
  // A operand of t^T = P G^T: row d1 = 16 T + l of sP, e = 32 c + 8 h ..: + 16 PSTR per T, + 64 bytes per c
  const char* const p_base = sP + l * PSTR + h * 16;
  // transposing reads of the M phase, KM rows per product: rows KM c + tr_row (+ 4), columns MW tile + tr_col; + 4 KiB per c
  constexpr int KM = D == 128 ? 16 : 32;
  const int g2 = lane >> 5;
  const int tr_row = 8 * (D == 128 ? g2 : h) + ((lane & 15) >> 2);
  const int tr_col = (D == 128 ? 16 * ((lane >> 4) & 1) : 0) + 4 * (lane & 3);
  uint32_t ma_off[2], mb_off[2][2];
#pragma unroll
  for (int hf = 0; hf < 2; ++hf) {
    ma_off[hf] = lbs_off<D>(tr_row + 4 * hf, MW * mt + tr_col);
#pragma unroll
    for (int t2 = 0; t2 < 2; ++t2) mb_off[hf][t2] = lbs_off<D>(tr_row + 4 * hf, MW * (nt0 + t2) + tr_col);
  }

  // dq rows leave a step late, every wave writing the 16 rows it computed (whole rows, 1 KiB per instruction), so
  // that only the wave's own order of LDS accesses matters.
  constexpr int FR = 64 / CPR;
  const int frow = 16 * wave + lane / CPR;            // + FR p
  uint32_t f_off[NF];
#pragma unroll
  for (int p = 0; p < NF; ++p) f_off[p] = lbs_off<D>(frow + FR * p, 8 * lp);
  i16x8_t rdq[NF];
  auto flush_dq = [&](int r0) __attribute__((always_inline)) {
#pragma unroll
    for (int p = 0; p < NF; ++p) {
      const int grow = r0 + frow + FR * p;
      const i16x8_t o16 = *reinterpret_cast<const i16x8_t*>(sO + f_off[p]);
      i32x4_t w = __builtin_bit_cast(i32x4_t, o16);
      if (ACC)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          w[j] = (int)E::pack2(E::to_float((uint16_t)o16[2 * j]) + E::to_float((uint16_t)rdq[p][2 * j]),
                               E::to_float((uint16_t)o16[2 * j + 1]) + E::to_float((uint16_t)rdq[p][2 * j + 1]));
      if (grow < row_end) *reinterpret_cast<i32x4_t*>(dqh + (size_t)grow * pitch + 8 * lp) = w;
    }
    wave_lds_fence();     // the row phase rewrites these rows of sO
  };

  for (int r0 = row_begin; r0 < row_end; r0 += TR) {
    // ---- tiles into LDS; db ----
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const uint32_t o = ld_off + p * 8192;
      *reinterpret_cast<i16x8_t*>(sQ + o) = rq[p];
      *reinterpret_cast<i16x8_t*>(sG + o) = rg[p];
#pragma unroll
      for (int e = 0; e < 8; ++e) bacc[e] += E::to_float((uint16_t)rg[p][e]);
    }
    lds_barrier();
    if (r0 + TR < row_end) fetch_qg(r0 + TR);
    // the previous step's dq rows leave now: what dq held was asked for a phase ago and has had time to arrive
    if (r0 > row_begin) flush_dq(r0 - TR);

    // ---- row phase ----
    {
      // (The raw rows stay packed until phi' needs them again, and what is formed from them is formed again: with the row's
      //  floats carried along, the rows fetched ahead were what the compiler spilled, and waited for.)
      i16x4_t xraw[NT];
#pragma unroll
      for (int T = 0; T < NT; ++T) xraw[T] = *reinterpret_cast<const i16x4_t*>(sQ + acc_off(T));
      i16x8_t gf[NC];
#pragma unroll
      for (int c = 0; c < NC; ++c) gf[c] = *reinterpret_cast<const i16x8_t*>(sG + g_off(c));
      __builtin_amdgcn_sched_barrier(0);
      // t^T = P G^T (tiles of 16 d1 x 16 rows) beside a = phi(q): a product's fragment is read some products ahead
      f32x4_t t[NT];
#pragma unroll
      for (int T = 0; T < NT; ++T) t[T] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int T = 0; T < NT; ++T)
          t[T] = E::mfma16(*reinterpret_cast<const i16x8_t*>(p_base + T * 16 * PSTR + c * 64), gf[c], t[T]);
      i32x2_t apk[NT];         // a = phi(q), 16 bit (it is a 16-bit tensor in the reference)
      float mx = 0.f, inv = 1.f;
      phi_quarters<Tag, FMAP, NT>(xraw, apk, mx, inv);
      constexpr int AHEAD = D == 128 ? 4 : 2;
      __builtin_amdgcn_sched_group_barrier(0x100, AHEAD, 0);
#pragma unroll
      for (int i = 0; i < NC * NT - AHEAD; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x002, FMAP == SLA_FMAP_RELU ? 4 : 10, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      }
      __builtin_amdgcn_sched_group_barrier(0x008, AHEAD, 0);
      __builtin_amdgcn_sched_barrier(0);
      // den: z as an A operand with sixteen equal rows, the summed index in the order a row's four lanes hold a
      i16x8_t zf[NC];
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const uint16_t* zp = sZ16 + 32 * c + 4 * h;
        zf[c] = concat4(*reinterpret_cast<const i16x4_t*>(zp), *reinterpret_cast<const i16x4_t*>(zp + 16));
      }
      f32x4_t dsum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const i32x4_t w = {apk[2 * c][0], apk[2 * c][1], apk[2 * c + 1][0], apk[2 * c + 1][1]};
        dsum = E::mfma16(zf[c], __builtin_bit_cast(i16x8_t, w), dsum);
      }
      float s = 0.f;
#pragma unroll
      for (int T = 0; T < NT; ++T)
#pragma unroll
        for (int j = 0; j < 4; ++j) s += unpack_quarter<Tag>(apk[T], j) * t[T][j];
      __builtin_amdgcn_sched_group_barrier(0x100, 2 * NC, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, NC, 0);
      __builtin_amdgcn_sched_barrier(0);
      const float inv_den = 1.0f / (dsum[0] + 1e-5f);
      s = sum_quarters(s);
      const float dden = -s * inv_den * inv_den;
      // SPLIT: unit / den = weight_g * p1 * p2 with powers of two that half precision holds, weight_g in [1/2, 1).  (A row whose
      // den is below unit / 2^30 counts with that weight.)
      float weight_g = inv_den, p1 = 1.f, p2 = 1.f, inv_p = 1.f;
      if constexpr (SPLIT) {
        const auto inverse = [](float p) __attribute__((always_inline)) { return __uint_as_float(0x7f000000u - __float_as_uint(p)); };
        const float x = *sUnit * inv_den;
        const float p = __uint_as_float((__float_as_uint(x) & 0x7f800000u) + 0x00800000u);
        p1 = fminf(fmaxf(p, 0x1p-14f), 0x1p15f);
        p2 = fminf(fmaxf(p * inverse(p1), 0x1p-14f), 0x1p15f);
        inv_p = inverse(p1) * inverse(p2);
        weight_g = p > 0x1p30f ? 1.f : x * inv_p;
      }
      // the weight of what sQ holds (a, a p1 p2 or a/den) in dz
      if (h == 0) sDD[prow] = SPLIT ? dden * inv_p : WEIGHT_G ? dden : -s * inv_den;
      f32x4_t zz[NT];
      const auto fetch_z = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int T = 0; T < NT; ++T) zz[T] = *reinterpret_cast<const f32x4_t*>(sZ + 16 * T + 4 * h);
        __builtin_amdgcn_sched_barrier(0);
      };
      if (!SPLIT) fetch_z();
      // a (with its power of two) or a/den takes the place of the raw row, G/den (its other factor) that of G (this lane's own places)
#pragma unroll
      for (int T = 0; T < NT; ++T) {
        i32x2_t w = apk[T];
        if (!WEIGHT_G)
#pragma unroll
          for (int j2 = 0; j2 < 2; ++j2)
            w[j2] = (int)E::pack2(unpack_quarter<Tag>(apk[T], 2 * j2) * inv_den, unpack_quarter<Tag>(apk[T], 2 * j2 + 1) * inv_den);
        if constexpr (SPLIT) {
          // (finite where a is: only a component in which no key has weight passes the format's largest number, and what it adds
          //  to the sums meets zeros.  a is not negative, so the patterns are in the values' order.)
          typedef unsigned short u16x2_t __attribute__((ext_vector_type(2)));
          const f16x2_t h1 = {(_Float16)p1, (_Float16)p1}, h2 = {(_Float16)p2, (_Float16)p2};
#pragma unroll
          for (int j2 = 0; j2 < 2; ++j2) {
            const int a2 = apk[T][j2];
            const u16x2_t most = __builtin_elementwise_max(__builtin_bit_cast(u16x2_t, a2), u16x2_t{0x7bff, 0x7bff});
            const f16x2_t y = __builtin_bit_cast(f16x2_t, a2) * h1 * h2;
            w[j2] = __builtin_bit_cast(int, __builtin_elementwise_min(__builtin_bit_cast(u16x2_t, y), most));
          }
        }
        *reinterpret_cast<i32x2_t*>(sQ + acc_off(T)) = w;
      }
      if (WEIGHT_G)
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          const i16x8_t gr = *reinterpret_cast<const i16x8_t*>(sG + g_off(c));
          i32x4_t w;
#pragma unroll
          for (int j = 0; j < 4; ++j)
            w[j] = (int)E::pack2(E::to_float((uint16_t)gr[2 * j]) * weight_g, E::to_float((uint16_t)gr[2 * j + 1]) * weight_g);
          *reinterpret_cast<i32x4_t*>(sG + g_off(c)) = w;
        }
      if (SPLIT) fetch_z();
      // da = t / den + dden z (in place), then dq = phi'(q) da
#pragma unroll
      for (int T = 0; T < NT; ++T)
#pragma unroll
        for (int j = 0; j < 4; ++j) t[T][j] = __builtin_fmaf(t[T][j], inv_den, dden * zz[T][j]);
      forget_floats<NT>(xraw);
      phi_quarters_backward<Tag, FMAP, NT>(xraw, mx, inv, t);
#pragma unroll
      for (int T = 0; T < NT; ++T) {
        i32x2_t w;
        w[0] = (int)E::pack2(t[T][0], t[T][1]);
        w[1] = (int)E::pack2(t[T][2], t[T][3]);
        *reinterpret_cast<i32x2_t*>(sO + acc_off(T)) = w;
      }
    }
    lds_barrier();

    // ---- M += a^T G / den ----
    // (what dq holds so far is asked for here, where the row phase's registers are free, and used in the next step)
    if (ACC)
#pragma unroll
    for (int p = 0; p < NF; ++p) rdq[p] = buf_load_b128(dq_rs, (uint32_t)(r0 + frow + FR * p) * pitch_b + 16 * lp);
    __builtin_amdgcn_sched_barrier(0);      // (asked for first: the loop's next wait on memory covers these too)
#pragma unroll
    for (int c = 0; c < TR / KM; ++c) {
      const uint16_t* pa0 = reinterpret_cast<const uint16_t*>(sQ + ma_off[0] + c * 4096);
      const uint16_t* pa1 = reinterpret_cast<const uint16_t*>(sQ + ma_off[1] + c * 4096);
      const i16x8_t af = concat4(lds_read_tr16(pa0), lds_read_tr16(pa1));
#pragma unroll
      for (int t2 = 0; t2 < 2; ++t2) {
        const uint16_t* pb0 = reinterpret_cast<const uint16_t*>(sG + mb_off[0][t2] + c * 4096);
        const uint16_t* pb1 = reinterpret_cast<const uint16_t*>(sG + mb_off[1][t2] + c * 4096);
        const i16x8_t bf = concat4(lds_read_tr16(pb0), lds_read_tr16(pb1));
        if constexpr (D == 128) macc[t2] = E::mfma32(af, bf, macc[t2]);
        else macc[t2] = E::mfma16(af, bf, macc[t2]);
      }
    }
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const i16x8_t an = *reinterpret_cast<const i16x8_t*>(sQ + ld_off + p * 8192);
      const float dd = sDD[lrow + RPP * p];
#pragma unroll
      for (int e = 0; e < 8; ++e) zacc[e] = __builtin_fmaf(dd, E::to_float((uint16_t)an[e]), zacc[e]);
    }
    lds_barrier();
  }
  flush_dq(row_begin + (row_end - 1 - row_begin) / TR * TR);

  // M^T partial [e][d1] (accumulator rows = d1, columns = e), fp32
  const float unscale = SPLIT ? 1.f / *sUnit : 1.f;
  const size_t pidx = (size_t)bh * nsplit + split;
  float* mo = m_part + pidx * D * D;
#pragma unroll
  for (int t2 = 0; t2 < 2; ++t2) {
    const int col = MW * (nt0 + t2) + (lane & (MW - 1));
#pragma unroll
    for (int i4 = 0; i4 < MR / 4; ++i4) {
      f32x4_t v4 = {macc[t2][4 * i4], macc[t2][4 * i4 + 1], macc[t2][4 * i4 + 2], macc[t2][4 * i4 + 3]};
      if (SPLIT) v4 *= unscale;
      *reinterpret_cast<f32x4_t*>(mo + (size_t)col * D + MW * mt + 8 * i4 + 4 * (D == 128 ? g2 : h)) = v4;
    }
  }
  lds_barrier();           // (the last dq rows have left sO)
  // the lanes of a wave that hold the same columns; then the waves
#pragma unroll
  for (int which = 0; which < 2; ++which) {
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      v[e] = which ? bacc[e] : zacc[e];
      if (CPR == 8)          // lane ^ 8
        v[e] += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v[e]), 0x128, 0xf, 0xf, true));
      v[e] = sum_quarters(v[e]);
    }
    if (lane < CPR)
#pragma unroll
      for (int x = 0; x < 2; ++x)
        *reinterpret_cast<f32x4_t*>(&sRed[which][wave][8 * lp + 4 * x]) = f32x4_t{v[4 * x], v[4 * x + 1], v[4 * x + 2], v[4 * x + 3]};
  }
  lds_barrier();
  if (tid < 2 * D) {
    const int which = tid / D, col = tid % D;
    float sum = 0.f;
#pragma unroll
    for (int w = 0; w < 8; ++w) sum += sRed[which][w][col];
    (which ? db_part : dz_part)[pidx * D + col] = sum;
  }
}

// Key side of the same backward: dv = c dS, dc = v dS^T + dz, dk = phi'(k) dc with c = phi(k).
// grid (slices of L, heads), 8 waves; dS [d1][d2] and dS^T [d2][d1] (16 bit, rows padded by 16 bytes) and dz stay in LDS,
// every wave walks its own 16-key tiles of the slice and never meets another wave after the staging barrier:
//   rows of k, v (fetched a tile ahead) -> two wave-private swizzled tiles; phi(k) takes the place of k;
//   dv^T = dS^T c^T and dc^T = dS v^T as 16x16x32 products (a key's row spread over 4 lanes, B operands read row-wise
//   from the wave's tiles); dk, dv go back over the tiles and leave as whole rows, added to what dk, dv held (asked
//   for at the start of the tile) when accumulating.
// The arithmetic is that of KeyTiles (linear_keys.h), which the attention's dK/dV kernel uses in launches with few key blocks: the same
// products, sums and roundings in the same order, to be kept so.
template <typename Tag, int D, int FMAP, bool ACC>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(D == 128 ? 2 : 4, D == 128 ? 2 : 4))) void linear_bwd_keys_kernel(
    const uint16_t* __restrict__ k, const uint16_t* __restrict__ v, const uint16_t* __restrict__ ds,
    const uint16_t* __restrict__ dst, const float* __restrict__ dz, uint16_t* __restrict__ dk, uint16_t* __restrict__ dv,
    const RowLayout lin, int L, int rows_per_split) {
  using E = Elem<Tag>;
  constexpr int CPR = D / 8;                     // 16-byte pieces per row
  constexpr int NF = CPR / 4, FR = 64 / CPR;     // passes over a wave's 16 rows, rows per pass
  constexpr int NT = D / 16, NC = D / 32;        // 16-column tiles of a row, 32-column fragments
  constexpr int PSTR = D * 2 + 16;               // row pitch of the staged matrices
  constexpr int WT = 16 * D * 2;                 // bytes of a wave's tile
  __shared__ __attribute__((aligned(16))) char smem[2 * D * PSTR + D * 4 + 8 * 2 * WT];
  char* const sDS = smem;                        // dS   [d1][d2]: A operand of dc^T = dS v^T
  char* const sDST = smem + D * PSTR;            // dS^T [d2][d1]: A operand of dv^T = dS^T c^T
  float* const sDZ = reinterpret_cast<float*>(smem + 2 * D * PSTR);

  const int split = blockIdx.x, bh = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  char* const tK = smem + 2 * D * PSTR + D * 4 + wave * 2 * WT;    // k rows, then phi(k), then dk
  char* const tV = tK + WT;                                          // v rows, then dv
  const int row_begin = split * rows_per_split;
  const int row_end = min(L, row_begin + rows_per_split);
  {
    const uint16_t* s0 = ds + (size_t)bh * D * D;
    const uint16_t* s1 = dst + (size_t)bh * D * D;
    for (int idx = tid; idx < D * D / 8; idx += 512) {
      const int row = idx / (D / 8), col = (idx % (D / 8)) * 8;
      *reinterpret_cast<i16x8_t*>(sDS + row * PSTR + col * 2) = *reinterpret_cast<const i16x8_t*>(s0 + (size_t)row * D + col);
      *reinterpret_cast<i16x8_t*>(sDST + row * PSTR + col * 2) = *reinterpret_cast<const i16x8_t*>(s1 + (size_t)row * D + col);
    }
    if (tid < D) sDZ[tid] = dz[(size_t)bh * D + tid];
  }
  lds_barrier();

  const uint32_t range = lin.head_range_bytes(L, D);
  const __amdgpu_buffer_rsrc_t k_rs = make_rsrc(k + lin.head(bh), range);
  const __amdgpu_buffer_rsrc_t v_rs = make_rsrc(v + lin.head(bh), range);
  const __amdgpu_buffer_rsrc_t dk_rs = make_rsrc(dk + lin.head(bh), range);
  const __amdgpu_buffer_rsrc_t dv_rs = make_rsrc(dv + lin.head(bh), range);
  uint16_t* const dkh = dk + lin.head(bh);
  uint16_t* const dvh = dv + lin.head(bh);
  const size_t pitch = (size_t)lin.sl;
  const uint32_t pitch_b = (uint32_t)lin.sl * 2u;

  // loader / writer layout of a wave's tile: lane -> row lane / CPR + FR p, 16-byte piece lane % CPR
  const int frow = lane / CPR, lp = lane % CPR;
  uint32_t f_off[NF];
#pragma unroll
  for (int p = 0; p < NF; ++p) f_off[p] = lbs_off<D>(frow + FR * p, 8 * lp);
  // product layout: lane = (key l of the tile's 16, quarter h): d = 16 T + 4 h + j
  const int l = lane & 15, h = lane >> 4;
  uint32_t acc_off[NT];        // (l, 16 T + 4 h)
#pragma unroll
  for (int T = 0; T < NT; ++T) acc_off[T] = lbs_off<D>(l, 16 * T + 4 * h);
  uint32_t b_off[NC];          // (l, 32 c + 8 h): B-operand order
#pragma unroll
  for (int c = 0; c < NC; ++c) b_off[c] = lbs_off<D>(l, 32 * c + 8 * h);
  const uint32_t a_base = (uint32_t)l * PSTR + (uint32_t)h * 16u;     // row 16 T + l of a staged matrix: + 16 PSTR per T, + 64 per c

  i16x8_t rk[NF], rv[NF];
  auto fetch_kv = [&](int r0) __attribute__((always_inline)) {
#pragma unroll
    for (int p = 0; p < NF; ++p) {
      const uint32_t o = (uint32_t)(r0 + frow + FR * p) * pitch_b + 16 * lp;      // rows past L read as zero
      rk[p] = buf_load_b128(k_rs, o);
      rv[p] = buf_load_b128(v_rs, o);
    }
  };
  const int first = row_begin + 16 * wave;
  if (first < row_end) fetch_kv(first);
  for (int r0 = first; r0 < row_end; r0 += 128) {
#pragma unroll
    for (int p = 0; p < NF; ++p) {
      *reinterpret_cast<i16x8_t*>(tK + f_off[p]) = rk[p];
      *reinterpret_cast<i16x8_t*>(tV + f_off[p]) = rv[p];
    }
    wave_lds_fence();
    // what dk, dv hold (for this tile) and the next tile's rows: both have the whole tile to arrive
    i16x8_t rdk[NF], rdv[NF];
    if (ACC)
#pragma unroll
    for (int p = 0; p < NF; ++p) {
      const uint32_t o = (uint32_t)(r0 + frow + FR * p) * pitch_b + 16 * lp;
      rdk[p] = buf_load_b128(dk_rs, o);
      rdv[p] = buf_load_b128(dv_rs, o);
    }
    if (r0 + 128 < row_end) fetch_kv(r0 + 128);

    i16x4_t xraw[NT];
#pragma unroll
    for (int T = 0; T < NT; ++T) xraw[T] = *reinterpret_cast<const i16x4_t*>(tK + acc_off[T]);
    i32x2_t apk[NT];
    float mx = 0.f, inv = 1.f;
    phi_quarters<Tag, FMAP, NT>(xraw, apk, mx, inv);
    // c = phi(k) over the raw rows (this lane's own places; a key's gradients depend on its own row only, so rows
    // past the end, which are never written, need no care)
#pragma unroll
    for (int T = 0; T < NT; ++T) *reinterpret_cast<i32x2_t*>(tK + acc_off[T]) = apk[T];
    wave_lds_fence();
    // dv^T = dS^T c^T ; dc^T = dS v^T
    f32x4_t dva[NT], dca[NT];
#pragma unroll
    for (int T = 0; T < NT; ++T) {
      dva[T] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      dca[T] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const i16x8_t cf = *reinterpret_cast<const i16x8_t*>(tK + b_off[c]);
      const i16x8_t vf = *reinterpret_cast<const i16x8_t*>(tV + b_off[c]);
#pragma unroll
      for (int T = 0; T < NT; ++T) {
        dva[T] = E::mfma16(*reinterpret_cast<const i16x8_t*>(sDST + a_base + T * 16 * PSTR + c * 64), cf, dva[T]);
        dca[T] = E::mfma16(*reinterpret_cast<const i16x8_t*>(sDS + a_base + T * 16 * PSTR + c * 64), vf, dca[T]);
      }
    }
    wave_lds_fence();      // (the tiles are rewritten below: every read of them above comes first)
    // dc += dz ; dk = phi'(k) dc
#pragma unroll
    for (int T = 0; T < NT; ++T) {
      const f32x4_t zz = *reinterpret_cast<const f32x4_t*>(sDZ + 16 * T + 4 * h);
#pragma unroll
      for (int j = 0; j < 4; ++j) dca[T][j] += zz[j];
    }
    phi_quarters_backward<Tag, FMAP, NT>(xraw, mx, inv, dca);
#pragma unroll
    for (int T = 0; T < NT; ++T) {
      i32x2_t wk, wv;
      wk[0] = (int)E::pack2(dca[T][0], dca[T][1]);
      wk[1] = (int)E::pack2(dca[T][2], dca[T][3]);
      wv[0] = (int)E::pack2(dva[T][0], dva[T][1]);
      wv[1] = (int)E::pack2(dva[T][2], dva[T][3]);
      *reinterpret_cast<i32x2_t*>(tK + acc_off[T]) = wk;
      *reinterpret_cast<i32x2_t*>(tV + acc_off[T]) = wv;
    }
    wave_lds_fence();
    // whole rows out; ACC: 16-bit value + what the tensor held, one rounded add
#pragma unroll
    for (int p = 0; p < NF; ++p) {
      const int grow = r0 + frow + FR * p;
      const i16x8_t k16 = *reinterpret_cast<const i16x8_t*>(tK + f_off[p]);
      const i16x8_t v16 = *reinterpret_cast<const i16x8_t*>(tV + f_off[p]);
      i32x4_t wk = __builtin_bit_cast(i32x4_t, k16), wv = __builtin_bit_cast(i32x4_t, v16);
      if (ACC)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        wk[j] = (int)E::pack2(E::to_float((uint16_t)k16[2 * j]) + E::to_float((uint16_t)rdk[p][2 * j]),
                              E::to_float((uint16_t)k16[2 * j + 1]) + E::to_float((uint16_t)rdk[p][2 * j + 1]));
        wv[j] = (int)E::pack2(E::to_float((uint16_t)v16[2 * j]) + E::to_float((uint16_t)rdv[p][2 * j]),
                              E::to_float((uint16_t)v16[2 * j + 1]) + E::to_float((uint16_t)rdv[p][2 * j + 1]));
      }
      if (grow < row_end) {
        *reinterpret_cast<i32x4_t*>(dkh + (size_t)grow * pitch + 8 * lp) = wk;
        *reinterpret_cast<i32x4_t*>(dvh + (size_t)grow * pitch + 8 * lp) = wv;
      }
    }
    wave_lds_fence();      // the next tile's rows go over these
  }
}

// From the slices' partials of a head (fp32, [e][d1]), added in ascending slice order to M^T, dz, db:
//   dS[d1][d2]    = sum_e  M^T[e][d1] * round16(W[e][d2])    -> ds [d1][d2] and dst [d2][d1], 16 bit
//   dW^T[d2][e]   = sum_d1 M[d1][e] * S[d1][d2]              -> dw_head [d2][e], fp32  (S^T = kvt[d2][d1], 16 bit)
// M stays in fp32 and meets the other factor on the fp32 matrix product (16x16x4).  One workgroup per head, sixteen indices
// and kind (neighbouring workgroups on one XCD):
//   kind 0: sums the columns d1 = i0 .. + 15 of every row e and forms 16 rows of dS;
//   kind 1: sums the rows e = i0 .. + 15 and forms 16 columns of dW^T.
// Either way it holds all its products need of M after one hand-over through LDS; the partials are read twice, from the
// caches.  The slices are summed in two halves side by side, whose sums are then added, eight slices' loads in flight.
// Against a kernel for the sums and one for the products (on the vector ALU, M through memory in both orientations): 9.3
// against 12.8 + 10.5 us (B2 H4 L4096).  With many slices of few heads linear_state_presum_kernel has added them up before (the same
// bits): 1 head x 75600 x 128 (197 slices) 45.9 us without it, 6.1 + 21.4 with it, the latter the lists' time; 2 heads x 20000 x 128 (79)
// 21.7 and 4.8 + 8.6.  Forward and backward: 1 x 75600 x 128 930 -> 916 us, 4 x 40000 x 64 556 -> 546, 2 x 20000 x 128 382 -> 372, 1 x 8000
// x 128 (63) 227 -> 217, 12 x 20000 x 64 (42) 461 -> 457.  The first `first_wg` workgroups, a multiple of eight, build the lists of the map for
// the attention backward: both are short and bound by latency.
template <typename Tag, int D>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(4))) void linear_bwd_finish_kernel(
    const float* __restrict__ m_part, const float* __restrict__ dz_part, const float* __restrict__ db_part,
    const float* __restrict__ weight, const uint16_t* __restrict__ kvt, uint16_t* __restrict__ ds, uint16_t* __restrict__ dst,
    float* __restrict__ dz, float* __restrict__ dw_head, float* __restrict__ db_head, int nsplit, int nsum, int total,
    int first_wg, const ColLists lists) {
  // (nsum: the slices to add up, all nsplit of a head or the first one alone, which then holds the sums)
  using E = Elem<Tag>;
  constexpr int DD = D * D;
  constexpr int NR = D / 64;               // f32x4 sums per thread
  constexpr int KQ = D / 4;                // products per tile: four summed indices each
  constexpr int EP = D + 1;                // row pitch of the strip of rows
  constexpr int S_HALF = NR * 256 * 4;
  constexpr int LDS = 4 * (S_HALF + 16 * EP) > COL_LDS ? 4 * (S_HALF + 16 * EP) : COL_LDS;
  __shared__ __attribute__((aligned(16))) char smem[LDS];
  float* const s_half = reinterpret_cast<float*>(smem);
  float* const sm = s_half + S_HALF;
  if ((int)blockIdx.x < first_wg) {
    if ((int)blockIdx.x < lists.wgs) col_lists_body(lists, blockIdx.x, smem);
    return;
  }
  const int logical = xcd_remap((int)blockIdx.x - first_wg, (int)gridDim.x - first_wg, total);
  if (logical < 0) return;
  const int bh = logical / (D / 8), rest = logical % (D / 8), kind = rest / (D / 16), i0 = 16 * (rest % (D / 16));
  const int tid = threadIdx.x & 255, half = threadIdx.x >> 8, lane = tid & 63, wave = threadIdx.x >> 6;
  const int l = lane & 15, h = lane >> 4;
  const int n0 = (nsum + 1) >> 1;
  const float* mp = m_part + (size_t)bh * nsplit * DD;
  const int er = kind == 0 ? tid >> 2 : tid >> 4, dc = kind == 0 ? 4 * (tid & 3) : 4 * (tid & 15);
  mp += kind == 0 ? (size_t)er * D + i0 + dc : (size_t)(i0 + er) * D + dc;
  const size_t vec = kind == 0 ? (size_t)64 * D : 64;
  f32x4_t acc[NR];
#pragma unroll
  for (int i = 0; i < NR; ++i) acc[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  sum_slices<NR>(mp + (half ? (size_t)n0 * DD : 0), half ? nsum - n0 : n0, DD, vec, acc);
  if (half)
#pragma unroll
    for (int i = 0; i < NR; ++i) *reinterpret_cast<f32x4_t*>(s_half + (i * 256 + tid) * 4) = acc[i];
  if (kind == 0 && half && tid < 32) {
    const float* q = (tid < 16 ? dz_part : db_part) + (size_t)bh * nsplit * D + i0 + (tid & 15);
    float sum = 0.f;
#pragma unroll 8
    for (int sp = 0; sp < nsum; ++sp) sum += q[(size_t)sp * D];
    (tid < 16 ? dz : db_head)[(size_t)bh * D + i0 + (tid & 15)] = sum;
  }
  __syncthreads();
  if (!half)
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      acc[i] += *reinterpret_cast<const f32x4_t*>(s_half + (i * 256 + tid) * 4);
      if (kind == 0) {
        *reinterpret_cast<f32x4_t*>(sm + (er + 64 * i) * 16 + dc) = acc[i];                    // [e][d1]
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) sm[er * EP + dc + 64 * i + j] = acc[i][j];                 // [e][d1]
      }
    }
  __syncthreads();
  const int tile = wave;                   // 16 wide; head dim 64: four of the eight waves
  if (tile >= D / 16) return;
  f32x4_t o = {0.f, 0.f, 0.f, 0.f};
  if (kind == 0) {
    // row d1 = l of M, column d2 = 16 tile + l of W; summed index e = 4 kk + h
    const int d2 = 16 * tile + l;
#pragma unroll
    for (int k0 = 0; k0 < KQ; k0 += 16) {
      float wb[16];
#pragma unroll
      for (int x = 0; x < 16; ++x) wb[x] = weight[(size_t)(4 * (k0 + x) + h) * D + d2];
#pragma unroll
      for (int x = 0; x < 16; ++x)
        o = __builtin_amdgcn_mfma_f32_16x16x4f32(sm[(4 * (k0 + x) + h) * 16 + l], round16<Tag>(wb[x]), o, 0, 0, 0);
    }
    // rows d1 = 4 h + i, column d2
    i32x2_t w;
    w[0] = (int)E::pack2(o[0], o[1]);
    w[1] = (int)E::pack2(o[2], o[3]);
    *reinterpret_cast<i32x2_t*>(dst + (size_t)bh * DD + (size_t)d2 * D + i0 + 4 * h) = w;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      ds[(size_t)bh * DD + (size_t)(i0 + 4 * h + i) * D + d2] = (uint16_t)((uint32_t)w[i >> 1] >> (16 * (i & 1)));
  } else {
    // row d2 = 16 tile + l of S^T, column e = l of M; summed index d1 = KQ h + kk (adjacent per lane)
    const uint16_t* st = kvt + (size_t)bh * DD + (size_t)(16 * tile + l) * D + KQ * h;
#pragma unroll
    for (int c = 0; c < KQ / 8; ++c) {
      const i16x8_t sf = *reinterpret_cast<const i16x8_t*>(st + 8 * c);
#pragma unroll
      for (int j = 0; j < 8; ++j)
        o = __builtin_amdgcn_mfma_f32_16x16x4f32(E::to_float((uint16_t)sf[j]), sm[l * EP + KQ * h + 8 * c + j], o, 0, 0, 0);
    }
    // rows d2 = 16 tile + 4 h + i, column e: the layout head_sums_body adds up
#pragma unroll
    for (int i = 0; i < 4; ++i) dw_head[(size_t)bh * DD + (size_t)(16 * tile + 4 * h + i) * D + i0 + l] = o[i];
  }
}

}  // namespace sla
