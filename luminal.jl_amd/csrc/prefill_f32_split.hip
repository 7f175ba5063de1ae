// Flash attention forward in fp32 on the 16-bit matrix pipe: every operand as pieces of 16 bits, three or six products for one.
//
// Up to head dim 96 every operand is split into three bf16 pieces (split.hpp); of the nine products of pieces the six with x_i y_j, i + j <= 4, are
// summed in fp32, the other three are below 2^-25 of x y. Six bf16 products take 6 / 16 of the time of the fp32 one. Error against
// 64 bits (2-norm): 1.9e-7 where the forms of prefill_f32.hip have 4.3e-7 (S = 1023 D = 80), 1.3e-7 and 2.7e-7 (S = 500 D = 96 causal).
// The pieces of V and of the weights are scaled, so that a result that is left to a small value or to small weights has all its
// bits (not through the exponent of the weights, which is rounded at its own magnitude: 2^-21 of a weight at 24). Q and K come as
// they are: what counts of a score is its absolute error, and the bits that their pieces lose lie below 2^-126. A workgroup that
// meets an infinity, a NaN, queries or keys so large that those bits would count, or an overflow takes its rows again with the fp32
// product, straight from memory: a launch all of whose workgroups do takes about five times as long (S = 1023 D = 80, 62 and 297 us).
//
// Same data flow as prefill_mfma.hip: a wave owns 32 query rows with the pieces of its Q fragments in registers, S^T = K Q^T so
// that a lane holds one query column, and the registers of P, split there, are the B operands of O^T = V^T P^T. Statistics, sums
// and accumulators are fp32 as in prefill_f32.hip. K and V tiles of 64 keys pass through registers: fetched as fp32 while the tile
// before is multiplied, split once per workgroup and stored as three planes each.
// Bound: the bf16 matrix pipe at the clock it gets, then the vector ALUs beside it. S = 1023 D = 80, 57 us: 36 with two of the six
// products, 52 without splitting K and V, 57 without splitting P (measurement variants).
//
// Head dims above 96 (HALF): three bf16 pieces of Q and K, with 160 bytes a lane in memory beside the registers of two waves per SIMD, are as fast as
// the fp32 product (B=1 H=16 S=2048 D=128 causal 178 us). Q and K are two fp16 pieces there, 22 to 24 bits: three products for one in S^T, hi lo and lo hi in
// accumulators of their own, lo lo left out (Ootomo and Yokota, "Recovering single precision accuracy from Tensor Cores while surpassing the FP32 theoretical
// peak performance", 2022), and two planes of K instead of three. The gain is half the products of S^T and a plane less; the causal kernel keeps 128 bytes in
// memory still, 48 of them V's on its way through the loop, the one without a mask none. What is lost weighs less than what the fp32 product
// rounds (2-norm against 64 bits, that product and this kernel): 4.6e-7 and 1.7e-7 (S = 2048 D = 128 causal), 5.7e-7 and 2.0e-7 (S = 1024),
// 5.6e-7 and 2.0e-7 (S = 1023 D = 112). Below it, against three bf16 pieces, it would weigh 0.05 to 0.2 more than nothing (S = 1023 D = 80
// 1.83e-7 and 1.90e-7, S = 2048 D = 64 causal 1.35e-7 and 1.52e-7), so these stay. The pieces are taken relative to a power of two, each query's
// own and that of the largest key so far, so what they lack is small beside what is there at any magnitude (S = 1024 causal, queries of 1e3 and keys of 1e-5:
// 1.6e-7 with the fp32 product, 0.7e-7; 3e3 and 1: 2.7e-5 and 1.1e-5). What still goes to the fp32 product: infinities and NaN, scores beyond 2^30, and walks whose
// largest key leaves so little of the others that bits of their scores would be lost (from about 2^20 on). That takes three times as long as
// the fp32 product's own kernel (S = 4096 1070 and 3370 us, B=8 H=16 S=300 47 and 159); until the pieces were relative, values of 1e3 took it too,
// and normal ones up to 2 % less. us, the fp32 product and this kernel: B=1 H=32/8 S=4096 D=128 causal 1068 and 591, H=16 S=2048 177 and 128,
// B=2 H=12 S=1023 D=112 115 and 69, B=8 H=16 S=300 D=128 causal 46.9 and 35.2. One tile of 64 keys
// is in LDS at a time; with K's next one beside it, and both split beside the MFMAs, the first two took 594 and 132 us, in another order 634 and 133.
#include <math.h>

#include <algorithm>
#include <type_traits>

#include "prefill_mfma.hpp"
#include "rope.hpp"
#include "split.hpp"

namespace lmh {
namespace {

constexpr float kLog2eRest = 1.9259629911e-8f;  // log2(e) - kLog2e

// NW waves: RW = NW / KSPLIT groups of 32 rows; KSPLIT = 2: half of the waves take the second 32 keys of every tile, folded
// through LDS at the end.
template <int D, bool CAUSAL, int NW, int KSPLIT>
__global__ __launch_bounds__(64 * NW, 2) void prefill_f32_split_kernel(Deal deal, PrefillArgs a) {
  request_args(a);
  request_args(deal);
  constexpr int RW = NW / KSPLIT, BM = 32 * RW, NT = 64 * NW;
  constexpr int BT = 64;                   // keys per tile
  constexpr int NKB = 2 / KSPLIT;          // 32-key blocks a wave takes of it
  constexpr bool HALF = D > 96;            // Q and K as two fp16 pieces
  constexpr int KS = D / 16;               // k-steps of the S^T product
  constexpr int DB = (D + 31) / 32;        // 32-row blocks of O^T
  constexpr int LDK = D + kPadK, LDV = 32 * DB + pad_v<32 * DB>();
  constexpr int kPlaneK = BT * LDK, kPlaneV = BT * LDV;
  constexpr int DC = D / 8, kChunks = 2 * BT * DC, R = (kChunks + NT - 1) / NT;  // chunks of eight elements, K's then V's
  // Two tiles where they fit (tile kt + 1 is split beside the MFMAs of tile kt, one barrier a tile), or one.
  constexpr int kPlanesK = HALF ? 2 : 3, kTile = kPlanesK * kPlaneK + 3 * kPlaneV;
  constexpr int NBUF = 4 * kTile <= 160 * 1024 && NW == 8 ? 2 : 1;
  __shared__ __attribute__((aligned(16))) uint16_t planes[NBUF * kTile];
  __shared__ int redo;
  __shared__ int key_top;  // HALF: exponent of the largest key so far

  int bh, tile_rank;
  if (!deal_tile(deal, blockIdx.x & 7, blockIdx.x >> 3, &bh, &tile_rank)) return;
  const int b = (int)((uint32_t)bh / deal.hq), hq = bh - b * a.Hq;
  const int kvh = kv_head_of(hq, a.Hq, a.Hkv, a.head_map);
  const int q_tile = CAUSAL ? (deal.tiles - 1 - tile_rank) : tile_rank;
  const int q0 = q_tile * BM - (CAUSAL ? causal_shift(deal.tiles, BM, a.Sq, BT) : 0);

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 31, g = lane >> 5;
  const int kg = wave / RW;
  const int wave_q_lo = q0 + (wave % RW) * 32, wave_q_hi = wave_q_lo + 31;
  const int qi = wave_q_lo + n;

  int n_keys = a.kv_len ? a.kv_len[b] : a.Sk;
  n_keys = min(max(n_keys, 0), a.Sk);
  int k_end = n_keys;
  if (CAUSAL) k_end = min(k_end, q0 + BM);
  const int n_kv_tiles = (k_end + BT - 1) / BT;

  const float *qp = reinterpret_cast<const float *>(a.q) + b * a.qs[0] + hq * a.qs[1];
  const float *kp = reinterpret_cast<const float *>(a.k) + b * a.ks[0] + kvh * a.ks[1];
  const float *vp = reinterpret_cast<const float *>(a.v) + b * a.vs[0] + kvh * a.vs[1];

  // ---- tile staging; columns past the tensors' own head dim and rows past n_keys arrive as zeros ----
  auto make_rsrc = [](const float *p, int64_t elements) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(p), 0, __builtin_amdgcn_readfirstlane((int)(elements * 4)), 0x00020000);
  };
  const __amdgpu_buffer_rsrc_t k_rsrc = make_rsrc(kp, (int64_t)n_keys * a.ks[2]);
  const __amdgpu_buffer_rsrc_t v_rsrc = make_rsrc(vp, (int64_t)n_keys * a.vs[2]);
  const int k_tile_bytes = (int)(BT * a.ks[2] * 4), v_tile_bytes = (int)(BT * a.vs[2] * 4);
  // Rounds of whole rows (HALF): one offset a tensor, and what a round adds is the same for every lane.
  constexpr int kRoundRows = HALF ? NT / DC : 0, kRoundsK = HALF ? BT / (NT / DC) : 0;
  static_assert(!HALF || (NT % DC == 0 && BT % (NT / DC) == 0), "whole rows a round");
  auto round_bytes = [&](int r, int64_t stride) { return (uint32_t)min((int64_t)r * kRoundRows * stride * 4, (int64_t)kOutOfRange); };
  int voff[HALF ? 2 : R], lds_off[HALF ? 2 : R];
#pragma unroll
  for (int r = 0; r < (HALF ? 2 : R); r++) {
    const int q = tid + r * (HALF ? BT * DC : NT), c = q % (BT * DC), row = c / DC, col = c % DC;
    const bool is_v = q >= BT * DC;
    const int64_t at = (row * (is_v ? a.vs[2] : a.ks[2]) + 8 * col) * 4;
    voff[r] = q < kChunks && 8 * col < a.D ? (int)(HALF ? min(at, (int64_t)kOutOfRange - 16) : at) : kOutOfRange - 16;
    lds_off[r] = is_v ? kPlanesK * kPlaneK + row * LDV + 8 * col : row * LDK + 8 * col;
  }
  floatx4_t x[R][2];
  float top = 0.f;  // the largest magnitude among this thread's values of Q and K (and a part of V's); HALF: of the K in its registers
  auto is_v_wave = [&](int r) { return wave * 64 + r * NT >= BT * DC; };  // (a wave's 64 chunks are K's or V's: 8 D is a multiple of 64)
  auto fetch = [&](int kt, int first, int last) {  // rounds first .. last - 1
#pragma unroll
    for (int r = 0; r < R; r++) {
      if (r < first || r >= last) continue;
      if (kChunks % NT != 0 && wave * 64 + r * NT >= kChunks) continue;
      if constexpr (HALF) {
        const bool is_v = r >= kRoundsK;
        // (the round's rows are part of the vector offset: a scalar one beyond the last key defeats the range check)
        // (unsigned: a column that is not there, kOutOfRange, and a round's bytes together stay below 2^32)
        const uint32_t off = (uint32_t)voff[is_v] + round_bytes(r - (is_v ? kRoundsK : 0), is_v ? a.vs[2] : a.ks[2]);
#pragma unroll
        for (int e = 0; e < 2; e++)
          x[r][e] = __builtin_bit_cast(floatx4_t, __builtin_amdgcn_raw_buffer_load_b128(is_v ? v_rsrc : k_rsrc, off + 16 * e, kt * (is_v ? v_tile_bytes : k_tile_bytes), 0));
        continue;
      }
#pragma unroll
      for (int e = 0; e < 2; e++)
        x[r][e] = __builtin_bit_cast(floatx4_t, is_v_wave(r) ? __builtin_amdgcn_raw_buffer_load_b128(v_rsrc, voff[r] + 16 * e, kt * v_tile_bytes, 0)
                                                             : __builtin_amdgcn_raw_buffer_load_b128(k_rsrc, voff[r] + 16 * e, kt * k_tile_bytes, 0));
    }
  };
  auto top_of = [](const floatx4_t &lo, const floatx4_t &hi, float so_far) {
#pragma unroll
    for (int e = 0; e < 4; e++) so_far = fmaxf(fmaxf(fabsf(lo[e]), fabsf(hi[e])), so_far);
    return so_far;
  };
  // HALF: Q and K are split relative to a power of two, a row's own of Q and that of the largest key so far of K, so that what two
  // pieces do not hold is small beside what is there, whatever the magnitude (half_up, half_down).
  int key_exp = kHalfLeast;
  auto note_top = [&]() {  // ahead of the barrier in front of split_tile; grows a few times in a walk
    float t = 0.f;
#pragma unroll
    for (int r = 0; r < kRoundsK; r++) t = top_of(x[r][0], x[r][1], t);
    if (__builtin_amdgcn_ballot_w64(half_exponent(t) > key_exp) == 0) return;
    const int wave_exp = __builtin_amdgcn_readfirstlane(half_exponent(max_over_wave_rows(max_over_row(t))));
    if (lane == 0) atomicMax(&key_top, wave_exp);
  };
  auto split_tile = [&](int buf) {
#pragma unroll
    for (int r = 0; r < R; r++) {
      if (kChunks % NT != 0 && wave * 64 + r * NT >= kChunks) continue;
      if constexpr (HALF) {
        const bool is_v = r >= kRoundsK;
        uint16_t *to = &planes[lds_off[is_v] + (r - (is_v ? kRoundsK : 0)) * kRoundRows * (is_v ? LDV : LDK)];
        if (is_v) {
          const Pieces f = split_8(x[r][0] * kPieceScale, x[r][1] * kPieceScale);
#pragma unroll
          for (int i = 0; i < 3; i++) *reinterpret_cast<bf16x8_t *>(to + i * kPlaneV) = f.p[i];
        } else {
          const HalfPieces f = split_half_8(x[r][0], x[r][1], half_up(key_exp));
          *reinterpret_cast<half8_t *>(to) = f.hi;
          *reinterpret_cast<half8_t *>(to + kPlaneK) = f.lo;
        }
        continue;
      }
      const int plane = is_v_wave(r) ? kPlaneV : kPlaneK;
      // V is scaled, K is not; a round of chunks that are all K's or all V's spares the other one's part
      if (r * NT < BT * DC) top = top_of(x[r][0], x[r][1], top);
      const float scale = (r + 1) * NT > BT * DC && is_v_wave(r) ? kPieceScale : 1.f;
      const Pieces f = split_8(x[r][0] * scale, x[r][1] * scale);
#pragma unroll
      for (int i = 0; i < 3; i++) *reinterpret_cast<bf16x8_t *>(&planes[buf * kTile + i * plane + lds_off[r]]) = f.p[i];
    }
  };
  if (n_kv_tiles > 0) fetch(0, 0, R);
  if (tid == 0) redo = 0, key_top = kHalfLeast;
  if (D % 32 != 0) {  // columns of the last block of O^T that no chunk fills
    for (int i = tid; i < NBUF * 3 * BT * (32 * DB - D); i += NT) {
      const int row = i / (32 * DB - D), col = i % (32 * DB - D), plane = row / BT;
      planes[plane / 3 * kTile + kPlanesK * kPlaneK + plane % 3 * kPlaneV + row % BT * LDV + D + col] = 0;
    }
  }

  // ---- Q: lane (n, g) holds q[qi][16 ks + 8 g .. + 7] ----
  floatx4_t q[KS][2];
  auto load_q = [&]() {
#pragma unroll
    for (int ks = 0; ks < KS; ks++)
#pragma unroll
      for (int e = 0; e < 2; e++) {
        q[ks][e] = (floatx4_t){0.f, 0.f, 0.f, 0.f};
        if ((uint32_t)qi < (uint32_t)a.Sq && 16 * ks + 8 * g < a.D) q[ks][e] = *reinterpret_cast<const floatx4_t *>(qp + (int64_t)qi * a.qs[2] + 16 * ks + 8 * g + 4 * e);
      }
    if (D % 32 == 0 && a.q_rope) {  // (the head dim equals the tiling: the partner of an element is in the same lane)
      const float pos = (float)((a.q_pos0 ? a.q_pos0[b] : a.q_prev_seq) + qi);
      if (!a.q_interleaved) {
#pragma unroll
        for (int ks = 0; ks < KS / 2; ks++)
#pragma unroll
          for (int e = 0; e < 8; e++) {
            float sn, cs, o0, o1;
            sincos_angle(pos * rope_inv_freq(16 * ks + 8 * g + e, D, a.q_log2_base), &sn, &cs);
            rope_rotate(q[ks][e >> 2][e & 3], q[ks + KS / 2][e >> 2][e & 3], sn, cs, &o0, &o1);
            q[ks][e >> 2][e & 3] = o0;
            q[ks + KS / 2][e >> 2][e & 3] = o1;
          }
      } else {
#pragma unroll
        for (int ks = 0; ks < KS; ks++)
#pragma unroll
          for (int e = 0; e < 8; e += 2) {
            float sn, cs, o0, o1;
            sincos_angle(pos * rope_inv_freq((16 * ks + 8 * g + e) / 2, D, a.q_log2_base), &sn, &cs);
            rope_rotate(q[ks][e >> 2][e & 3], q[ks][e >> 2][(e & 3) + 1], sn, cs, &o0, &o1);
            q[ks][e >> 2][e & 3] = o0;
            q[ks][e >> 2][(e & 3) + 1] = o1;
          }
      }
    }
  };
  // Two pieces of the queries take scale log2(e) along, up to the power of two `unit`: as a factor of the scores its rounding would weigh
  // as much as what the pieces lack.
  const float c = a.scale * kLog2e;
  const float unit = HALF ? __int_as_float(__float_as_int(c) & 0x7f800000) : c, grow = 1.f / unit;
  std::conditional_t<HALF, HalfPieces, Pieces> qf[KS];
  load_q();
  if (HALF) __syncthreads();  // (key_top is there)
#pragma unroll
  for (int ks = 0; ks < KS; ks++) top = top_of(q[ks][0], q[ks][1], top);
  const int q_exp = half_exponent(max_over_wave_halves(top) * (c * grow));
  const float row_unit = unit * half_down(q_exp);  // of a score whose K is as it came
#pragma unroll
  for (int ks = 0; ks < KS; ks++) {
    if constexpr (HALF) qf[ks] = split_half_8(q[ks][0], q[ks][1], c * grow * half_up(q_exp), fmaf(a.scale, kLog2eRest, fmaf(a.scale, kLog2e, -c)) * grow * half_up(q_exp));
    else qf[ks] = split_8(q[ks][0], q[ks][1]);
  }

  floatx16_t oacc[DB];
  float m_i, l_i;
  auto clear = [&]() {
    m_i = -INFINITY;
    l_i = 0.f;
#pragma unroll
    for (int db = 0; db < DB; db++)
#pragma unroll
      for (int i = 0; i < 16; i++) oacc[db][i] = 0.f;
  };
  clear();
  const int last_key = (CAUSAL ? min(qi, n_keys - 1) : n_keys - 1) - 4 * g;  // that the lane's row sees, less the lane's own offset
  // Mask, running max, weights and their sum; register i of block kb is key k0 + 32 kb + 8 (i / 4) + 4 g + i % 4. `unit` is what a score is in log2
  // units; the running max is a score, HALF: one in log2 units. `exponent` is that of a weight, from its score. HALF: what the smaller products
  // add to a score is masked as well (it may be NaN), and counts in the max of large scores only (`whole`), where it could move a weight by more
  // than its exponent holds.
  auto soften = [&](auto &s, auto &small, int blocks, int k0, float unit, const auto &exponent, const auto &whole) {
    if (k0 + 32 * blocks > n_keys || (CAUSAL && k0 + 32 * blocks - 1 > wave_q_lo)) {
#pragma unroll
      for (int kb = 0; kb < blocks; kb++)
#pragma unroll
        for (int i = 0; i < 16; i++) {
          const int key = k0 + 32 * kb + 8 * (i >> 2) + (i & 3);
          if (HALF ? key > last_key : key + 4 * g >= n_keys || (CAUSAL && key + 4 * g > qi)) {
            if (HALF) small[kb][i] = 0.f;
            s[kb][i] = -INFINITY;
          }
        }
    }
    auto top_score = [&](const auto &score) {
      float mx = score(0, 0);
#pragma unroll
      for (int kb = 0; kb < blocks; kb++)
#pragma unroll
        for (int i = 0; i < 16; i++) mx = fmaxf(mx, score(kb, i));
      return max_over_wave_halves(mx);
    };
    float mx = top_score([&](int kb, int i) { return s[kb][i]; });
    if (HALF) {
      mx *= unit;
      if (__builtin_amdgcn_ballot_w64(fabsf(mx) > 1024.f) != 0) mx = top_score(whole) * unit;
      unit = 1.f;
    }
    if (__builtin_amdgcn_ballot_w64((mx - m_i) * unit > kLazyRescale) != 0) {
      const float m_new = fmaxf(m_i, mx);
      const float alpha = m_i == -INFINITY ? 0.f : __builtin_amdgcn_exp2f((m_i - m_new) * unit);
      m_i = m_new;
      l_i *= alpha;
#pragma unroll
      for (int db = 0; db < DB; db++)
#pragma unroll
        for (int i = 0; i < 16; i++) oacc[db][i] *= alpha;
    }
    const float mc = m_i == -INFINITY ? 0.f : m_i * unit;
    float l0 = 0.f, l1 = 0.f;
#pragma unroll
    for (int kb = 0; kb < blocks; kb++)
#pragma unroll
      for (int i = 0; i < 16; i += 2) {
        s[kb][i] = __builtin_amdgcn_exp2f(exponent(kb, i, mc));
        s[kb][i + 1] = __builtin_amdgcn_exp2f(exponent(kb, i + 1, mc));
        l0 += s[kb][i];
        l1 += s[kb][i + 1];
      }
    l_i += l0 + l1;
  };

  const int k_frag = (32 * NKB * kg + n) * LDK + 8 * g;
  // the transposing read: within each 16 lanes, lane i supplies row i / 4 and columns 4 (i % 4) of a 4-key x 16-column patch
  const int i16 = lane & 15;
  const int v_frag = (32 * NKB * kg + 4 * g + (i16 >> 2)) * LDV + 16 * ((lane >> 4) & 1) + 4 * (i16 & 3);
  // The five smaller products are summed ahead of the large one, those of the scores in accumulators of their own: their sums are
  // rounded at 2^-8 of the result's magnitude. A tile's share of O^T is summed from zero and added once.
  constexpr int kX[6] = {2, 0, 1, 1, 0, 0}, kY[6] = {0, 2, 1, 0, 1, 0};

  if (NBUF == 2 && n_kv_tiles > 0) {
    split_tile(0);
    if (n_kv_tiles > 1) fetch(1, 0, R);
  }
  for (int kt = 0; kt < n_kv_tiles; kt++) {
    const int buf = NBUF == 2 ? kt & 1 : 0;
    if constexpr (HALF) note_top();
    __syncthreads();  // everyone is done with tile kt - 1 (and, with two tiles, tile kt is in LDS)
    if (NBUF == 1) {
      if constexpr (HALF) key_exp = __builtin_amdgcn_readfirstlane(key_top);
      split_tile(0);
      if (kt + 1 < n_kv_tiles) fetch(kt + 1, 0, HALF ? kRoundsK : R);
      __syncthreads();  // tile kt is in LDS
    }
    auto prepare_next = [&]() {
      if (HALF && kt + 1 < n_kv_tiles) fetch(kt + 1, kRoundsK, R);  // (V's registers are not to be had beside the scores' products)
      if (NBUF == 1) return;
      split_tile(buf ^ 1);  // (of the last tile again, behind the last one: nobody reads it)
      if (kt + 2 < n_kv_tiles) fetch(kt + 2, 0, R);
    };
    const int k0 = kt * BT + 32 * NKB * kg;
    if ((CAUSAL && k0 > wave_q_hi) || k0 >= k_end) {
      prepare_next();
      continue;
    }
    const uint16_t *Kp = planes + buf * kTile, *Vp = Kp + kPlanesK * kPlaneK;

    floatx16_t s[NKB], small[NKB];
#pragma unroll
    for (int kb = 0; kb < NKB; kb++)
#pragma unroll
      for (int i = 0; i < 16; i++) s[kb][i] = small[kb][i] = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
      if constexpr (HALF) {
        half8_t kf[NKB][2];
#pragma unroll
        for (int kb = 0; kb < NKB; kb++)
#pragma unroll
          for (int i = 0; i < 2; i++) kf[kb][i] = *reinterpret_cast<const half8_t *>(&Kp[i * kPlaneK + k_frag + 32 * kb * LDK + 16 * ks]);
#pragma unroll
        for (int j = 0; j < 3; j++)
#pragma unroll
          for (int kb = 0; kb < NKB; kb++) {
            floatx16_t &acc = j < 2 ? small[kb] : s[kb];
            acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[kb][j == 0], j == 1 ? qf[ks].lo : qf[ks].hi, acc, 0, 0, 0);
          }
        continue;
      } else {
      bf16x8_t kf[NKB][3];
#pragma unroll
      for (int kb = 0; kb < NKB; kb++)
#pragma unroll
        for (int i = 0; i < 3; i++) kf[kb][i] = *reinterpret_cast<const bf16x8_t *>(&Kp[i * kPlaneK + k_frag + 32 * kb * LDK + 16 * ks]);
#pragma unroll
      for (int j = 0; j < 6; j++)
#pragma unroll
        for (int kb = 0; kb < NKB; kb++) {
          floatx16_t &acc = j < 5 ? small[kb] : s[kb];
          acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[kb][kX[j]], qf[ks].p[kY[j]], acc, 0, 0, 0);
        }
      }
    }
    prepare_next();
    if constexpr (HALF) {
      const float by = row_unit * half_down(key_exp);
      soften(s, small, NKB, k0, by, [&](int kb, int i, float mc) { return fmaf(small[kb][i], by * (1.f / kHalfGap), fmaf(s[kb][i], by, -mc)); },
             [&](int kb, int i) { return fmaf(small[kb][i], 1.f / kHalfGap, s[kb][i]); });
    } else {
#pragma unroll
      for (int kb = 0; kb < NKB; kb++)
#pragma unroll
        for (int i = 0; i < 16; i++) s[kb][i] += small[kb][i];
      auto score = [&](int kb, int i) { return s[kb][i]; };
      soften(s, small, NKB, k0, c, [&](int kb, int i, float mc) { return s[kb][i] * c - mc; }, score);
    }
    Pieces pf[NKB][2];
#pragma unroll
    for (int kb = 0; kb < NKB; kb++)
#pragma unroll
      for (int t = 0; t < 2; t++) {
        floatx4_t lo, hi;
#pragma unroll
        for (int e = 0; e < 4; e++) {
          lo[e] = s[kb][8 * t + e] * kPieceScale;
          hi[e] = s[kb][8 * t + 4 + e] * kPieceScale;
        }
        pf[kb][t] = split_8(lo, hi);
      }
#pragma unroll
    for (int db = 0; db < DB; db++) {
      floatx16_t o;
#pragma unroll
      for (int i = 0; i < 16; i++) o[i] = 0.f;
#pragma unroll
      for (int kb = 0; kb < NKB; kb++) {
        bf16x8_t vf[2][3];
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
          for (int i = 0; i < 3; i++) {
            const uint16_t *p = &Vp[i * kPlaneV + v_frag + (32 * kb + 16 * t) * LDV + 32 * db];
            const shortx4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_shortx4_t *)p);
            const shortx4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_shortx4_t *)(p + 8 * LDV));
            vf[t][i] = __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
          }
#pragma unroll
        for (int j = 0; j < 6; j++)
#pragma unroll
          for (int t = 0; t < 2; t++) o = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[t][kX[j]], pf[kb][t].p[kY[j]], o, 0, 0, 0);
      }
#pragma unroll
      for (int i = 0; i < 16; i++) oacc[db][i] += o[i];
    }
  }

  // ---- values that pieces do not hold, anywhere in the workgroup: its rows again with the fp32 product ----
  // (up to here the lost bits of Q and K move a scaled score by less than 2^-37)
  // (two pieces: what Q and K lack of 2^-36 of 2^15 each, D times, moves one by less than 2^-22, or than half an fp32 unit of the row's
  // largest score, which the sum of its products is rounded to anyway; below 2^-38 the units of small queries and keys would be subnormal)
  const bool held = HALF ? row_unit * half_down(key_exp) * (16.f * D) <= fmaxf(4.f, fabsf(m_i) - kLazyRescale) && unit >= 0x1p-38f && unit < 0x1p100f
                         : fmaxf(top, 1.f) * a.scale <= 0x1p80f;
  float finite = 0.f;
#pragma unroll
  for (int db = 0; db < DB; db++)
#pragma unroll
    for (int i = 0; i < 16; i++) finite = fmaf(oacc[db][i], 0.f, finite);
  finite = fmaf(l_i, 0.f, finite);
  __syncthreads();
  if (!held || finite != 0.f || finite != finite) redo = 1;
  __syncthreads();
  float unscale = kPieceUnscale * kPieceUnscale;
  if (redo) {
    unscale = 1.f;
    clear();
    load_q();
    for (int k0 = 32 * kg; k0 < k_end; k0 += 32 * KSPLIT) {
      if (CAUSAL && k0 > wave_q_hi) break;
      floatx16_t s[1];
#pragma unroll
      for (int i = 0; i < 16; i++) s[0][i] = 0.f;
      const bool in = k0 + n < n_keys;
#pragma unroll
      for (int ks = 0; ks < KS; ks++)
#pragma unroll
        for (int e = 0; e < 2; e++) {
          floatx4_t kf = {0.f, 0.f, 0.f, 0.f};
          if (in && 16 * ks + 8 * g < a.D) kf = *reinterpret_cast<const floatx4_t *>(kp + (int64_t)(k0 + n) * a.ks[2] + 16 * ks + 8 * g + 4 * e);
#pragma unroll
          for (int i = 0; i < 4; i++) s[0] = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[i], q[ks][e][i], s[0], 0, 0, 0);
        }
      auto score = [&](int, int i) { return s[0][i]; };
      soften(s, s, 1, k0, c, [&](int, int i, float mc) { return s[0][i] * c - mc; }, score);
      auto v_at = [&](int key, int db) { return key < n_keys && 32 * db + n < a.D ? vp[(int64_t)key * a.vs[2] + 32 * db + n] : 0.f; };
      if (!CAUSAL || k0 + 31 <= wave_q_lo) {
#pragma unroll
        for (int i = 0; i < 16; i++)
#pragma unroll
          for (int db = 0; db < DB; db++)
            oacc[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(v_at(k0 + 8 * (i >> 2) + 4 * g + (i & 3), db), s[0][i], oacc[db], 0, 0, 0);
      } else {
        // on the diagonal key by key: a value that is not finite stays out of the rows that do not see it (zero times it is NaN)
#pragma unroll
        for (int i = 0; i < 16; i++)
          for (int half = 0; half < 2; half++) {
            const int key = k0 + 8 * (i >> 2) + 4 * half + (i & 3);
#pragma unroll
            for (int db = 0; db < DB; db++) {
              const floatx16_t with = __builtin_amdgcn_mfma_f32_32x32x2f32(g == half ? v_at(key, db) : 0.f, g == half ? s[0][i] : 0.f, oacc[db], 0, 0, 0);
              if (key <= qi) oacc[db] = with;
            }
          }
      }
    }
  }

  // ---- fold the second key group's (m, l, O) into the first's; lane for lane the same layout ----
  if constexpr (KSPLIT > 1) {
    constexpr int NF = DB * 16 + 2;
    static_assert(RW * NF * 64 * 4 <= (int)sizeof(planes), "the partial results fit the planes");
    float *xch = reinterpret_cast<float *>(planes) + (wave % RW) * (NF * 64) + lane;
    const float in_c = HALF ? 1.f : c;  // (what the max is a multiple of)
    if (kg > 0) {
      xch[0] = m_i;
      xch[64] = l_i;
#pragma unroll
      for (int db = 0; db < DB; db++)
#pragma unroll
        for (int i = 0; i < 16; i++) xch[(2 + db * 16 + i) * 64] = oacc[db][i];
    }
    __syncthreads();
    if (kg > 0) return;
    const float m1 = xch[0], m_all = fmaxf(m_i, m1);
    const float a0 = m_i == -INFINITY ? 0.f : __builtin_amdgcn_exp2f((m_i - m_all) * in_c);
    const float a1 = m1 == -INFINITY ? 0.f : __builtin_amdgcn_exp2f((m1 - m_all) * in_c);
    l_i = l_i * a0 + xch[64] * a1;
#pragma unroll
    for (int db = 0; db < DB; db++)
#pragma unroll
      for (int i = 0; i < 16; i++) oacc[db][i] = oacc[db][i] * a0 + xch[(2 + db * 16 + i) * 64] * a1;
  }

  const float l_tot = sum_over_wave_halves(l_i);
  const float inv = l_tot > 0.f ? unscale / l_tot : 0.f;
  if ((uint32_t)qi < (uint32_t)a.Sq) {
    float *op = reinterpret_cast<float *>(a.out) + b * a.os[0] + hq * a.os[1] + (int64_t)qi * a.os[2];
#pragma unroll
    for (int db = 0; db < DB; db++)
#pragma unroll
      for (int i4 = 0; i4 < 4; i4++) {
        const int d = db * 32 + 8 * i4 + 4 * g;
        if (d >= a.D) continue;
        *reinterpret_cast<float4 *>(op + d) = make_float4(oacc[db][4 * i4 + 0] * inv, oacc[db][4 * i4 + 1] * inv,
                                                          oacc[db][4 * i4 + 2] * inv, oacc[db][4 * i4 + 3] * inv);
      }
  }
}

template <int D, int NW, int KSPLIT>
int launch_form(const PrefillArgs &a, hipStream_t stream) {
  constexpr int BM = 32 * NW / KSPLIT;
  const int n_q_tiles = (a.Sq + BM - 1) / BM;
  const int64_t wgs = deal_grid((int64_t)a.B * a.Hq, n_q_tiles);
  const int rc = check_grid(wgs, 64 * NW);
  if (rc != LMH_OK) return rc;
  dim3 grid((uint32_t)wgs), block(64 * NW);
  if (plan_only("prefill_f32_split_kernel<D=%d, %s, key groups=%d> rows=%d, workgroups=%u", D, a.causal ? "causal" : "full", KSPLIT, BM, grid.x)) return LMH_OK;
  const Deal deal = make_deal(a.B, a.Hq, n_q_tiles, a.causal ? 8 / NW : 0, device_cu_count());
  if (a.causal) hipLaunchKernelGGL((prefill_f32_split_kernel<D, true, NW, KSPLIT>), grid, block, 0, stream, deal, a);
  else hipLaunchKernelGGL((prefill_f32_split_kernel<D, false, NW, KSPLIT>), grid, block, 0, stream, deal, a);
  LMH_HIP_TRY(hipGetLastError());
  return LMH_OK;
}

template <int D>
int launch_for_d(const PrefillArgs &a, int form, hipStream_t stream) {
  if (form == 0) return launch_form<D, 4, 2>(a, stream);
  if (form == 1) return launch_form<D, 8, 2>(a, stream);
  return launch_form<D, 8, 1>(a, stream);
}

}  // namespace

// Estimated microseconds of the cheapest form (0: 64 rows, two workgroups on a CU; 1: 128 rows; 2: 256 rows), from the launch's own
// tiles as in prefill_mfma.hip: without a mask whole rounds, causal the longest workgroup and the mean over the CUs. Fitted to 330
// launches of drawn sizes, rms 3 to 10 %.
double prefill_f32_split_cost(const PrefillArgs &a, int *form) {
  struct Cost { double fixed, alone, per_wg, shared; };  // a tile of 64 keys in a CU's only workgroup, and in one of several
  const int64_t cus = device_cu_count(), heads = (int64_t)a.B * a.Hq, row_tiles = (a.Sk + 63) / 64;
  if (a.D > 96) {  // in 128 rows only; fitted to 2300 launches, rms 4 to 8 %
    static const Cost wide[2][2] = {{{-0.68, 3.68, 9.29, 3.97}, {1.13, 3.44, 8.35, 4.30}}, {{-0.68, 3.70, 10.75, 4.06}, {0.89, 3.48, 9.58, 4.52}}};  // [up to 112, 128][causal]
    const Cost &c = wide[a.D > 112][a.causal != 0];
    const int64_t n = (a.Sq + 127) / 128, rounds = (heads * n + cus - 1) / cus;
    *form = 1;
    if (!a.causal) return c.fixed + row_tiles * (rounds <= 1 ? c.alone : c.shared * rounds) + c.per_wg * rounds;
    // the last workgroup of a head ends at its last row, the others 128 rows apart (causal_shift): of `diagonal` key tiles, two less each, `all` walk every key
    const int64_t diagonal = (a.Sq + 63) / 64, all = std::min(n, std::max<int64_t>(0, (diagonal - row_tiles + 1) / 2));
    const double longest = (double)std::min(row_tiles, diagonal) * c.alone;
    if (rounds <= 1) return c.fixed + longest + c.per_wg;
    const double mean = (double)heads * (all * row_tiles + (n - all) * (diagonal - (n - 1 + all))) / cus * c.shared;
    return c.fixed + sqrt(sqrt(longest * longest * longest * longest + mean * mean * mean * mean)) + c.per_wg * (heads * n) / cus;
  }
  static const Cost costs[3][3][2] = {  // [head dims up to 64, 80, 96][form][causal]
      {{{3.3, 1.89, 1.8, 1.33}, {3.6, 1.86, 1.8, 1.40}}, {{1.3, 2.26, 5.7, 0.}, {1.5, 2.13, 6.4, 2.47}}, {{0., 4.26, 8.4, 0.}, {0., 3.98, 8.4, 4.13}}},
      {{{2.6, 2.61, 2.4, 1.76}, {3.3, 2.51, 2.7, 1.85}}, {{0., 3.00, 7.0, 0.}, {0., 2.86, 8.0, 3.28}}, {{0., 4.96, 10.3, 0.}, {0., 4.46, 10.1, 5.47}}},
      {{{0.2, 3.36, 5.0, 2.28}, {2.3, 3.17, 5.5, 2.19}}, {{0., 3.30, 8.9, 0.}, {0., 3.03, 10.3, 3.44}}, {{0., 6.3, 11.6, 0.}, {0., 5.73, 10.0, 6.74}}}};
  double least = INFINITY;
  for (int f = 0; f < 3; f++) {
    const Cost &c = costs[a.D <= 64 ? 0 : a.D <= 80 ? 1 : 2][f][a.causal != 0];
    const int64_t step = int64_t(1) << f, n = (a.Sq + 64 * step - 1) / (64 * step), rounds = (heads * n + cus - 1) / cus;
    double t;
    if (!a.causal) {
      const int64_t pairs = f == 0 ? rounds / 2 : 0;
      t = c.fixed + row_tiles * (pairs * std::max(c.alone, 2 * c.shared) + (rounds - 2 * pairs) * c.alone) + c.per_wg * rounds;
    } else {
      const int64_t ramp = std::min(n, row_tiles / step);
      const double longest = (double)std::min(row_tiles, n * step) * c.alone;
      const double mean = (double)heads * (step * ramp * (ramp + 1) / 2 + (n - ramp) * row_tiles) / cus * c.shared;
      t = rounds <= 1 ? c.fixed + longest + c.per_wg
                      : c.fixed + sqrt(sqrt(longest * longest * longest * longest + mean * mean * mean * mean)) + c.per_wg * (heads * n) / cus;
    }
    if (t < least) least = t, *form = f;
  }
  return least;
}

int launch_prefill_f32_split(const PrefillArgs &a, int form, hipStream_t stream) {
  if (a.D <= 64) return launch_for_d<64>(a, form, stream);
  if (a.D <= 80) return launch_for_d<80>(a, form, stream);
  if (a.D <= 96) return launch_for_d<96>(a, form, stream);
  return launch_form<128, 8, 2>(a, stream);
}

}  // namespace lmh
