// Flash attention forward in fp32 on the gfx950 matrix cores (v_mfma_f32_16x16x4_f32).
//
// fp32 is the reference's only element type (flash_attn_cpu, reference src/Execution.jl:453-479), and its parity budget
// (1e-5 of the output range) rules out half-precision operands, so this kernel keeps Q, K, V and P in fp32 end to end; only
// the order of the fp32 additions differs from the reference's loop.
//
// Bound: the fp32 matrix pipe (157 TFLOP/s, 64 flops per cycle and SIMD; softmax, LDS reads and staging hide behind it).
// Same data flow as prefill_mfma.hip: scores are computed transposed, S^T = K Q^T, so a lane holds one query column; the
// accumulator registers that hold P are directly the B operands of O^T = V^T P^T; K and V tiles are staged by LDS-writing
// buffer loads, one tile ahead. A wave works on 16 query rows and 16 keys at a time. The 32 x 32 x 2 product runs at the
// same rate; the smaller blocks buy
//   * balance: a wave's share of a launch is 16 rows and, with KG key groups, 1 / KG of the keys, so that a few hundred
//     128-row workgroups' worth of work spreads evenly over the 1024 SIMDs;
//   * latency: where a launch is one wave's walk over its keys, that walk is a quarter as long per key group;
//   * padding: head dims go in steps of 16, where 32 x 32 blocks of O^T pad 80 to 96 and 112 to 128;
//   * registers: 64 for Q and 64 for O at head dim 256, which the larger blocks cannot hold.
// Measured, us, with 32 x 32 blocks -> now: B=1 H=8 S=128 D=64 causal 7.3 -> 5.5, B=2 H=12 S=1023 D=80 103 -> 77, B=1 H=16
// S=2048 D=64 causal 143 -> 85, B=1 H=8 S=1000 D=128 causal 76 -> 38, B=4 H=20 448 x 1500 D=64 194 -> 148, B=1 H=32 S=4096
// D=96 causal 822 -> 803 (128 TFLOP/s, 82 % of the peak). Without a mask, where all workgroups are equally long and fill the
// chip, the 32 x 32 blocks stay ahead by 1 to 13 %: prefill_f32_full.hip.
//
// Layout of the 16 x 16 x 4 product: lane (n = lane % 16, g = lane / 16); A and B give element k = g of row / column n, the
// result register i is row 4 g + i of column n. The head dim is contracted in the order d = 16 j + 4 g + e, so a 128-bit K
// fragment feeds four MFMAs; the keys in the order 4 g + i, so register i of a block's P is the B operand of MFMA i and V
// comes as one 32-bit LDS read per MFMA (row stride D + 4 floats: the four rows of a read fall on different banks, and so do
// the 16 rows of a K fragment read).
#include <math.h>

#include "common.hpp"
#include "dtypes.hpp"
#include "rope.hpp"

namespace lmh {
namespace {

constexpr float kLog2e = 1.4426950408889634f;
constexpr int kOutOfRange = 0x7ffffff0;   // byte offset no K/V slice reaches: a buffer load there returns zeros
constexpr float kLazyRescale = 8.0f;      // the running max is raised only when outgrown by 2^8 (see prefill_mfma.hpp)

// RW waves own 16 rows each, KG waves share 16 rows by taking the kg-th 16 NK keys of every staged tile of 16 NK KG keys.
template <int D, int RW, int KG, int NK> constexpr int tile_blocks() { return (16 * NK * KG * (D / 4 + 1) + 63) / 64; }  // 1 KB blocks
template <int D, bool CAUSAL, int RW, int KG, int NK>
__global__ __launch_bounds__(64 * RW * KG, 1) void prefill_f32_kernel(Deal deal, PrefillArgs a) {
  request_args(a);
  request_args(deal);
  constexpr int NW = RW * KG;
  constexpr int BM = 16 * RW;            // query rows per workgroup
  constexpr int BW = 16 * NK;            // keys a wave takes per tile
  constexpr int BT = BW * KG;            // keys per staged tile
  constexpr int J = D / 16;              // 128-bit K fragments per 16 keys = 16-row blocks of O^T
  constexpr int LD = D + 4;              // LDS row stride in floats
  constexpr int C = LD / 4;              // 16-byte chunks per LDS row (the last is padding)
  constexpr int BLOCKS = tile_blocks<D, RW, KG, NK>();
  __shared__ __attribute__((aligned(16))) float Ks2[2][BLOCKS * 256];
  __shared__ __attribute__((aligned(16))) float Vs2[2][BLOCKS * 256];

  // ---- which (b, hq, query tile): a head's tiles on one XCD, causal tiles heaviest first (see prefill_mfma.hip) ----
  int bh, tile_rank;
  if (!deal_tile(deal, blockIdx.x & 7, blockIdx.x >> 3, &bh, &tile_rank)) return;
  const int b = (int)((uint32_t)bh / deal.hq), hq = bh - b * a.Hq;
  const int kvh = kv_head_of(hq, a.Hq, a.Hkv, a.head_map);
  const int q_tile = CAUSAL ? (deal.tiles - 1 - tile_rank) : tile_rank;
  const int q0 = q_tile * BM - (CAUSAL ? causal_shift(deal.tiles, BM, a.Sq, BT) : 0);

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int n = lane & 15, g = lane >> 4;
  const int kg = wave / RW;
  const int wave_q_lo = q0 + (wave % RW) * 16;
  const int wave_q_hi = wave_q_lo + 15;
  const int qi = wave_q_lo + n;

  int n_keys = a.kv_len ? a.kv_len[b] : a.Sk;
  n_keys = min(max(n_keys, 0), a.Sk);
  int k_end = n_keys;
  if (CAUSAL) k_end = min(k_end, q0 + BM);
  const int n_kv_tiles = (k_end + BT - 1) / BT;

  const float *qp = reinterpret_cast<const float *>(a.q) + b * a.qs[0] + hq * a.qs[1];
  const float *kp = reinterpret_cast<const float *>(a.k) + b * a.ks[0] + kvh * a.ks[1];
  const float *vp = reinterpret_cast<const float *>(a.v) + b * a.vs[0] + kvh * a.vs[1];

  // ---- tile staging (see prefill_mfma.hip): wave w issues blocks w, w + NW, ... of K, then of V ----
  typedef int32_t i32x4_t __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) void lds_void_t;
  constexpr int BPW = (BLOCKS + NW - 1) / NW;
  const int wave_u = __builtin_amdgcn_readfirstlane(wave);
  __builtin_assume(wave_u >= 0 && wave_u < NW);
  auto make_desc = [](const float *base, int bytes) {
    const uint64_t p = (uint64_t)base;
    i32x4_t d;
    d[0] = __builtin_amdgcn_readfirstlane((int)(uint32_t)p);
    d[1] = __builtin_amdgcn_readfirstlane((int)((p >> 32) & 0xffff));  // stride 0: raw buffer
    d[2] = __builtin_amdgcn_readfirstlane(bytes);
    d[3] = 0x00020000;
    return d;
  };
  const i32x4_t k_desc = make_desc(kp, (int)((int64_t)n_keys * a.ks[2] * 4));
  const i32x4_t v_desc = make_desc(vp, (int)((int64_t)n_keys * a.vs[2] * 4));
  const int cpr = a.D / 4;  // the tensors' own head dim may be smaller than D: the missing columns are zeros, never stored
  int k_voff[BPW], v_voff[BPW];
#pragma unroll
  for (int j = 0; j < BPW; j++) {
    const int ch = (wave + NW * j) * 64 + lane;
    const int row = ch / C, col = ch % C;
    const bool in = row < BT && col < cpr;
    k_voff[j] = in ? (int)((row * a.ks[2] + col * 4) * 4) : kOutOfRange;
    v_voff[j] = in ? (int)((row * a.vs[2] + col * 4) * 4) : kOutOfRange;
  }
  const int k_tile_bytes = (int)(BT * a.ks[2] * 4), v_tile_bytes = (int)(BT * a.vs[2] * 4);
  const uint32_t k_lds0 = (uint32_t)(uintptr_t)(lds_void_t *)&Ks2[0][0] + wave_u * 1024;
  const uint32_t v_lds0 = (uint32_t)(uintptr_t)(lds_void_t *)&Vs2[0][0] + wave_u * 1024;
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"  // m0 is a reserved register; it is only written here
  auto load_block = [](i32x4_t desc, uint32_t lds_addr, int voff, int soff) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 :: "s"(lds_addr), "v"(voff), "s"(desc), "s"(soff) : "memory", "m0");
  };
#pragma clang diagnostic pop
  auto load_tile = [&](int kt, int buf) {
#pragma unroll
    for (int j = 0; j < BPW; j++)
      if (wave_u + NW * j < BLOCKS) load_block(k_desc, k_lds0 + buf * (BLOCKS * 1024) + j * (NW * 1024), k_voff[j], kt * k_tile_bytes);
#pragma unroll
    for (int j = 0; j < BPW; j++)
      if (wave_u + NW * j < BLOCKS) load_block(v_desc, v_lds0 + buf * (BLOCKS * 1024) + j * (NW * 1024), v_voff[j], kt * v_tile_bytes);
  };

  // ---- Q fragments: lane (n, g) holds q[qi][16 j + 4 g .. + 3] ----
  floatx4_t qf[J];
#pragma unroll
  for (int j = 0; j < J; j++) {
    float4 raw = make_float4(0.f, 0.f, 0.f, 0.f);
    if ((uint32_t)qi < (uint32_t)a.Sq && 16 * j + 4 * g < a.D) raw = *reinterpret_cast<const float4 *>(qp + (int64_t)qi * a.qs[2] + 16 * j + 4 * g);
    qf[j] = (floatx4_t){raw.x, raw.y, raw.z, raw.w};
  }
  if (n_kv_tiles > 0) load_tile(0, 0);

  floatx4_t oacc[J];
#pragma unroll
  for (int db = 0; db < J; db++) oacc[db] = floatx4_t{0.f, 0.f, 0.f, 0.f};
  float m_i = -INFINITY;  // running max of the raw scores of query qi (the same in its four lanes)
  float l_i = 0.f;        // this lane's share of the running sum
  const float c = a.scale * kLog2e;

  // Rotary embedding of the query fragments (PrefillArgs::q_rope; the head dim equals D, a multiple of 32): the partner of
  // element 16 j + 4 g + e is in fragment j + D/32 of the same lane, interleaved pairs are neighbours. inv_freq is computed
  // once per workgroup into the second K buffer, which nothing writes before the loop's first barrier.
  if constexpr (J % 2 == 0) {
    if (a.q_rope) {
      float *table = &Ks2[1][0];
      for (int i = tid; i < D / 2; i += 64 * NW) table[i] = rope_inv_freq(i, D, a.q_log2_base);
      __syncthreads();
      const float pos = (float)((a.q_pos0 ? a.q_pos0[b] : a.q_prev_seq) + qi);
      if (!a.q_interleaved) {
#pragma unroll
        for (int j = 0; j < J / 2; j++)
#pragma unroll
          for (int e = 0; e < 4; e++) {
            float sn, cs, o0, o1;
            sincos_angle(pos * table[16 * j + 4 * g + e], &sn, &cs);
            rope_rotate(qf[j][e], qf[j + J / 2][e], sn, cs, &o0, &o1);
            qf[j][e] = o0;
            qf[j + J / 2][e] = o1;
          }
      } else {
#pragma unroll
        for (int j = 0; j < J; j++)
#pragma unroll
          for (int e = 0; e < 4; e += 2) {
            float sn, cs, o0, o1;
            sincos_angle(pos * table[(16 * j + 4 * g + e) / 2], &sn, &cs);
            rope_rotate(qf[j][e], qf[j][e + 1], sn, cs, &o0, &o1);
            qf[j][e] = o0;
            qf[j][e + 1] = o1;
          }
      }
    }
  }
  // The compiler does not model the asm loads or the asm wait below: make it wait for Q here, not inside the loop.
#pragma unroll
  for (int j = 0; j < J; j++) asm volatile("" :: "v"(qf[j]));

  const int k_frag_off = n * LD + 4 * g;  // + 16 kb LD + 16 j
  const int v_frag_off = 4 * g * LD + n;  // + (16 kb + i) LD + 16 db

  for (int kt = 0; kt < n_kv_tiles; kt++) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's blocks of tile kt are in LDS
    __syncthreads();  // ... and everyone's; tile kt - 1 has been consumed, its buffer is free
    if (kt + 1 < n_kv_tiles) load_tile(kt + 1, (kt + 1) & 1);
    const float *Ks = Ks2[kt & 1] + kg * (BW * LD);
    const float *Vs = Vs2[kt & 1] + kg * (BW * LD);
    const int k0 = kt * BT + kg * BW;         // first key of this wave's share of the tile
    if (CAUSAL && k0 > wave_q_hi) continue;   // all of it above this wave's diagonal
    if (KG > 1 && k0 >= k_end) continue;      // ... or past the last key

    // ---- S^T = K Q^T; the NK blocks' accumulator chains alternate ----
    floatx4_t sacc[NK];
#pragma unroll
    for (int kb = 0; kb < NK; kb++) sacc[kb] = floatx4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < J; j++) {
      floatx4_t kf[NK];
#pragma unroll
      for (int kb = 0; kb < NK; kb++) kf[kb] = *reinterpret_cast<const floatx4_t *>(&Ks[k_frag_off + 16 * kb * LD + 16 * j]);
#pragma unroll
      for (int e = 0; e < 4; e++)
#pragma unroll
        for (int kb = 0; kb < NK; kb++) sacc[kb] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[kb][e], qf[j][e], sacc[kb], 0, 0, 0);
    }

    // ---- masking (diagonal tiles and the ragged last tile only) ----
    if ((k0 + BW > n_keys) || (CAUSAL && k0 + BW - 1 > wave_q_lo)) {
#pragma unroll
      for (int kb = 0; kb < NK; kb++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const int key = k0 + 16 * kb + 4 * g + i;
          if (key >= n_keys || (CAUSAL && key > qi)) sacc[kb][i] = -INFINITY;
        }
    }

    // ---- online softmax over the lane's 4 NK keys and the four lanes of a query ----
    float mx = sacc[0][0];
#pragma unroll
    for (int kb = 0; kb < NK; kb++)
#pragma unroll
      for (int i = 0; i < 4; i++) mx = fmaxf(mx, sacc[kb][i]);
    mx = max_over_wave_rows(mx);
    if (__builtin_amdgcn_ballot_w64((mx - m_i) * c > kLazyRescale) != 0) {  // wave-uniform
      const float m_new = fmaxf(m_i, mx);
      // (a key group's first tile may be hidden from some of the wave's rows: their max stays -inf)
      const float alpha = m_i == -INFINITY ? 0.f : __builtin_amdgcn_exp2f((m_i - m_new) * c);
      m_i = m_new;
      l_i *= alpha;
#pragma unroll
      for (int db = 0; db < J; db++) oacc[db] *= alpha;
    }
    const float mc = m_i == -INFINITY ? 0.f : m_i * c;
#pragma unroll
    for (int kb = 0; kb < NK; kb++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        sacc[kb][i] = __builtin_amdgcn_exp2f(sacc[kb][i] * c - mc);
        l_i += sacc[kb][i];
      }

    // ---- O^T += V^T P^T ----
#pragma unroll
    for (int kb = 0; kb < NK; kb++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const float *vrow = &Vs[v_frag_off + (16 * kb + i) * LD];
#pragma unroll
        for (int db = 0; db < J; db++) oacc[db] = __builtin_amdgcn_mfma_f32_16x16x4f32(vrow[16 * db], sacc[kb][i], oacc[db], 0, 0, 0);
      }
  }

  // ---- fold the other key groups' (m, l, O) into group 0's, lane for lane the same layout ----
  if constexpr (KG > 1) {
    constexpr int NF = J * 4 + 2;  // floats per lane
    static_assert((KG - 1) * RW * NF * 64 * 4 <= (int)(sizeof(Ks2)), "the partial results fit the K tiles");
    float *xch = &Ks2[0][0] + (wave % RW) * (NF * 64) + lane;  // [KG - 1][RW][NF][64 lanes]
    __syncthreads();  // every wave has read its last tile
    if (kg > 0) {
      float *w = xch + (kg - 1) * (RW * NF * 64);
      w[0] = m_i;
      w[64] = l_i;
#pragma unroll
      for (int db = 0; db < J; db++)
#pragma unroll
        for (int i = 0; i < 4; i++) w[(2 + db * 4 + i) * 64] = oacc[db][i];
    }
    __syncthreads();
    if (kg > 0) return;
    float m_all = m_i;
#pragma unroll
    for (int og = 0; og < KG - 1; og++) m_all = fmaxf(m_all, xch[og * (RW * NF * 64)]);
    // a group that saw no key has m = -inf, l = 0, O = 0
    const float a0 = m_i == -INFINITY ? 0.f : __builtin_amdgcn_exp2f((m_i - m_all) * c);
    l_i *= a0;
#pragma unroll
    for (int db = 0; db < J; db++) oacc[db] *= a0;
#pragma unroll
    for (int og = 0; og < KG - 1; og++) {
      const float *r = xch + og * (RW * NF * 64);
      const float a1 = r[0] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f((r[0] - m_all) * c);
      l_i += r[64] * a1;
#pragma unroll
      for (int db = 0; db < J; db++)
#pragma unroll
        for (int i = 0; i < 4; i++) oacc[db][i] += r[(2 + db * 4 + i) * 64] * a1;
    }
  }

  // ---- epilogue: out[qi][16 db + 4 g + i] = O^T / l ----
  const float l_tot = sum_over_wave_rows(l_i);
  const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
  if ((uint32_t)qi < (uint32_t)a.Sq) {
    float *op = reinterpret_cast<float *>(a.out) + b * a.os[0] + hq * a.os[1] + (int64_t)qi * a.os[2];
#pragma unroll
    for (int db = 0; db < J; db++) {
      const int d = 16 * db + 4 * g;
      if (d < a.D) *reinterpret_cast<float4 *>(op + d) = make_float4(oacc[db][0] * inv, oacc[db][1] * inv, oacc[db][2] * inv, oacc[db][3] * inv);
    }
  }
}

template <int D, int RW, int KG, int NK> constexpr int resident() {  // workgroups of a form that fit a CU
  const int by_lds = 160 * 1024 / (4 * 1024 * tile_blocks<D, RW, KG, NK>()), by_waves = (D > 128 ? 8 : 16) / (RW * KG);
  return by_lds < 1 ? 1 : by_lds < by_waves ? by_lds : by_waves;
}

// (dealing backwards: B=1 H=16 S=2048 D=128 causal in 64-row workgroups 218 -> 179 us, H=32 in 128-row ones 368 -> 283 us)
template <int D, int RW, int KG, int NK>
int launch_form(const PrefillArgs &a, hipStream_t stream) {
  const int n_q_tiles = (a.Sq + 16 * RW - 1) / (16 * RW);
  const int64_t wgs = deal_grid((int64_t)a.B * a.Hq, n_q_tiles);
  const int rc = check_grid(wgs, 64 * RW * KG);
  if (rc != LMH_OK) return rc;
  dim3 grid((uint32_t)wgs), block(64 * RW * KG);
  if (plan_only("prefill_f32_kernel<D=%d, %s, key groups=%d> rows=%d, workgroups=%u", D, a.causal ? "causal" : "full", KG, 16 * RW, grid.x))
    return LMH_OK;
  const Deal deal = make_deal(a.B, a.Hq, n_q_tiles, a.causal ? resident<D, RW, KG, NK>() : 0, device_cu_count());
  if (a.causal) hipLaunchKernelGGL((prefill_f32_kernel<D, true, RW, KG, NK>), grid, block, 0, stream, deal, a);
  else hipLaunchKernelGGL((prefill_f32_kernel<D, false, RW, KG, NK>), grid, block, 0, stream, deal, a);
  LMH_HIP_TRY(hipGetLastError());
  return LMH_OK;
}

// Expected time of a form: the walk of the busiest SIMD, in keys of one wave, times a weight for what the form pays per key
// (64-row workgroups = 1). Without a mask the workgroups are equal and go round in whole rounds of the CUs; causal ones end
// up near the mean of their lengths, a little above it where every one is resident from the start and by a quarter of the
// longest where they turn over. Causal launches with fewer than three waves per SIMD leave some of the LDS latency in sight,
// the equally long ones up to head dim 128 with fewer than two (D=96, B=1 H=16 S=1024: 64 rows, one wave, 70 us, 32 rows x 2 key groups, two,
// 68; B=1 H=32 S=1024: two waves in 128 rows 113, in 64 rows 116, four in 32 rows 122).
template <int D, int RW, int KG, int NK>
double form_cost(const PrefillArgs &a, double weight) {
  constexpr int tile = 16 * NK * KG;
  const double n_cus = device_cu_count();
  const int keys = a.causal && a.Sq < a.Sk ? a.Sq : a.Sk;
  const double wgs = (double)a.B * a.Hq * ((a.Sq + 16 * RW - 1) / (16 * RW));
  const double walk = (double)((keys + tile - 1) / tile) * tile / KG * (RW * KG / 4);
  const double occupancy = fmin(wgs / n_cus, resident<D, RW, KG, NK>()) * (RW * KG / 4);
  if (keys >= 256 && occupancy < (a.causal || D > 128 ? 3.0 : 2.0)) weight *= 1.15;
  if (!a.causal) return weight * walk * ceil(wgs / n_cus);
  const double mean = 0.5 * walk * wgs / n_cus;
  if (wgs <= n_cus) return weight * walk;
  return weight * (wgs <= resident<D, RW, KG, NK>() * n_cus ? 1.12 * fmax(walk, mean) : fmax(walk, mean + 0.25 * walk));
}

// The weights were taken from launches that fill the chip (S = 4096 causal D = 96: 128 rows 803 us, 64 rows 833, 32 rows x 2
// key groups 877 us, the same with two blocks of keys per wave and tile 1184, 16 rows x 4 key groups 1524); with up to one
// (causal: two) workgroups per CU the last two pay little of that.
template <int D>
int launch_for_d(const PrefillArgs &a, hipStream_t stream) {
  const int64_t n_cus = device_cu_count(), heads = (int64_t)a.B * a.Hq;
  auto tiles = [&](int rows) { return heads * ((a.Sq + rows - 1) / rows); };
  const double w32 = !a.causal && D > 96 ? 1.3 : 1.08;
  if constexpr (D > 128) {
    if (form_cost<D, 2, 2, 1>(a, w32) < form_cost<D, 4, 1, 1>(a, 1.0)) return launch_form<D, 2, 2, 1>(a, stream);
    return launch_form<D, 4, 1, 1>(a, stream);
  } else {
    // Without a mask, in blocks of 32 x 32 (prefill_f32_full.hip), where the head dim needs no more padding for it: a wave walks
    // twice the rows per key. Weights from launches that fill the chip (D=96, B=1 H=32 S=1024: 106 us against 113 for the
    // 128-row form here; D=128, two key groups on B=1 H=16 S=1024 78 against 89).
    constexpr bool kFull = D == 64 || D == 96 || D == 128;
    double f128 = INFINITY, f64 = INFINITY;
    if (kFull && !a.causal) {
      auto cost = [&](int rows, int tile, double weight) {
        return weight * (double)((a.Sk + tile - 1) / tile) * tile * (rows / 64) * ceil((double)tiles(rows) / n_cus);
      };
      f128 = cost(128, 32, 0.92);
      if (D == 128 && tiles(64) <= n_cus) f64 = cost(64, 64, 1.07);  // (narrower ones of more than 256 keys go over to the pieces)
    }
    const bool many = tiles(128) >= 4 * n_cus;
    const double c128 = form_cost<D, 8, 1, 2>(a, 0.96);
    // In pieces (prefill_f32_split.hip), up to head dim 96: by the time that the cost of the form here stands for, in us (a part
    // per launch, a part per key of the walk; fitted to 240 launches of drawn sizes, rms 2 to 13 %). Of 330 such launches 159 go
    // over, none loses more than 4 %, and together the 330 gain 12 %: B=2 H=12 S=1023 D=80 without a mask 76 -> 57 us, B=1 H=32
    // S=2048 D=96 380 -> 255, causal 214 -> 150, B=1 H=48 S=1100 D=64 causal 79 -> 58. The small launches stay because their waves
    // walk the keys alone (B=1 H=6 S=846 D=96 causal), and without a mask what the pieces would take less than 14.5 us for, where
    // the fit overrates the forms here: D=72 to 96 on up to 170 keys 4 to 14 us here, up to 2 times that there (H=12 502 x 167
    // D=72 13.5 and 14.0), while above it 55 of 60 drawn launches of up to 340 keys gain (20 x 300 x 119 D=80, B=4, 28.9 -> 21.2) and
    // the worst loses 7 % (H=4 1981 x 163 D=96, B=2, 16.3 and 17.5).
    // Above it, up to head dim 128, the same by a fit of each form's own (2300 launches, rms 2 to 11 %): where its cost stands for a time by one fit for all, an
    // error of 20 % counts for more than what the pieces gain on a launch of one round (B=8 H=12 S=189 D=128 causal 18.7 here and 22.6 in pieces, H=32 S=305,
    // B=2, 26.2 and 30.5). Of 2000 other drawn launches of head dims 104 to 128 (24 to 6000 workgroups, a third with lengths) 1168 go over: 29 % off all of
    // them together, 18 lose more than 5 %, the worst 11 % (B=9 H=8 S=219 without a mask, with lengths, 22.5 and 25.3); by one fit 55 lost that, up to 19 %.
    // Causal launches of one round are closest. Below 18 us by the estimate, a round of two key tiles, the other costs of a launch decide: they stay.
    enum Here { kC128, kC64, kC32, kC32x2, kC16, kF128, kF64 };
    auto pieces = [&](double here, Here which, int *form) {
      const double split = prefill_f32_split_cost(a, form);
      if constexpr (D > 96) {
        constexpr double fit[2][2][7][2] = {  // [D = 112, 128][causal][Here]
            {{{6.7, 0.0577}, {5.7, 0.0621}, {6.6, 0.0550}, {4.9, 0.0674}, {3.7, 0.0723}, {}, {}},
             {{11.4, 0.0550}, {11.8, 0.0545}, {10.7, 0.0530}, {8.1, 0.0599}, {6.0, 0.0636}, {}, {}}},
            {{{6.7, 0.0701}, {6.7, 0.0701}, {7.6, 0.0640}, {5.5, 0.0756}, {4.4, 0.0812}, {7.6, 0.0681}, {6.6, 0.0654}},
             {{16.2, 0.0614}, {19.1, 0.0590}, {11.7, 0.0604}, {7.6, 0.0709}, {5.7, 0.0768}, {}, {}}}};
        const auto &f = fit[D == 128][a.causal != 0][which];
        const bool close = D == 128 && a.causal && tiles(128) <= n_cus;
        return split >= 18.0 && split < (close ? 0.92 : 0.96) * (f[0] + f[1] * here);
      } else {
        constexpr double fit[5][2][2] = {{{6.6, 0.0178}, {4.3, 0.0197}}, {{6.1, 0.0249}, {5.1, 0.0277}}, {{5.6, 0.0352}, {5.7, 0.0351}},
                                         {{7.5, 0.0419}, {6.4, 0.0451}}, {{6.2, 0.0527}, {8.6, 0.0505}}};  // D = 32, 48, 64, 80, 96
        const auto &f = fit[D / 16 - 2][a.causal != 0];
        return (a.causal || split >= 14.5) && split < 0.95 * (f[0] + f[1] * here);
      }
    };
    int split_form = 0;
    if (many && (kFull && !a.causal ? pieces(f128, kF128, &split_form) : pieces(c128, kC128, &split_form))) return launch_prefill_f32_split(a, split_form, stream);
    if (many) return kFull && !a.causal ? launch_prefill_f32_full(a, 1, stream) : launch_form<D, 8, 1, 2>(a, stream);
    const bool few32 = tiles(32) <= (a.causal ? 2 : 1) * n_cus, few16 = tiles(16) <= 2 * n_cus;
    const double c64 = form_cost<D, 4, 1, 2>(a, 1.0), c32 = form_cost<D, 2, 2, 1>(a, w32),
                 c32x2 = form_cost<D, 2, 2, 2>(a, few32 ? 1.0 : D <= 64 ? 1.15 : 1.4), c16 = form_cost<D, 1, 4, 1>(a, few16 ? 1.2 : D <= 64 ? 1.5 : 1.8);
    const double best = fmin(fmin(c128, c64), fmin(fmin(c32, c32x2), c16));
    const Here which = fmin(f128, f64) < best ? (f64 < f128 ? kF64 : kF128) : best == c128 ? kC128 : best == c64 ? kC64 : best == c32 ? kC32 : best == c32x2 ? kC32x2 : kC16;
    if (pieces(fmin(best, fmin(f128, f64)), which, &split_form)) return launch_prefill_f32_split(a, split_form, stream);
    switch (which) {
      case kF128: return launch_prefill_f32_full(a, 1, stream);
      case kF64: return launch_prefill_f32_full(a, 2, stream);
      case kC128: return launch_form<D, 8, 1, 2>(a, stream);
      case kC64: return launch_form<D, 4, 1, 2>(a, stream);
      case kC32: return launch_form<D, 2, 2, 1>(a, stream);
      case kC32x2: return launch_form<D, 2, 2, 2>(a, stream);
      case kC16: break;
    }
    return launch_form<D, 1, 4, 1>(a, stream);
  }
}

}  // namespace

// (above 128 the head dims that are odd multiples of 8 stay on the vector-ALU kernel, as in prefill_mfma.hip)
bool prefill_f32_mfma_supported(int dtype, int D) { return dtype == LMH_F32 && D >= 8 && (D <= 128 ? D % 8 == 0 : D <= 256 && D % 16 == 0); }

int launch_prefill_f32_mfma(const PrefillArgs &a, hipStream_t stream) {
  if (a.D <= 32) return launch_for_d<32>(a, stream);
  if (a.D <= 48) return launch_for_d<48>(a, stream);
  if (a.D <= 64) return launch_for_d<64>(a, stream);
  if (a.D <= 80) return launch_for_d<80>(a, stream);
  if (a.D <= 96) return launch_for_d<96>(a, stream);
  if (a.D <= 112) return launch_for_d<112>(a, stream);
  if (a.D <= 128) return launch_for_d<128>(a, stream);
  if (a.D <= 160) return launch_for_d<160>(a, stream);
  if (a.D <= 192) return launch_for_d<192>(a, stream);
  if (a.D <= 256) return launch_for_d<256>(a, stream);
  return fail(LMH_E_UNSUPPORTED, "fp32 MFMA flash attention: head dim %d not tiled", a.D);
}

}  // namespace lmh
