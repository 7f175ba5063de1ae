// Flash attention forward in fp32 without a mask, in 32 x 32 blocks (v_mfma_f32_32x32x2_f32).
//
// The companion of prefill_f32.hip for launches whose workgroups are all equally long: where nothing has to be balanced and a
// round of workgroups fills the chip, the larger block wins, because it reads half as much from LDS per product (a 128-bit K
// fragment feeds 32 rows instead of 16, a V fragment as well) at the same rate of the matrix pipe. Measured, us, the best of the
// 16 x 16 forms against this file: B=1 H=32 S=1024 D=64 86 -> 76, D=96 113 -> 106, D=128 146 -> 136; H=8 S=4096 D=96 410 -> 404,
// D=128 537 -> 519; B=1 H=16 S=1024 (two key groups) D=128 89 -> 78. Where the rows or the head dim do not fill
// the blocks the smaller ones stay ahead (B=2 H=12 S=1023 D=96 105 here, 92 there; D=80 padded to 96 104 here, 94 there), and so
// they do under the causal mask; launch_for_d in prefill_f32.hip compares the two. Error against 64 bits: that of the 16 x 16 forms
// with as many key groups (0.99 to 1.00 of it over drawn shapes), 5 to 8e-7 in the 2-norm at 1000 to 2000 keys.
//
// Same structure as there: fp32 throughout, a wave owns 32 query rows with its Q fragments in registers, S^T = K Q^T so that a
// lane holds one query column, and the registers of P are the B operands of O^T = V^T P^T. The head dim is contracted in the
// order d = 8 j + 4 g + e (g: half of the wave), a 128-bit K fragment feeding four MFMAs; the keys so that MFMA i of a 32-key
// tile pairs key 8 (i / 4) + i % 4 from lanes 0-31 with the key four further from lanes 32-63.
#include "common.hpp"
#include "dtypes.hpp"
#include "rope.hpp"

namespace lmh {
namespace {

constexpr int BN = 32;    // keys a wave takes per tile
constexpr int kPadK = 4;  // floats: a row stride of D + 4 puts 16 consecutive rows' 16-byte reads on distinct banks
constexpr int kPadV = 8;  // floats: rows key and key + 4 (the two halves of a wave) land 32 banks apart
constexpr float kLog2e = 1.4426950408889634f;
constexpr int kOutOfRange = 0x7ffffff0;  // byte offset no K/V slice reaches: a buffer load there returns zeros
constexpr float kLazyRescale = 8.0f;     // the running max is raised only when outgrown by 2^8 (see prefill_mfma.hpp)
typedef float floatx4_t __attribute__((ext_vector_type(4)));

// KG = 1: the four waves own 4 x 32 query rows and walk the same 32-key tiles. KG = 2, for launches of at most one workgroup of
// 64 rows per CU: the waves own 2 x 32 rows, tiles have 64 keys, and each half of the waves takes 32 of them with a running max,
// sum and output of its own, folded through LDS at the end.
template <int D, int KG>
__global__ __launch_bounds__(256, (KG > 1 ? 1 : D <= 96 ? 3 : 2)) void prefill_f32_full_kernel(Deal deal, PrefillArgs a) {
  request_args(a);
  request_args(deal);
  constexpr int BM = 128 / KG;      // query rows per workgroup
  constexpr int BT = BN * KG;       // keys per staged tile
  constexpr int RG = 4 / KG;        // waves (32-row groups) per key group
  constexpr int KJ = D / 8;         // 128-bit K fragments per tile (4 MFMAs each)
  constexpr int DB = D / 32;        // 32-row blocks of O^T
  constexpr int LDK = D + kPadK;    // LDS row strides in floats
  constexpr int LDV = D + kPadV;
  constexpr int KC = LDK / 4, VC = LDV / 4;                          // 16-byte chunks per LDS row
  const int cpr = a.D / 4;  // the tensors' own head dim may be smaller than D: the missing columns are zeros, never stored

  constexpr int KI = (BT * KC + 63) / 64, VI = (BT * VC + 63) / 64;  // 1 KB blocks per tile (the last may be half used)
  __shared__ __attribute__((aligned(16))) float Ks2[2][KI * 256];     // double-buffered tiles, whole blocks
  __shared__ __attribute__((aligned(16))) float Vs2[2][VI * 256];

  // ---- which (b, hq, query tile) this workgroup owns ----
  int bh, q_tile;
  if (!deal_tile(deal, blockIdx.x & 7, blockIdx.x >> 3, &bh, &q_tile)) return;
  const int b = (int)((uint32_t)bh / deal.hq), hq = bh - b * a.Hq;
  const int kvh = kv_head_of(hq, a.Hq, a.Hkv, a.head_map);
  const int q0 = q_tile * BM;

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int n = lane & 31, g = lane >> 5;
  const int kg = wave / RG;  // key group of this wave (always 0 when KG == 1)
  const int qi = q0 + (wave % RG) * 32 + n;

  int n_keys = a.kv_len ? a.kv_len[b] : a.Sk;
  n_keys = min(max(n_keys, 0), a.Sk);
  const int n_kv_tiles = (n_keys + BT - 1) / BT;

  const float *qp = reinterpret_cast<const float *>(a.q) + b * a.qs[0] + hq * a.qs[1];
  const float *kp = reinterpret_cast<const float *>(a.k) + b * a.ks[0] + kvh * a.ks[1];
  const float *vp = reinterpret_cast<const float *>(a.v) + b * a.vs[0] + kvh * a.vs[1];

  // ---- Q fragments: lane (n, g) holds q[qi][8j + 4g .. + 3] for every j ----
  floatx4_t qf[KJ];
#pragma unroll
  for (int j = 0; j < KJ; j++) {
    float4 raw = make_float4(0.f, 0.f, 0.f, 0.f);
    if (qi < a.Sq && 8 * j + 4 * g < a.D) raw = *reinterpret_cast<const float4 *>(qp + (int64_t)qi * a.qs[2] + 8 * j + 4 * g);
    qf[j] = (floatx4_t){raw.x, raw.y, raw.z, raw.w};
  }

  floatx16_t oacc[DB];
#pragma unroll
  for (int db = 0; db < DB; db++)
#pragma unroll
    for (int i = 0; i < 16; i++) oacc[db][i] = 0.f;
  float m_i = -INFINITY;  // running max of the raw (unscaled) scores of query qi
  float l_i = 0.f;        // this lane's half of the running sum
  const float c = a.scale * kLog2e;

  // ---- tile staging, one tile ahead (see prefill_mfma.hip): lanes on a padding chunk, past the tile's last row or past the
  // tensors' head dim fetch out of range (zeros), rows past n_keys read as zero through the descriptor's bounds ----
  typedef int32_t i32x4_t __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) void lds_void_t;
  constexpr int KBW = (KI + 3) / 4, VBW = (VI + 3) / 4;  // blocks per wave (rounded up)
  const int wave_u = __builtin_amdgcn_readfirstlane(wave);
  __builtin_assume(wave_u >= 0 && wave_u < 4);
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
  int k_voff[KBW], v_voff[VBW];
#pragma unroll
  for (int j = 0; j < KBW; j++) {
    const int ch = (wave + 4 * j) * 64 + lane;
    const int row = ch / KC, col = ch % KC;
    k_voff[j] = (row < BT && col < cpr) ? (int)((row * a.ks[2] + col * 4) * 4) : kOutOfRange;
  }
#pragma unroll
  for (int j = 0; j < VBW; j++) {
    const int ch = (wave + 4 * j) * 64 + lane;
    const int row = ch / VC, col = ch % VC;
    v_voff[j] = (row < BT && col < cpr) ? (int)((row * a.vs[2] + col * 4) * 4) : kOutOfRange;
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
    for (int j = 0; j < KBW; j++)
      if (wave_u + 4 * j < KI) load_block(k_desc, k_lds0 + buf * (KI * 1024) + j * 4096, k_voff[j], kt * k_tile_bytes);
#pragma unroll
    for (int j = 0; j < VBW; j++)
      if (wave_u + 4 * j < VI) load_block(v_desc, v_lds0 + buf * (VI * 1024) + j * 4096, v_voff[j], kt * v_tile_bytes);
  };

  const int k_frag_off = n * LDK + 4 * g;  // + 8 * j
  const int v_frag_off = 4 * g * LDV + n;  // + (8 * (i / 4) + i % 4) * LDV + 32 * db

  if (n_kv_tiles > 0) load_tile(0, 0);
  // Rotary embedding of the query fragments in registers (PrefillArgs::q_rope; the head dim equals the tiling). Lane
  // (n, g) holds elements 8 j + 4 g + e: the partner j' + D/2 of element j' is fragment j + D/16 of the same lane, the
  // interleaved pairs are neighbours. inv_freq is computed once per workgroup into the second K buffer, which nothing
  // writes before the loop's first barrier.
  if (a.q_rope) {
    float *table = &Ks2[1][0];
    if (tid < D / 2) table[tid] = rope_inv_freq(tid, D, a.q_log2_base);
    __syncthreads();
    const float pos = (float)((a.q_pos0 ? a.q_pos0[b] : a.q_prev_seq) + qi);
    if (!a.q_interleaved) {
#pragma unroll
      for (int j = 0; j < KJ / 2; j++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
          float sn, cs, o0, o1;
          sincos_angle(pos * table[8 * j + 4 * g + e], &sn, &cs);
          rope_rotate(qf[j][e], qf[j + KJ / 2][e], sn, cs, &o0, &o1);
          qf[j][e] = o0;
          qf[j + KJ / 2][e] = o1;
        }
    } else {
#pragma unroll
      for (int j = 0; j < KJ; j++)
#pragma unroll
        for (int e = 0; e < 4; e += 2) {
          float sn, cs, o0, o1;
          sincos_angle(pos * table[(8 * j + 4 * g + e) / 2], &sn, &cs);
          rope_rotate(qf[j][e], qf[j][e + 1], sn, cs, &o0, &o1);
          qf[j][e] = o0;
          qf[j][e + 1] = o1;
        }
    }
  }
  // The compiler does not model the asm loads or the asm wait below: make it wait for Q here, not inside the loop.
#pragma unroll
  for (int j = 0; j < KJ; j++) asm volatile("" :: "v"(qf[j]));

  for (int kt = 0; kt < n_kv_tiles; kt++) {
    // One barrier per tile: tile kt (fetched during the previous iteration) becomes visible, and every
    // wave is done with tile kt-1, whose buffer the fetch of tile kt+1 now overwrites.
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's blocks of tile kt are in LDS
    __syncthreads();
    if (kt + 1 < n_kv_tiles) load_tile(kt + 1, (kt + 1) & 1);
    const float *Ks = Ks2[kt & 1] + kg * (BN * LDK);
    const float *Vs = Vs2[kt & 1] + kg * (BN * LDV);

    const int k0 = kt * BT + kg * BN;         // first key of this wave's share of the tile
    if (KG > 1 && k0 >= n_keys) continue;     // all of it past the last key

    // ---- S^T = K Q^T: 32 keys x 32 queries, contraction over the head dim two elements per MFMA ----
    floatx16_t sacc;
#pragma unroll
    for (int i = 0; i < 16; i++) sacc[i] = 0.f;
#pragma unroll
    for (int j = 0; j < KJ; j++) {
      const floatx4_t kf = *reinterpret_cast<const floatx4_t *>(&Ks[k_frag_off + 8 * j]);
#pragma unroll
      for (int e = 0; e < 4; e++) sacc = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[e], qf[j][e], sacc, 0, 0, 0);
    }

    if (k0 + BN > n_keys) {  // the ragged last tile
#pragma unroll
      for (int i = 0; i < 16; i++)
        if (k0 + 8 * (i >> 2) + 4 * g + (i & 3) >= n_keys) sacc[i] = -INFINITY;
    }

    // ---- online softmax; all statistics are per lane (one query column) ----
    float mx = sacc[0];
#pragma unroll
    for (int i = 1; i < 16; i++) mx = fmaxf(mx, sacc[i]);
    mx = max_over_wave_halves(mx);
    if (__builtin_amdgcn_ballot_w64((mx - m_i) * c > kLazyRescale) != 0) {  // wave-uniform
      const float m_new = fmaxf(m_i, mx);
      const float alpha = m_i == -INFINITY ? 0.f : __builtin_amdgcn_exp2f((m_i - m_new) * c);
      m_i = m_new;
      l_i *= alpha;
#pragma unroll
      for (int db = 0; db < DB; db++)
#pragma unroll
        for (int i = 0; i < 16; i++) oacc[db][i] *= alpha;
    }
    const float mc = m_i == -INFINITY ? 0.f : m_i * c;
    float l0 = 0.f, l1 = 0.f;
#pragma unroll
    for (int i = 0; i < 16; i += 2) {
      sacc[i] = __builtin_amdgcn_exp2f(sacc[i] * c - mc);
      sacc[i + 1] = __builtin_amdgcn_exp2f(sacc[i + 1] * c - mc);
      l0 += sacc[i];
      l1 += sacc[i + 1];
    }
    l_i += l0 + l1;

    // ---- O^T += V^T P^T: MFMA i contracts the two keys lanes (., 0) and (., 1) hold in register i ----
#pragma unroll
    for (int i = 0; i < 16; i++) {
      const float *vrow = &Vs[v_frag_off + (8 * (i >> 2) + (i & 3)) * LDV];
#pragma unroll
      for (int db = 0; db < DB; db++) oacc[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(vrow[32 * db], sacc[i], oacc[db], 0, 0, 0);
    }
  }

  // ---- fold the second key group's (m, l, O) into the first's; lane for lane the same layout ----
  if constexpr (KG > 1) {
    static_assert(KG == 2, "one partial result per row");
    constexpr int NF = DB * 16 + 2;  // floats per lane
    static_assert(RG * NF * 64 * 4 <= (int)sizeof(Ks2), "the partial results fit the K tiles");
    float *xch = &Ks2[0][0] + (wave % RG) * (NF * 64) + lane;  // [RG][NF][64 lanes]
    __syncthreads();  // every wave has read its last tile
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
    // a group that saw no key has m = -inf, l = 0, O = 0
    const float a0 = m_i == -INFINITY ? 0.f : __builtin_amdgcn_exp2f((m_i - m_all) * c);
    const float a1 = m1 == -INFINITY ? 0.f : __builtin_amdgcn_exp2f((m1 - m_all) * c);
    l_i = l_i * a0 + xch[64] * a1;
#pragma unroll
    for (int db = 0; db < DB; db++)
#pragma unroll
      for (int i = 0; i < 16; i++) oacc[db][i] = oacc[db][i] * a0 + xch[(2 + db * 16 + i) * 64] * a1;
  }

  // ---- epilogue: out[qi][d] = O^T[d][qi] / l ----
  const float l_tot = sum_over_wave_halves(l_i);
  const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
  if (qi < a.Sq) {
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

template <int D, int KG>
int launch_form(const PrefillArgs &a, hipStream_t stream) {
  const int n_q_tiles = (a.Sq + 128 / KG - 1) / (128 / KG);
  const int64_t wgs = deal_grid((int64_t)a.B * a.Hq, n_q_tiles);
  const int rc = check_grid(wgs, 256);
  if (rc != LMH_OK) return rc;
  dim3 grid((uint32_t)wgs), block(256);
  if (plan_only("prefill_f32_full_kernel<D=%d, key groups=%d> rows=%d, workgroups=%u", D, KG, 128 / KG, grid.x)) return LMH_OK;
  const Deal deal = make_deal(a.B, a.Hq, n_q_tiles, 0, device_cu_count());
  hipLaunchKernelGGL((prefill_f32_full_kernel<D, KG>), grid, block, 0, stream, deal, a);
  LMH_HIP_TRY(hipGetLastError());
  return LMH_OK;
}

}  // namespace

int launch_prefill_f32_full(const PrefillArgs &a, int key_groups, hipStream_t stream) {
  if (a.D <= 64) return launch_form<64, 1>(a, stream);
  if (a.D <= 96) return launch_form<96, 1>(a, stream);
  return key_groups == 2 ? launch_form<128, 2>(a, stream) : launch_form<128, 1>(a, stream);
}

}  // namespace lmh
