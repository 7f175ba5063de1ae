// Flash attention forward on the gfx950 matrix cores (fp16 / bf16 in, fp32 accumulate).
//
// Same mathematics as flash_attn_cpu (reference src/Execution.jl:453-479) — online softmax with a
// running max m, running sum l and an un-normalised output row — evaluated 64 keys at a time for
// 128 or 256 query rows per workgroup instead of one (i, j) pair at a time.
//
// Tiling (wave64, v_mfma_f32_32x32x16):
//   * workgroup = 4 waves = 128 query rows of one (b, hq) (8 waves = 256 rows in launches large
//     enough to stay balanced with them); each wave owns 32 query rows and keeps their Q
//     fragments in registers for the whole kernel;
//   * the scores are computed TRANSPOSED, S^T = K Q^T (M = keys, N = queries). In the MFMA
//     accumulator layout a lane then holds one query column (n = lane % 32) and 16 of the 32 keys
//     of a block, so the softmax statistics (max, sum, rescale factor) are per-lane scalars and
//     the only cross-lane traffic is one exchange with lane ^ 32;
//   * the same registers, converted to half precision, are directly the B operand of the second
//     product O^T = V^T P^T (M = head dim, N = queries, contraction over keys), so P never
//     touches LDS;
//   * K and V tiles (64 keys) go from global memory straight into double-buffered LDS, row-major,
//     with LDS-writing buffer loads (no register staging, no LDS store instructions); the K
//     fragment is a plain 128-bit LDS read (contraction over the contiguous head dim), the V^T
//     fragment uses the gfx950 transposing LDS read ds_read_b64_tr_b16, which hands each lane 4
//     consecutive keys of its head-dim column;
//   * causal: key tiles beyond the workgroup's last query are never loaded, a wave skips tiles that
//     lie entirely above its diagonal, and only diagonal tiles pay for masking;
//   * blockIdx -> work mapping keeps all query tiles of a head on one XCD (private L2) and, for
//     causal, issues the long rows first.
#include <math.h>

#include <algorithm>
#include <type_traits>

#include "prefill_mfma.hpp"
#include "rope.hpp"

#if (defined(LMH_FOLD_SCALE) || defined(LMH_ONLY_XCDS) || defined(LMH_WIDE_MARGIN) || defined(LMH_W64_KERNEL) || defined(LMH_NO_PAIR_KERNEL) || \
     defined(LMH_BF16_SPLIT_P) || defined(LMH_NO_MIXED_KEY_GROUPS)) && \
    !defined(LMH_MEASUREMENT_BUILD)
#error "LMH_FOLD_SCALE / LMH_ONLY_XCDS / LMH_WIDE_MARGIN / LMH_W64_KERNEL / LMH_NO_PAIR_KERNEL / LMH_BF16_SPLIT_P / LMH_NO_MIXED_KEY_GROUPS are experiment switches: they need -DLMH_MEASUREMENT_BUILD, which marks the library"
#endif

#ifndef LMH_WIDE_MARGIN
#define LMH_WIDE_MARGIN 0.9
#endif

namespace lmh {
namespace {


// Rotary embedding of the wave's query fragments in registers (PrefillArgs::q_rope). Lane (n, g) holds elements
// 16 ks + 8 g + e of its row; with the head dim equal to the tiling, the partner j + D/2 of element j sits in
// fragment ks + D/32 of the same lane (the interleaved pairs are neighbours inside a fragment). inv_freq does not
// depend on the row: the workgroup computes its D/2 values once into `table` (LDS that nothing else uses before the
// next barrier) and every lane multiplies them by its own position. Every thread of the workgroup must call this.
template <typename MT, int D>
__device__ inline void rotate_q_fragments_with_table(typename MT::vec8 (&qreg)[D / 16], const PrefillArgs &a, int b, int qi, int g, const float *table);
template <typename MT, int D>
__device__ inline void rotate_q_fragments(typename MT::vec8 (&qreg)[D / 16], const PrefillArgs &a, int b, int qi, int g, float *table) {
  if ((int)threadIdx.x < D / 2) table[threadIdx.x] = rope_inv_freq(threadIdx.x, D, a.q_log2_base);
  __syncthreads();
  rotate_q_fragments_with_table<MT, D>(qreg, a, b, qi, g, table);
}
// the rotation itself, given the workgroup's table of D / 2 inverse frequencies
template <typename MT, int D>
__device__ inline void rotate_q_fragments_with_table(typename MT::vec8 (&qreg)[D / 16], const PrefillArgs &a, int b, int qi, int g, const float *table) {
  constexpr int KS = D / 16, HK = D / 32;
  const float pos = (float)((a.q_pos0 ? a.q_pos0[b] : a.q_prev_seq) + qi);
  if (!a.q_interleaved) {
#pragma unroll
    for (int ks = 0; ks < HK; ks++)
#pragma unroll
      for (int e = 0; e < 8; e++) {
        float sn, cs, o0, o1;
        sincos_angle(pos * table[16 * ks + 8 * g + e], &sn, &cs);
        rope_rotate((float)qreg[ks][e], (float)qreg[ks + HK][e], sn, cs, &o0, &o1);
        qreg[ks][e] = MT::cvt(o0);
        qreg[ks + HK][e] = MT::cvt(o1);
      }
  } else {
#pragma unroll
    for (int ks = 0; ks < KS; ks++)
#pragma unroll
      for (int e = 0; e < 8; e += 2) {
        float sn, cs, o0, o1;
        sincos_angle(pos * table[(16 * ks + 8 * g + e) / 2], &sn, &cs);
        rope_rotate((float)qreg[ks][e], (float)qreg[ks][e + 1], sn, cs, &o0, &o1);
        qreg[ks][e] = MT::cvt(o0);
        qreg[ks][e + 1] = MT::cvt(o1);
      }
  }
}

// NW waves per workgroup, 32 query rows each, walking the same 64-key tiles (KSPLIT = 1).
// NW = 8 (256 query rows) stages every K/V tile once per 256 rows instead of once per 128: 3-8 % faster
// wherever there are enough workgroups to keep the balance. Head dims up to 96: two such workgroups =
// 4 waves per SIMD on a CU, at most 128 registers. D = 128: one workgroup per CU, 2 waves per SIMD, as
// with the 128-row workgroups there.
// KSPLIT = 2: for launches too small to fill the chip. The workgroup owns 64 query rows; waves 0-1
// take them against the first 32 keys of every tile, waves 2-3 against the second 32, each pair
// with its own running max / sum / output, merged through LDS at the end. Twice the workgroups,
// and a wave's share of a tile is half as long. With NW = 8 (head dims above 128) the workgroup owns 128 rows: the two
// waves of a SIMD hide each other's LDS latency.
// KSPLIT = 4 and 8: for launches that leave CUs without a workgroup or with one only. What bounds those is the serial chain of a
// wave, a fetch, two products and a softmax per tile (0.46 us for a tile of 64 keys at head dim 64 in two key groups, where its MFMAs
// take 0.1), so a tile is four or eight groups of 32 keys, and a wave walks a quarter or an eighth of the keys. 64 rows on eight waves,
// at head dims up to 64 also 32 rows on four or, with tiles of 256 keys, on eight, which no CU holds more than once. The groups are
// folded two by two. fp16, us in two groups and here: 1 x 2 heads 988 x 7818 D=128 97.6 and 72.1, B=6 H=1 S=1295 D=64 causal 14.1 and 10.3, H=4
// S=4066 D=40 causal 35.4 and 23.5, H=3 S=3910 D=64 causal 33.9 and 19.8, 24 x 7127 keys of 18 rows 57.6 and 29.9; bf16 H=8 S=3169 D=64
// causal 38.3 and 30.5. (32 rows on four waves at head dims 96 and 128: 0 to 25 % behind 64 rows on eight, one wave per SIMD.)
// The second launch bound is waves per SIMD.
// WPS: waves per SIMD the register budget is set for (3 x 4 waves, 2 x 8 waves or 1 x 8 waves per CU).
template <int D, int NW> constexpr int default_wps() { return D > 128 ? 1 : D > 96 ? 2 : NW == 8 ? 4 : 3; }
// AHEAD: the loop that is a tile ahead with its scores, for one wave per SIMD.
// HEADS = 2: the waves' second half takes the same rows of another query head of the KV head, so that a tile is staged, and in bf16 rewritten
// as fp16, once for both, in row tiles half as high as NW waves of one head have. B=3 H=32/8 S=1337 D=128 causal fp16 61.2 -> 57.4 us, bf16
// 70.5 -> 67.0 (ragged 65.8 -> 64.0), a prompt of B=4 T=777 fp16 54.9 -> 51.8.
template <typename MT, int D, bool CAUSAL, int KSPLIT, int NW, int WPS, bool AHEAD, int HEADS = 1>
__global__ __launch_bounds__(64 * NW, WPS) void prefill_mfma_kernel(Deal deal, PrefillArgs a, QueryCopy queries) {
  request_args(a);
  request_args(deal);
  using vec8 = typename MT::vec8;
  constexpr int BM = 32 * NW / KSPLIT / HEADS;  // query rows per workgroup
  // keys per staged tile: 64; 128 where one workgroup has the CU to itself and LDS and registers allow (half the
  // barriers and per-tile bookkeeping: 114.2 -> 111.9 us on B=1 H=32 S=4096 causal)
  constexpr int BT = KSPLIT == 8 ? 4 * BN : (NW == 8 && WPS == 2 && D <= 96 && KSPLIT == 1) || KSPLIT == 4 ? 2 * BN : BN;
  constexpr int RG = NW / KSPLIT;   // waves (32-row groups) per key group
  constexpr int RH = RG / HEADS;    // ... and of a head
  constexpr int NKB = BT / 32 / KSPLIT;   // 32-key blocks a wave takes per tile
  constexpr int BW = 32 * NKB;      // ... in keys
  constexpr int KS = D / 16;       // k-steps of the S^T product
  constexpr int DB = D / 32;       // 32-row blocks of O^T
  // D is the tiled head dim; the tensors' own head dim a.D may be smaller (any multiple of 8): the
  // missing columns are never fetched (zeros in Q, K and V) and never stored.
  const int cpr = a.D / 8;         // 16-byte chunks per K/V row in memory
  constexpr bool CV = MT::kConvertV;  // V tiles rewritten as fp16 on their way into LDS
  using pvec8 = typename MT::pvec8;
  constexpr int LDK = D + kPadK;   // LDS row strides in elements
  constexpr int LDV = D + pad_v<D>();
  // Forms whose loop takes every register there is: what the masks and the stores need is made where they are, for what is held over the
  // loop goes to memory in front of it and comes back behind it, with a wait for every load. us before 16-byte stores and masks of one
  // compare, with both and now: 12 x 16 heads Sq=3300 Sk=20 D=96 bf16 69.7, 61.5, 52.8 (fp32 results 105.8, 110.8, 92.9), 6 x 32 Sq=2019 Sk=138
  // 64.3, 62.2, 54.7, 14 x 20 Sq=1813 Sk=500 D=80 169.0, 173.0, 164.6, V as fp16 15 x 32 Sq=323 Sk=1393 175.6, 175.2, 160.9, causal 15 x 32/8
  // S=709 D=72 96.4, 96.5, 92.5; fp16 7 x 32/8 Sq=3000 Sk=60 fp32 results 100.0, 113.1, 99.7.
  constexpr bool TIGHT = D == 96 && (WPS == 4 || (CV && !CAUSAL));

  // Head dims above 128 in four key groups: the LDS holds one tile of 128 keys. Its K is fetched beside the second product of the tile
  // before and its V beside the first product and the softmax, with a barrier in front of either.
  constexpr bool IN_TURN = D > 128 && KSPLIT == 4;
  constexpr int RING = 3;  // fragments in flight there (left to itself the compiler reads one, waits, multiplies; four: 2 % slower, or spills)

  __shared__ __attribute__((aligned(16))) uint16_t Ks2[IN_TURN ? 1 : 2][BT * LDK];  // double-buffered tiles
  __shared__ __attribute__((aligned(16))) uint16_t Vs2[IN_TURN ? 1 : 2][BT * LDV];

#ifdef LMH_ONLY_XCDS
  // Measurement build (results wrong by construction): only workgroups dispatched to the first LMH_ONLY_XCDS XCDs
  // work, the rest exit at once — the same instruction stream with part of the chip idle.
  if ((blockIdx.x & 7) >= LMH_ONLY_XCDS) return;
#endif
  // ---- which (b, hq, query tile) this workgroup owns ----
  int bh, tile_rank;
  if (!deal_tile(deal, blockIdx.x & 7, blockIdx.x >> 3, &bh, &tile_rank)) return;
  const int b = (int)((uint32_t)bh / deal.hq);
  int hq = bh - b * (a.Hq / HEADS), hq_step = 0;  // the (first) query head; with HEADS = 2 the waves' second half takes another one
  if constexpr (HEADS == 2) {  // hq counts the pairs of heads of one KV head
    hq_step = a.head_map == LMH_HEADMAP_BLOCKED ? 1 : a.Hkv;
    hq = a.head_map == LMH_HEADMAP_BLOCKED ? 2 * hq : hq + hq / a.Hkv * a.Hkv;
  }
  const int kvh = kv_head_of(hq, a.Hq, a.Hkv, a.head_map);
  // Causal rows grow with the query index: long rows are issued first so that the short ones fill
  // the tail of the launch. (Pairing tile r with tile n-1-r in one workgroup equalises the work but
  // halves the number of workgroups; measured 15 % slower on the S = 4096 workload.)
  const int q_tile = CAUSAL ? (deal.tiles - 1 - tile_rank) : tile_rank;
  const int q0 = q_tile * BM - (CAUSAL ? causal_shift(deal.tiles, BM, a.Sq, BT) : 0);

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int n = lane & 31, g = lane >> 5;
  const int kg = wave / RG;  // key group of this wave (always 0 when KSPLIT == 1)
  const int wave_q_lo = q0 + (wave % RH) * 32;
  const int own_hq = HEADS == 1 ? hq : hq + __builtin_amdgcn_readfirstlane(wave % RG / RH) * hq_step;
  const int wave_q_hi = wave_q_lo + 31;
  const int qi = wave_q_lo + n;

  int n_keys = a.kv_len ? a.kv_len[b] : a.Sk;
  n_keys = min(max(n_keys, 0), a.Sk);
  int k_end = n_keys;
  if (CAUSAL) k_end = min(k_end, q0 + BM);
  const int n_kv_tiles = (k_end + BT - 1) / BT;

  const uint16_t *qp = reinterpret_cast<const uint16_t *>(a.q) + b * a.qs[0] + own_hq * a.qs[1];
  const uint16_t *kp = reinterpret_cast<const uint16_t *>(a.k) + b * a.ks[0] + kvh * a.ks[1];
  const uint16_t *vp = reinterpret_cast<const uint16_t *>(a.v) + b * a.vs[0] + kvh * a.vs[1];

  // ---- Q fragments: B operand of S^T = K Q^T; lane (n, g) holds q[qi][16*ks + 8*g .. +7] ----
  vec8 qreg[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ks++) {
    uint4 raw = make_uint4(0, 0, 0, 0);
    if ((uint32_t)qi < (uint32_t)a.Sq && 16 * ks + 8 * g < a.D) raw = *reinterpret_cast<const uint4 *>(qp + (int64_t)qi * a.qs[2] + 16 * ks + 8 * g);
    qreg[ks] = __builtin_bit_cast(vec8, raw);
#ifdef LMH_FOLD_SCALE
    // Measurement build, not the shipped path: scale * log2(e) multiplied into the Q fragments (rounded to the element
    // type once more), the running max kept in log2 units and handed to the first QK^T MFMA of a block as its
    // accumulator input, so that the MFMAs deliver the argument of exp2 and the per-score v_fma disappears. The extra
    // rounding moves a logit by up to 2^-12 of its magnitude: 1.5e-4 of the output range at a row max of 4 (log2 units),
    // 4.5e-4 at 16, 1.5e-3 at 45, over the 2e-3 budget at a few hundred (the large-logit parity tests fail).
#pragma unroll
    for (int e = 0; e < 8; e++) qreg[ks][e] = MT::cvt((float)qreg[ks][e] * (a.scale * kLog2e));
#endif
  }

  floatx16_t oacc[DB];
#pragma unroll
  for (int db = 0; db < DB; db++)
#pragma unroll
    for (int i = 0; i < 16; i++) oacc[db][i] = 0.f;
  float m_i = -INFINITY;  // running max of the raw (unscaled) scores of query qi
  float l_i = 0.f;        // this lane's half of the running sum
  const float c = a.scale * kLog2e;
#ifdef LMH_FOLD_SCALE
  float neg_mc = 0.f;     // minus the running max, in log2 units ...
  floatx16_t neg_mc16;    // ... and as the accumulator input of a block's first MFMA (rewritten only when the max is raised)
#pragma unroll
  for (int i = 0; i < 16; i++) neg_mc16[i] = 0.f;
  bool have_m = false;
#endif

  // ---- tile staging: global memory -> LDS directly (buffer_load_dwordx4 ... lds), one tile ahead ----
  // A tile of BT rows x LD elements is BT * LD / 512 blocks of 1 KB. One wave-wide load fills one block:
  // lane l's 16 bytes land at block + 16 l, fetched from that lane's own global offset, so the
  // padded row layout needs no register staging and no LDS store instructions. Lanes that fall on
  // a padding chunk fetch out of range. The descriptor's size is the end of the last valid key row:
  // rows past n_keys arrive as zeros without a branch, and the per-lane offsets are loop
  // invariants. Wave w issues blocks w, w + NW, ...
  // The load is written in asm because the compiler, when it knows of an LDS-writing load in
  // flight, waits for it before the next LDS read of the same array — which would serialise the
  // prefetch of tile kt + 1 with the fragment reads of tile kt. The wait that matters (this wave's
  // loads have landed, then the workgroup barrier) is written out at the top of the loop.
  typedef int32_t i32x4_t __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) void lds_void_t;
  constexpr int KC = LDK / 8, VC = LDV / 8;            // 16-byte chunks per LDS row
  constexpr int KI = KC * BT / 64, VI = VC * BT / 64;  // 1 KB blocks per tile
  constexpr int KJ = (KI + NW - 1) / NW, VJ = (VI + NW - 1) / NW;  // blocks per wave (rounded up)
  const int wave_u = __builtin_amdgcn_readfirstlane(wave);
  __builtin_assume(wave_u >= 0 && wave_u < NW);
  auto make_desc = [](const uint16_t *base, int bytes) {
    const uint64_t p = (uint64_t)base;
    i32x4_t d;
    d[0] = __builtin_amdgcn_readfirstlane((int)(uint32_t)p);
    d[1] = __builtin_amdgcn_readfirstlane((int)((p >> 32) & 0xffff));  // stride 0: raw buffer
    d[2] = __builtin_amdgcn_readfirstlane(bytes);
    d[3] = 0x00020000;
    return d;
  };
  const i32x4_t k_desc = make_desc(kp, (int)((int64_t)n_keys * a.ks[2] * 2));
  const i32x4_t v_desc = make_desc(vp, (int)((int64_t)n_keys * a.vs[2] * 2));
  int k_voff[KJ], v_voff[VJ];
#pragma unroll
  for (int j = 0; j < KJ; j++) {
    const int ch = (wave + NW * j) * 64 + lane;
    const int row = ch / KC, col = ch % KC;
    k_voff[j] = col < cpr ? (int)((row * a.ks[2] + col * 8) * 2) : kOutOfRange;
  }
#pragma unroll
  for (int j = 0; j < VJ; j++) {
    const int ch = (wave + NW * j) * 64 + lane;
    const int row = ch / VC, col = ch % VC;
    v_voff[j] = col < cpr ? (int)((row * a.vs[2] + col * 8) * 2) : kOutOfRange;
  }
  const int k_tile_bytes = (int)(BT * a.ks[2] * 2), v_tile_bytes = (int)(BT * a.vs[2] * 2);
  const uint32_t k_lds0 = (uint32_t)(uintptr_t)(lds_void_t *)&Ks2[0][0] + wave_u * 1024;
  const uint32_t v_lds0 = (uint32_t)(uintptr_t)(lds_void_t *)&Vs2[0][0] + wave_u * 1024;
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"  // m0 is a reserved register; it is only written here
  auto load_block = [](i32x4_t desc, uint32_t lds_addr, int voff, int soff) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 :: "s"(lds_addr), "v"(voff), "s"(desc), "s"(soff) : "memory", "m0");
  };
#pragma clang diagnostic pop
  auto load_k_block = [&](int kt, int buf, int j) __attribute__((always_inline)) {
    if (wave_u + NW * j < KI)
      load_block(k_desc, k_lds0 + buf * (BT * LDK * 2) + j * (NW * 1024), k_voff[j], kt * k_tile_bytes);
  };
  auto load_v_block = [&](int kt, int buf, int j) __attribute__((always_inline)) {
    if (wave_u + NW * j < VI)
      load_block(v_desc, v_lds0 + buf * (BT * LDV * 2) + j * (NW * 1024), v_voff[j], kt * v_tile_bytes);
  };
  auto load_k = [&](int kt, int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < KJ; j++) load_k_block(kt, buf, j);
  };
  auto load_v = [&](int kt, int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < VJ; j++) load_v_block(kt, buf, j);
  };
  auto load_tile = [&](int kt, int buf) __attribute__((always_inline)) {
    load_k(kt, buf);
    if constexpr (!CV && !IN_TURN) load_v(kt, buf);
  };

  // ---- MT::kConvertV: V tiles pass through registers and are stored in LDS as fp16 relative to the largest finite |v|
  // met so far. Tile kt + 1 is rewritten during iteration kt from registers loaded during iteration kt - 1; the
  // workgroup agrees on the largest value through v_top[parity of the tile], posted before the tile's barrier (only by
  // threads whose own largest exponent exceeds what they already know of) and read by everyone after it. A slot is
  // posted to again two barriers later, after every thread has read it, and never shrinks. ----
  constexpr int DC = D / 8;                                              // 16-byte chunks per tiled V row
  constexpr int VR = CV ? (BT * DC + 64 * NW - 1) / (64 * NW) : 1;       // chunks per thread and tile
  __shared__ uint32_t v_top[2];
  uint4 vreg[VR];
  int vr_voff[VR], vr_lds[VR];
  uint32_t top_run = 0;    // largest finite |v| bits up to the tile last rewritten (the same in every thread)
  int thr_next = 0, thr_cur = 0, thr_acc = 0;  // exponent base of the tile last rewritten / in use / of the accumulators
  bool v_special = false;  // this thread's registers hold an infinity or a NaN
  const __amdgpu_buffer_rsrc_t v_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t *>(vp), 0, __builtin_amdgcn_readfirstlane((int)((int64_t)n_keys * a.vs[2] * 2)), 0x00020000);
  if constexpr (CV) {
#pragma unroll
    for (int j = 0; j < VR; j++) {
      const int ch = tid + j * (64 * NW);
      const int row = ch / DC, col = ch % DC;
      vr_voff[j] = (ch < BT * DC && col < cpr) ? (int)((row * a.vs[2] + col * 8) * 2) : kOutOfRange;
      vr_lds[j] = (row * LDV + col * 8) * 2;
    }
  }
  auto fetch_v = [&](int kt) {
    const int soff = __builtin_amdgcn_readfirstlane(kt * v_tile_bytes);
#pragma unroll
    for (int j = 0; j < VR; j++) vreg[j] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(v_rsrc, vr_voff[j], soff, 0));
  };
  auto post_top = [&](int slot) {
    // (four at a time: a packed maximum that waits for the one before it costs two instructions)
    u16x2_t part[4] = {{0, 0}, {0, 0}, {0, 0}, {0, 0}};
#pragma unroll
    for (int j = 0; j < VR; j++) {
      const uint32_t w[4] = {vreg[j].x, vreg[j].y, vreg[j].z, vreg[j].w};
#pragma unroll
      for (int e = 0; e < 4; e++) part[e] = __builtin_elementwise_max(part[e], __builtin_bit_cast(u16x2_t, w[e] & 0x7fff7fffu));
    }
    const u16x2_t all = __builtin_elementwise_max(__builtin_elementwise_max(part[0], part[1]), __builtin_elementwise_max(part[2], part[3]));
    uint32_t m = max((uint32_t)all[0], (uint32_t)all[1]);
    v_special = m >= 0x7f80u;
    if (v_special) {
      m = 0;
#pragma unroll
      for (int j = 0; j < VR; j++) {
        m = bf16x2_finite_top(vreg[j].x, m);
        m = bf16x2_finite_top(vreg[j].y, m);
        m = bf16x2_finite_top(vreg[j].z, m);
        m = bf16x2_finite_top(vreg[j].w, m);
      }
    }
    if ((m >> 7) > (top_run >> 7)) atomicMax(&v_top[slot], m);
  };
  auto rewrite_v = [&](int buf) {  // after the barrier that follows post_top(buf)
    top_run = max(top_run, v_top[buf]);
    thr_next = max((int)(top_run >> 7) - 29, 0);
    const uint32_t tb2 = ((uint32_t)thr_next << 7) * 0x00010001u;
    char *dst = reinterpret_cast<char *>(&Vs2[buf][0]);
    uint4 o[VR];
#pragma unroll
    for (int j = 0; j < VR; j++)
      o[j] = make_uint4(bf16x2_to_scaled_f16x2(vreg[j].x, tb2), bf16x2_to_scaled_f16x2(vreg[j].y, tb2),
                        bf16x2_to_scaled_f16x2(vreg[j].z, tb2), bf16x2_to_scaled_f16x2(vreg[j].w, tb2));
    if (v_special) {
#pragma unroll
      for (int j = 0; j < VR; j++)
        o[j] = make_uint4(bf16x2_to_scaled_f16x2_any(vreg[j].x, tb2), bf16x2_to_scaled_f16x2_any(vreg[j].y, tb2),
                          bf16x2_to_scaled_f16x2_any(vreg[j].z, tb2), bf16x2_to_scaled_f16x2_any(vreg[j].w, tb2));
    }
#pragma unroll
    for (int j = 0; j < VR; j++) {
      if ((BT * DC) % (64 * NW) != 0 && tid + j * (64 * NW) >= BT * DC) continue;
      *reinterpret_cast<uint4 *>(dst + vr_lds[j]) = o[j];
    }
  };

  // lane-constant pieces of the LDS addresses
  const int k_frag_off = n * LDK + 8 * g;  // + kb*32*LDK + 16*ks
  // transposing V read: within each 16-lane block, lane i supplies row (i / 4) and 4-column group
  // (i % 4) of a 4-key x 16-column patch and receives the 4 keys of column i.
  const int i16 = lane & 15;
  const int v_frag_off = (4 * g + (i16 >> 2)) * LDV + 16 * ((lane >> 4) & 1) + 4 * (i16 & 3);
  // + (kb*32 + 16*t [+8]) * LDV + db*32

  if (n_kv_tiles > 0) load_tile(0, 0);
  if constexpr (CV) {
    if (tid < 2) v_top[tid] = 0;
    if (n_kv_tiles > 0) fetch_v(0);
    __syncthreads();
    if (n_kv_tiles > 0) {
      post_top(0);
      __syncthreads();
      rewrite_v(0);
      if (n_kv_tiles > 1) fetch_v(1);
    }
  }
  // (the second K buffer is not written before the loop's first barrier: room for the inv_freq table)
  if (a.q_rope) rotate_q_fragments<MT, D>(qreg, a, b, qi, g, reinterpret_cast<float *>(IN_TURN ? &Vs2[0][0] : &Ks2[1][0]));
  // The compiler does not model the asm loads or the asm wait below. Make it wait for Q here;
  // otherwise it puts its own vmcnt(0) in front of the first MFMA inside the loop, after the
  // prefetch of the next tile has been issued.
#pragma unroll
  for (int ks = 0; ks < KS; ks++) asm volatile("" :: "v"(qreg[ks]));

  // ---- One wave per SIMD (head dims above 128): no other wave fills the matrix pipe during the softmax, so the scores of tile
  // kt + 1 are computed beside the softmax of tile kt, in one stretch of code with that tile's second product. K is staged two
  // tiles ahead, V one. The order of the stretch is written out, an MFMA with its share of the other work at a time. What bounds
  // it is what the wave can issue: of 3130 cycles a tile (bf16, D = 256, 64 rows) the MFMAs take 1536. B=1 H=16/8 S=1500 D=256
  // causal bf16 51.1 -> 41.8 us, D=192 42 -> 34; B=1 H=8 S=2048 D=256 without a mask 65 -> 54. ----
  if constexpr (AHEAD) {
    static_assert(!CV && WPS == 1, "V tiles staged as they are, accumulation registers");
    auto k_frag = [&](int buf, int i) __attribute__((always_inline)) {  // the i-th MFMA of a tile's scores: key block i % NKB, k-step i / NKB
      return *reinterpret_cast<const vec8 *>(&Ks2[buf][kg * (BW * LDK) + k_frag_off + (i % NKB) * 32 * LDK + 16 * (i / NKB)]);
    };
    auto v_frag = [&](int buf, int i) __attribute__((always_inline)) {  // the i-th V fragment of a tile: 32 rows i % DB of O^T, keys 16 (i / DB)
      const uint16_t *vaddr = &Vs2[buf][kg * (BW * LDV) + v_frag_off + 16 * (i / DB) * LDV + (i % DB) * 32];
      const shortx4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_shortx4_t *)(vaddr));
      const shortx4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_shortx4_t *)(vaddr + 8 * LDV));
      return __builtin_bit_cast(vec8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    };
    constexpr int NQ = KS * NKB, NV = 2 * DB * NKB, NP = 8 * NKB;  // MFMAs of the scores, V fragments, pairs of weights, per tile
    constexpr int RING = 4;  // fragments in flight (eight: the same)
    constexpr int LOADS_FROM = 8;  // MFMA at which a tile's loads begin: the first ones have the exponentials beside them
    static_assert(LOADS_FROM + KI / NW + VI / NW <= NQ + NV, "a place for every load");
    float mx = 0.f;  // largest of a query's scores in s
    auto largest = [&](const floatx16_t (&s)[NKB]) __attribute__((always_inline)) {
      float mx = s[0][0];
#pragma unroll
      for (int kb = 0; kb < NKB; kb++)
#pragma unroll
        for (int i = 0; i < 16; i++) mx = fmaxf(mx, s[kb][i]);
      return max_over_wave_halves(mx);
    };
    // (With the lane's end taken once, as below, these forms are slower: bf16 S=1500 D=256 41.0 us instead of 40.0.)
    auto mask = [&](int k0, floatx16_t (&s)[NKB]) __attribute__((always_inline)) {
#pragma unroll
      for (int kb = 0; kb < NKB; kb++)
#pragma unroll
        for (int i = 0; i < 16; i++) {
          const int key = k0 + kb * 32 + 8 * (i >> 2) + 4 * g + (i & 3);
          if (key >= n_keys || (CAUSAL && key > qi)) s[kb][i] = -INFINITY;
        }
    };
    const int kg0 = wave_u / RG * BW, q_lo = q0 + wave_u % RH * 32, q_hi = q_lo + 31;  // (the branches below are the wave's)
    auto masked = [&](int k0) __attribute__((always_inline)) { return (k0 + BW > n_keys) || (CAUSAL && k0 + BW - 1 > q_lo); };
    // tiles in which a key of this wave's share is before its diagonal and the last key
    const int n_live = ((CAUSAL ? min(k_end, q_hi + 1) : k_end) - kg0 + BT - 1) / BT;
    // Scores of tile kt + 1 and, with_tile, softmax and second product of tile kt, whose masked scores are in s. Beside the MFMAs
    // of the first product this wave's loads of K of tile k_tile and V of tile v_tile.
    floatx16_t s[NKB], next[NKB];
    floatx16_t zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    asm volatile("" : "+a"(zero));
    auto compute = [&](auto with_tile, int kt, int k_tile, int v_tile) __attribute__((always_inline)) {
      constexpr bool TILE = decltype(with_tile)::value;
      const int k_buf = (kt + 1) & 1, v_buf = kt & 1;
      const float mc = m_i * c;
      uint32_t w[NP], w_lo[NP];  // weights, packed in pairs
      vec8 ring[RING];
#pragma unroll
      for (int i = 0; i < RING; i++) ring[i] = k_frag(k_buf, i);
      __builtin_amdgcn_sched_barrier(0);
      auto pairs = [&](int from, int to) __attribute__((always_inline)) {
#pragma unroll
        for (int j = from; j < to; j++) {
          const float p0 = __builtin_amdgcn_exp2f(s[j / 8][2 * (j % 8)] * c - mc), p1 = __builtin_amdgcn_exp2f(s[j / 8][2 * (j % 8) + 1] * c - mc);
          w[j] = MT::cvt_pair(p0, p1);
          if (MT::kSplitP) w_lo[j] = MT::cvt_pair(p0 - MT::low(w[j]), p1 - MT::high(w[j]));
          if (j % 4 == 3) {
            l_i = MT::sum8(__builtin_bit_cast(pvec8, make_uint4(w[j - 3], w[j - 2], w[j - 1], w[j])), l_i);
            if (MT::kSplitP) l_i = MT::sum8(__builtin_bit_cast(pvec8, make_uint4(w_lo[j - 3], w_lo[j - 2], w_lo[j - 1], w_lo[j])), l_i);
          }
        }
      };
      auto stage = [&](int i) __attribute__((always_inline)) {
        if (i < 0) return;
        if (i < KI / NW) load_k_block(k_tile, v_buf, i);
        else if (i < KI / NW + VI / NW) load_v_block(v_tile, k_buf, i - KI / NW);
      };
#pragma unroll
      for (int i = 0; i < NQ; i++) {
        next[i % NKB] = MT::mfma(ring[i % RING], qreg[i / NKB], i < NKB ? zero : next[i % NKB]);
        if (i + RING < NQ) ring[i % RING] = k_frag(k_buf, i + RING);
        else if (TILE) ring[i % RING] = v_frag(v_buf, i + RING - NQ);
        if constexpr (TILE) {
          stage(i - LOADS_FROM);
          pairs(i * NP / NQ, (i + 1) * NP / NQ);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (TILE) {
#pragma unroll
        for (int i = 0; i < NV; i++) {
          const int j = 4 * (i / DB), r = (i + NQ) % RING;
          oacc[i % DB] = MT::mfma_pv(ring[r], __builtin_bit_cast(pvec8, make_uint4(w[j], w[j + 1], w[j + 2], w[j + 3])), oacc[i % DB]);
          if (MT::kSplitP) oacc[i % DB] = MT::mfma_pv(ring[r], __builtin_bit_cast(pvec8, make_uint4(w_lo[j], w_lo[j + 1], w_lo[j + 2], w_lo[j + 3])), oacc[i % DB]);
          if (i + RING < NV) ring[r] = v_frag(v_buf, i + RING);
          stage(NQ + i - LOADS_FROM);
          if (i == NV / 2) {
#pragma unroll
            for (int kb = 0; kb < NKB; kb++) s[kb] = next[kb];
            mx = largest(s);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      } else {
#pragma unroll
        for (int kb = 0; kb < NKB; kb++) s[kb] = next[kb];
        mx = largest(s);
      }
      const int k0 = (kt + 1) * BT + kg0;
      if (__builtin_expect(masked(k0), 0)) {
        mask(k0, s);
        mx = largest(s);
      }
    };
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();  // (and the inv_freq table has been read)
    if (n_kv_tiles > 1) load_k(1, 1);
    if (n_live > 0) compute(std::false_type{}, -1, 0, 0);
    // The last tiles load the last one again instead of none: a branch between the MFMAs lets the compiler move the softmax behind
    // it. And the accumulators are named as accumulation registers wherever they enter or leave the loop or the rescale: left to
    // the compiler, which sees the rescale's vector instructions, they live in vector registers between the tiles, and two copies
    // of each, 256 instructions a tile, cost what working ahead gains.
    auto in_place = [&]() __attribute__((always_inline)) {
#pragma unroll
      for (int db = 0; db < DB; db++) asm volatile("" : "+a"(oacc[db]));
    };
    in_place();
    int kt = 0;
    for (; kt < n_live; kt++) {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();  // K of tile kt + 1 and V of tile kt are there, K of tile kt and V of tile kt - 1 done with
      const int k_tile = min(kt + 2, n_kv_tiles - 1), v_tile = min(kt + 1, n_kv_tiles - 1);
#pragma unroll
      for (int i = KI / NW; i < KJ; i++) load_k_block(k_tile, kt & 1, i);  // (that not every wave has to issue)
#pragma unroll
      for (int i = VI / NW; i < VJ; i++) load_v_block(v_tile, (kt + 1) & 1, i);
      if (__builtin_expect(__builtin_amdgcn_ballot_w64((mx - m_i) * c > kLazyRescale) != 0, 0)) {
        const float m_new = fmaxf(m_i, mx);
        const float alpha = __builtin_amdgcn_exp2f((m_i - m_new) * c);
        m_i = m_new;
        l_i *= alpha;
        in_place();
#pragma unroll
        for (int db = 0; db < DB; db++)
#pragma unroll
          for (int i = 0; i < 16; i++) oacc[db][i] *= alpha;
        in_place();
      }
      compute(std::true_type{}, kt, k_tile, v_tile);  // (after the last tile scores of whatever the buffer holds, for nobody)
      in_place();
    }
    for (; kt < n_kv_tiles; kt++) {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      load_k(min(kt + 2, n_kv_tiles - 1), kt & 1);
      load_v(min(kt + 1, n_kv_tiles - 1), (kt + 1) & 1);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (before the LDS is used for something else)
  } else {
  // IN_TURN: the tiles of which the wave has keys come first (with a branch around the others' products the accumulators are held twice)
  const int live_end = CAUSAL ? min(k_end, wave_q_hi + 1) : k_end;
  const int n_own = IN_TURN ? __builtin_amdgcn_readfirstlane(max(live_end - kg * BW + BT - 1, 0) / BT) : n_kv_tiles;
  for (int kt = 0; kt < n_own; kt++) {
    // One barrier per tile: tile kt (fetched during the previous iteration) becomes visible, and every
    // wave is done with tile kt-1, whose buffer the fetch of tile kt+1 now overwrites.
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's blocks of tile kt are in LDS
    if constexpr (CV)
      if (kt + 1 < n_kv_tiles) post_top((kt + 1) & 1);  // (its registers hold V of tile kt + 1)
    __syncthreads();  // ... and everyone's; tile kt-1 has been consumed, its buffer is free
    if constexpr (IN_TURN) load_v(kt, 0);  // (V of tile kt - 1 has been consumed)
    else if (kt + 1 < n_kv_tiles) load_tile(kt + 1, (kt + 1) & 1);  // in flight while tile kt is computed
    auto k_after_v = [&]() __attribute__((always_inline)) {  // IN_TURN: V of tile kt is there, K of it has been consumed
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      if (kt + 1 < n_kv_tiles) load_k(kt + 1, 0);
    };
    if constexpr (CV) thr_cur = thr_next;
    const uint16_t *Ks = Ks2[IN_TURN ? 0 : kt & 1] + kg * (BW * LDK);
    const uint16_t *Vs = Vs2[IN_TURN ? 0 : kt & 1] + kg * (BW * LDV);

    const int k0 = kt * BT + kg * BW;         // first key of this wave's share of the tile
    // all of it above this wave's diagonal, or past the last key (second half of the last tile)
    if (!IN_TURN && ((CAUSAL && k0 > wave_q_hi) || (KSPLIT > 1 && k0 >= k_end))) {
      if constexpr (CV) {
        rewrite_v((kt + 1) & 1);
        if (kt + 2 < n_kv_tiles) fetch_v(kt + 2);
      }
      continue;
    }

    // ---- S^T = K Q^T for the wave's 32-key blocks, two at a time: their fragments are fetched first, then
    // the two accumulator chains alternate so that neither waits on LDS or on its own previous MFMA ----
    floatx16_t sacc[NKB];
#pragma unroll
    for (int kb = 0; kb < NKB; kb++)
#pragma unroll
      for (int i = 0; i < 16; i++) sacc[kb][i] = 0.f;
    constexpr int KBG = NKB < 2 ? NKB : 2;  // key blocks whose fragments are fetched together
#pragma unroll
    for (int kb0 = 0; kb0 < NKB; kb0 += KBG) {
      if constexpr (D <= 128) {
        // (as one turn of the loop below the same instructions come in another order: B=1 H=32 S=512 D=64 causal fp16 7.9
        // -> 8.2 us, B=2 H=16 S=256 D=128 8.0 -> 8.2, B=8 H=32/8 S=512 D=128 causal bf16 40.3 -> 42.4)
        vec8 kf[KBG][KS];
#pragma unroll
        for (int ks = 0; ks < KS; ks++)
#pragma unroll
          for (int kb = 0; kb < KBG; kb++)
            kf[kb][ks] = *reinterpret_cast<const vec8 *>(&Ks[k_frag_off + (kb0 + kb) * 32 * LDK + 16 * ks]);
#pragma unroll
        for (int ks = 0; ks < KS; ks++)
#pragma unroll
          for (int kb = 0; kb < KBG; kb++) {
#ifdef LMH_FOLD_SCALE
            sacc[kb0 + kb] = MT::mfma(kf[kb][ks], qreg[ks], ks == 0 ? neg_mc16 : sacc[kb0 + kb]);
#else
            sacc[kb0 + kb] = MT::mfma(kf[kb][ks], qreg[ks], sacc[kb0 + kb]);
#endif
          }
      } else if constexpr (IN_TURN) {
        vec8 kf[KS];
        auto read_k = [&](int ks) __attribute__((always_inline)) { kf[ks] = *reinterpret_cast<const vec8 *>(&Ks[k_frag_off + 16 * ks]); };
#pragma unroll
        for (int ks = 0; ks < RING; ks++) read_k(ks);
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
          __builtin_amdgcn_sched_barrier(0);
          sacc[0] = MT::mfma(kf[ks], qreg[ks], sacc[0]);
          if (ks + RING < KS) read_k(ks + RING);
        }
        __builtin_amdgcn_sched_barrier(0);
      } else {
        constexpr int KSG = WPS == 2 ? 4 : KS / 2;  // long rows: as many k-steps at a time as the registers hold
#pragma unroll
        for (int ks0 = 0; ks0 < KS; ks0 += KSG) {
          vec8 kf[KBG][KS];
#pragma unroll
          for (int ks = ks0; ks < ks0 + KSG; ks++)
#pragma unroll
            for (int kb = 0; kb < KBG; kb++)
              kf[kb][ks] = *reinterpret_cast<const vec8 *>(&Ks[k_frag_off + (kb0 + kb) * 32 * LDK + 16 * ks]);
          // (with one wave per SIMD the compiler sinks every read to its MFMA and waits for it there: B=1 H=16/8 S=1500
          // D=256 causal bf16 54.2 -> 52.8 us; all sixteen reads at once spill and measure the same)
          if constexpr (WPS == 1) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int ks = ks0; ks < ks0 + KSG; ks++)
#pragma unroll
            for (int kb = 0; kb < KBG; kb++) {
#ifdef LMH_FOLD_SCALE
              sacc[kb0 + kb] = MT::mfma(kf[kb][ks], qreg[ks], ks == 0 ? neg_mc16 : sacc[kb0 + kb]);
#else
              sacc[kb0 + kb] = MT::mfma(kf[kb][ks], qreg[ks], sacc[kb0 + kb]);
#endif
            }
        }
      }
    }

    // The next V tile is rewritten here, in the shadow of the MFMAs just issued. (After the last tile this rewrites
    // stale registers into the buffer of tile kt - 1, which nobody reads any more.)
    if constexpr (CV) {
      rewrite_v((kt + 1) & 1);
      if (kt + 2 < n_kv_tiles) fetch_v(kt + 2);
    }

    // ---- masking (diagonal tiles and the ragged last tile only) ----
    // One compare a score, against the lane's own end: with the key's index built and compared with both limits, four instructions a
    // score, causal fp16 B=4 S=1024 D=128 took 46.9 us instead of 45.9, bf16 S=1100 D=64 42.1 instead of 41.3.
    const bool need_mask = (k0 + BW > n_keys) || (CAUSAL && k0 + BW - 1 > wave_q_lo);
    if (need_mask) {
      const int end = (CAUSAL ? min(n_keys, qi + 1) : n_keys) - k0 - 4 * g;  // of the keys that the lane's query sees
      constexpr bool kTwoCompares = TIGHT && (MT::kSplitP || !CAUSAL);  // (`end` is a register over the loop)
#pragma unroll
      for (int kb = 0; kb < NKB; kb++)
#pragma unroll
        for (int i = 0; i < 16; i++) {
          const int at = kb * 32 + 8 * (i >> 2) + (i & 3), key = k0 + at + 4 * g;
          if (kTwoCompares ? key >= n_keys || (CAUSAL && key > qi) : at >= end) sacc[kb][i] = -INFINITY;
        }
    }

    // ---- online softmax; all statistics are per lane (one query column) ----
    float mx = sacc[0][0];
#pragma unroll
    for (int kb = 0; kb < NKB; kb++)
#pragma unroll
      for (int i = 0; i < 16; i++) mx = fmaxf(mx, sacc[kb][i]);
    mx = max_over_wave_halves(mx);
#ifdef LMH_FOLD_SCALE
    // the scores are c s - c m already: raise m (and re-base this tile) where a row exceeds it by 2^8, and on the first tile
    if (!have_m || __builtin_amdgcn_ballot_w64(mx > kLazyRescale) != 0) {
      const float d = have_m ? fmaxf(mx, 0.f) : mx;
      const float alpha = have_m ? __builtin_amdgcn_exp2f(-d) : 1.f;
      have_m = true;
      neg_mc -= d;
#pragma unroll
      for (int i = 0; i < 16; i++) neg_mc16[i] = neg_mc;
      l_i *= alpha;
#pragma unroll
      for (int db = 0; db < DB; db++)
#pragma unroll
        for (int i = 0; i < 16; i++) oacc[db][i] *= alpha;
#pragma unroll
      for (int kb = 0; kb < NKB; kb++)
#pragma unroll
        for (int i = 0; i < 16; i++) sacc[kb][i] -= d;
    }
#else
    // m_i is finite after the first tile (key 0 is visible to every query); -inf before it.
    if (__builtin_amdgcn_ballot_w64((mx - m_i) * c > kLazyRescale) != 0) {  // wave-uniform
      const float m_new = fmaxf(m_i, mx);
      const float alpha = __builtin_amdgcn_exp2f((m_i - m_new) * c);
      m_i = m_new;
      l_i *= alpha;
#pragma unroll
      for (int db = 0; db < DB; db++)
#pragma unroll
        for (int i = 0; i < 16; i++) oacc[db][i] *= alpha;
    }
#endif
    const float mc = m_i * c;
    pvec8 pf[NKB][2], pf_lo[NKB][2];
#pragma unroll
    for (int kb = 0; kb < NKB; kb++)
#pragma unroll
      for (int t = 0; t < 2; t++) {
#pragma unroll
        for (int e = 0; e < 8; e++) {
#ifdef LMH_FOLD_SCALE
          const float p = __builtin_amdgcn_exp2f(sacc[kb][8 * t + e]);
#else
          const float p = __builtin_amdgcn_exp2f(sacc[kb][8 * t + e] * c - mc);
#endif
          pf[kb][t][e] = MT::cvt_p(p);
          if (MT::kSplitP) pf_lo[kb][t][e] = MT::cvt_p(p - (float)pf[kb][t][e]);
        }
        l_i = MT::sum8(pf[kb][t], l_i);
        if (MT::kSplitP) l_i = MT::sum8(pf_lo[kb][t], l_i);
      }

    // ---- O^T += V^T P^T ----
    if constexpr (IN_TURN) k_after_v();
    if constexpr (CV) {
      if (thr_cur != thr_acc) {  // this tile's V is stored against a larger value than the accumulated ones
        const int d = thr_cur - thr_acc;
        const float f = d < 127 ? __uint_as_float((uint32_t)(127 - d) << 23) : 0.f;
        thr_acc = thr_cur;
#pragma unroll
        for (int db = 0; db < DB; db++)
#pragma unroll
          for (int i = 0; i < 16; i++) oacc[db][i] *= f;
      }
    }
    if constexpr (IN_TURN) {
      shortx8_t vf[2 * DB];
      auto read_v = [&](int i) __attribute__((always_inline)) {
        const uint16_t *vaddr = &Vs[v_frag_off + 16 * (i / DB) * LDV + i % DB * 32];
        const shortx4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_shortx4_t *)(vaddr));
        const shortx4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_shortx4_t *)(vaddr + 8 * LDV));
        vf[i] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
      };
#pragma unroll
      for (int i = 0; i < RING; i++) read_v(i);
#pragma unroll
      for (int i = 0; i < 2 * DB; i++) {
        __builtin_amdgcn_sched_barrier(0);
        oacc[i % DB] = MT::mfma_pv(__builtin_bit_cast(vec8, vf[i]), pf[0][i / DB], oacc[i % DB]);
        if (MT::kSplitP) oacc[i % DB] = MT::mfma_pv(__builtin_bit_cast(vec8, vf[i]), pf_lo[0][i / DB], oacc[i % DB]);
        if (i + RING < 2 * DB) read_v(i + RING);
      }
    } else
#pragma unroll
    for (int kb = 0; kb < NKB; kb++) {
#pragma unroll
      for (int t = 0; t < 2; t++) {
#pragma unroll
        for (int db = 0; db < DB; db++) {
          const uint16_t *vaddr = &Vs[v_frag_off + (kb * 32 + 16 * t) * LDV + db * 32];
          const shortx4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_shortx4_t *)(vaddr));
          const shortx4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_shortx4_t *)(vaddr + 8 * LDV));
          const shortx8_t v8 = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
          oacc[db] = MT::mfma_pv(__builtin_bit_cast(vec8, v8), pf[kb][t], oacc[db]);
          if (MT::kSplitP) oacc[db] = MT::mfma_pv(__builtin_bit_cast(vec8, v8), pf_lo[kb][t], oacc[db]);
        }
      }
    }
  }
  if constexpr (IN_TURN) {
    for (int kt = n_own; kt < n_kv_tiles; kt++) {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      load_v(kt, 0);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      if (kt + 1 < n_kv_tiles) load_k(kt + 1, 0);
    }
  }
  }

#ifdef LMH_FOLD_SCALE
  m_i = have_m ? -neg_mc / c : -INFINITY;  // back to the units the merge below works in
#endif
  if constexpr (CV) {  // the accumulators hold O * 2^(112 - thr_acc)
    const float f = __uint_as_float((uint32_t)(thr_acc + 15) << 23);
#pragma unroll
    for (int db = 0; db < DB; db++)
#pragma unroll
      for (int i = 0; i < 16; i++) oacc[db][i] *= f;
  }
  // ---- the queries' copy, where the workgroups of a CU are at different places of their tiles: beside the loads of Q all
  // workgroups would store at once (B=4 H=32/8 T=777 D=128 fp16: 53.4 us, here 51.2, without a copy 46.0; a launch for the copy
  // 8). Workgroups of their own for it, between or behind the others, took 67 and 56 us. Not above head dim 128, where one
  // workgroup has the CU (D=256, 1500 rows: 1 % slower without a copy to make). ----
  auto store_queries = [&]() {
    const int first = max(q0, 0);
#pragma unroll
    for (int h = 0; h < HEADS; h++) {
      const int64_t at = ((int64_t)(b * a.Hq + hq + h * hq_step) * a.Sq + first) * a.D * 2;
      copy_span<64 * NW, (D / 16 + KSPLIT - 1) / KSPLIT>((char *)queries.dst + at, (const char *)queries.src + at, (min(q0 + BM, a.Sq) - first) * a.D * 2, wave_u);
    }
  };
  if (CAUSAL && KSPLIT > 1 && D <= 128 && queries.dst) store_queries();  // (before its second key group's waves end)

  // ---- key groups: fold group 1's (m, l, O) into group 0's; lane for lane the same layout ----
  if constexpr (IN_TURN) {
    // two by two and in two halves of the head dim, which fill the K tile
    constexpr int PARTS = 2, PB = DB / 2, NF = PB * 16 + 2;
    const int own_kg = wave_u / RG;  // (uniform: with branches by lane the accumulators are held twice)
    static_assert(DB % 2 == 0 && KSPLIT / 2 * RG * NF * 64 * 4 <= (int)sizeof(Ks2), "merge buffer must fit in the K tile");
#pragma unroll
    for (int half = KSPLIT / 2; half > 0; half /= 2) {
      float *xch = reinterpret_cast<float *>(&Ks2[0][0]) + (own_kg % half * RG + wave_u % RG) * (NF * 64) + lane;  // [half][RG][NF][64 lanes]
      float a0 = 0.f, a1 = 0.f;
#pragma unroll
      for (int part = 0; part < PARTS; part++) {
        __syncthreads();  // every wave has read its last tile, or what it folds
        if (own_kg >= half && own_kg < 2 * half) {
          xch[0] = m_i;
          xch[64] = l_i;
#pragma unroll
          for (int db = 0; db < PB; db++)
#pragma unroll
            for (int i = 0; i < 16; i++) xch[(2 + db * 16 + i) * 64] = oacc[part * PB + db][i];
        }
        __syncthreads();
        if (own_kg >= half) {
          if (half == 1 && part == PARTS - 1) return;
          continue;
        }
        if (part == 0) {
          const float m1 = xch[0], l1 = xch[64], m_new = fmaxf(m_i, m1);
          // a group that saw no key has m = -inf, l = 0, O = 0
          a0 = m_i == -INFINITY ? 0.f : __builtin_amdgcn_exp2f((m_i - m_new) * c);
          a1 = m1 == -INFINITY ? 0.f : __builtin_amdgcn_exp2f((m1 - m_new) * c);
          m_i = m_new;
          l_i = l_i * a0 + l1 * a1;
        }
#pragma unroll
        for (int db = 0; db < PB; db++)
#pragma unroll
          for (int i = 0; i < 16; i++) oacc[part * PB + db][i] = oacc[part * PB + db][i] * a0 + xch[(2 + db * 16 + i) * 64] * a1;
      }
    }
  } else if constexpr (KSPLIT > 1 && RG * (DB * 16 + 2) * 64 * 4 > (int)sizeof(Ks2)) {
    // in two halves of the head dim: the K tiles hold one at a time
    constexpr int PARTS = 2, PB = (DB + 1) / 2;
    constexpr int NF = PB * 16 + 2;  // floats per lane
    static_assert(RG * NF * 64 * 4 <= (int)sizeof(Ks2), "merge buffer must fit in the K tiles");
    float *xch = reinterpret_cast<float *>(&Ks2[0][0]) + (wave % RG) * (NF * 64) + lane;  // [NF][64 lanes]
    float a0 = 0.f, a1 = 0.f;
#pragma unroll
    for (int part = 0; part < PARTS; part++) {
      const int db0 = part * PB, db1 = db0 + PB < DB ? db0 + PB : DB;
      __syncthreads();  // every wave has read its last tile, or the part before
      if (kg == 1) {
        xch[0] = m_i;
        xch[64] = l_i;
#pragma unroll
        for (int db = db0; db < db1; db++)
#pragma unroll
          for (int i = 0; i < 16; i++) xch[(2 + (db - db0) * 16 + i) * 64] = oacc[db][i];
      }
      __syncthreads();
      if (kg == 1) {
        if (part == PARTS - 1) return;
        continue;
      }
      if (part == 0) {
        const float m1 = xch[0], l1 = xch[64];
        const float m_new = fmaxf(m_i, m1);
        // a group that saw no key has m = -inf, l = 0, O = 0
        a0 = m_i == -INFINITY ? 0.f : __builtin_amdgcn_exp2f((m_i - m_new) * c);
        a1 = m1 == -INFINITY ? 0.f : __builtin_amdgcn_exp2f((m1 - m_new) * c);
        l_i = l_i * a0 + l1 * a1;
      }
#pragma unroll
      for (int db = db0; db < db1; db++)
#pragma unroll
        for (int i = 0; i < 16; i++) oacc[db][i] = oacc[db][i] * a0 + xch[(2 + (db - db0) * 16 + i) * 64] * a1;
    }
  } else if (KSPLIT == 2) {
    constexpr int NF = DB * 16 + 2;  // floats per lane
    static_assert(KSPLIT != 2 || RG * NF * 64 * 4 <= (int)sizeof(Ks2), "merge buffer must fit in the K tiles");
    float *xch = reinterpret_cast<float *>(&Ks2[0][0]) + (wave % RG) * (NF * 64) + lane;  // [NF][64 lanes]
    __syncthreads();  // every wave has read its last tile
    if (kg == 1) {
      xch[0] = m_i;
      xch[64] = l_i;
#pragma unroll
      for (int db = 0; db < DB; db++)
#pragma unroll
        for (int i = 0; i < 16; i++) xch[(2 + db * 16 + i) * 64] = oacc[db][i];
    }
    __syncthreads();
    if (kg == 1) return;
    const float m1 = xch[0], l1 = xch[64];
    const float m_new = fmaxf(m_i, m1);
    // a group that saw no key has m = -inf, l = 0, O = 0
    const float a0 = m_i == -INFINITY ? 0.f : __builtin_amdgcn_exp2f((m_i - m_new) * c);
    const float a1 = m1 == -INFINITY ? 0.f : __builtin_amdgcn_exp2f((m1 - m_new) * c);
    l_i = l_i * a0 + l1 * a1;
#pragma unroll
    for (int db = 0; db < DB; db++)
#pragma unroll
      for (int i = 0; i < 16; i++) oacc[db][i] = oacc[db][i] * a0 + xch[(2 + db * 16 + i) * 64] * a1;
  } else if (KSPLIT > 2) {
    constexpr int NF = DB * 16 + 2;  // floats per lane
    static_assert(KSPLIT <= 2 || KSPLIT / 2 * RG * NF * 64 * 4 <= (int)sizeof(Ks2), "merge buffer must fit in the K tiles");
    // (the upper half into the lower one, until one is left. As the way of two groups too, this cost head dims above 128 5 to 9 %.)
#pragma unroll
    for (int half = KSPLIT / 2; half > 0; half /= 2) {
      float *xch = reinterpret_cast<float *>(&Ks2[0][0]) + (kg % half * RG + wave % RG) * (NF * 64) + lane;  // [half][RG][NF][64 lanes]
      __syncthreads();  // every wave has read its last tile, or what it folds
      if (kg >= half && kg < 2 * half) {
        xch[0] = m_i;
        xch[64] = l_i;
#pragma unroll
        for (int db = 0; db < DB; db++)
#pragma unroll
          for (int i = 0; i < 16; i++) xch[(2 + db * 16 + i) * 64] = oacc[db][i];
      }
      __syncthreads();
      if (kg >= half) {
        if (half == 1) return;
        continue;
      }
      const float m1 = xch[0], l1 = xch[64];
      const float m_new = fmaxf(m_i, m1);
      // a group that saw no key has m = -inf, l = 0, O = 0
      const float a0 = m_i == -INFINITY ? 0.f : __builtin_amdgcn_exp2f((m_i - m_new) * c);
      const float a1 = m1 == -INFINITY ? 0.f : __builtin_amdgcn_exp2f((m1 - m_new) * c);
      m_i = m_new;
      l_i = l_i * a0 + l1 * a1;
#pragma unroll
      for (int db = 0; db < DB; db++)
#pragma unroll
        for (int i = 0; i < 16; i++) oacc[db][i] = oacc[db][i] * a0 + xch[(2 + db * 16 + i) * 64] * a1;
    }
  }

  // ---- epilogue: out[qi][d] = O^T[d][qi] / l ----
  const float l_tot = sum_over_wave_halves(l_i);
  const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
  int row = qi, half = g;
  if (TIGHT && !CAUSAL) {  // (the row and its place from the lane's number, so that no register holds them until here)
    const int own_lane = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0));
    row = q0 + wave_u % RH * 32 + (own_lane & 31);
    half = own_lane >> 5;
  } else if (TIGHT) {
    asm volatile("" : "+v"(half));  // (or the offsets 16 j + 8 g of Q's loads are kept for the stores)
  }
  if ((uint32_t)row < (uint32_t)a.Sq) {
    const int64_t off = b * a.os[0] + own_hq * a.os[1] + (int64_t)row * a.os[2];
    store_out_rows<MT, DB>(oacc, inv, a.out, off, half, a.D, a.out_f32);
  }
  if (CAUSAL && KSPLIT == 1 && D <= 128 && queries.dst) store_queries();
}

// One workgroup per CU for non-causal launches with too few query rows to go round: the workgroup owns R
// consecutive 32-row blocks of one (b, hq) and runs R x KG waves — wave (r, kg) takes row block r against the kg-th
// 32 keys of every staged tile of 32 KG keys, with its own running max / sum / output; the KG partial results of a
// row block are folded through LDS at the end. With KG chosen so that R x KG is close to a multiple of four, every
// SIMD of the CU carries the same share of the workgroup's (rows x keys) area, which equal 64-row workgroups dealt
// two or three to a CU do not achieve, and every K/V tile is staged once for all R row blocks.
// Measured against those workgroups (B=4 H=20 Sq=448 D=64 fp16, five row blocks x three key groups): 1500 keys 28.7 ->
// 25.3 us, 3000 keys 51.4 -> 43.7, 750 keys 17.0 -> 16.4, 256 keys 9.2 -> 10.5 (one prologue per CU instead of three
// that overlap). Taller tiles (two blocks per wave and tile) and a third tile buffer were 1 % and 7 % slower.
// `mixed`: with five or seven row blocks no equal number of key groups fills four SIMDs evenly (5 x 3 = 15 waves: 4, 4, 4, 3).
// Then the workgroup runs 16 waves on tiles of 128 keys, some row blocks split between two waves (two 32-key blocks of a
// tile each) and the others between four, so that every SIMD walks R / 4 of a block's keys: 1.25 against 1.33 at R = 5
// (B=4 H=20 Sq=448 Sk=1500 D=64: 23.85 -> 23.55 us; D=96 with 3000 keys 54.9 -> 53.5), 1.75 against 2 at R = 7 (Sq=672:
// 37.4 us on the 64-row workgroups -> 32.7 us here).
constexpr int kWideMaxKeyGroups = 6;  // tiles of up to 192 keys: two buffers of them fit the LDS at D = 96
template <typename MT, int D>
__global__ __launch_bounds__(1024, 4) void prefill_mfma_wide_kernel(PrefillArgs a, int wgs_per_head, int n_whole, int mixed) {
  request_args(a);
  request_arg(wgs_per_head);
  request_arg(n_whole);
  request_arg(mixed);
  using vec8 = typename MT::vec8;
  constexpr int KS = D / 16, DB = D / 32;
  constexpr int LDK = D + kPadK, LDV = D + pad_v<D>();
  constexpr int KG_MAX = kWideMaxKeyGroups, BT_MAX = 32 * KG_MAX;  // keys per staged tile at most
  constexpr int NBUF = 2;  // tile kt + 1 is in flight while tile kt is computed
  constexpr int KC = LDK / 8, VC = LDV / 8;         // 16-byte chunks per LDS row
  constexpr int NW_MIN = 12;                        // the host launches 12 to 16 waves
  constexpr int KJ = (KC * BT_MAX / 64 + NW_MIN - 1) / NW_MIN, VJ = (VC * BT_MAX / 64 + NW_MIN - 1) / NW_MIN;
  constexpr int NF = DB * 16 + 2;                   // floats per lane of a partial result
  constexpr int K_BUF = BT_MAX * LDK, V_BUF = BT_MAX * LDV;  // elements per tile buffer
  constexpr int kWideMaxSlots = 12;  // (KG - 1) x R partial results at most; the host picks KG accordingly
  constexpr int kTileElems = NBUF * (K_BUF + V_BUF), kMergeElems = kWideMaxSlots * NF * 64 * 2;
  __shared__ __attribute__((aligned(16))) uint16_t lds[kTileElems > kMergeElems ? kTileElems : kMergeElems];  // tiles, then partials
  static_assert(sizeof(lds) <= 160 * 1024, "LDS of a CU");

  const int cpr = a.D / 8;
  int bh, j_wg;
  if (!deal_tile_by_head(a.B * a.Hq, wgs_per_head, n_whole, blockIdx.x & 7, blockIdx.x >> 3, &bh, &j_wg)) return;
  const int b = bh / a.Hq, hq = bh % a.Hq;
  const int kvh = kv_head_of(hq, a.Hq, a.Hkv, a.head_map);
  // row blocks of this workgroup: the head's ceil(Sq / 32) blocks dealt evenly to its workgroups
  const int n_blocks = (a.Sq + 31) / 32;
  const int base = n_blocks / wgs_per_head, extra = n_blocks % wgs_per_head;
  const int R = base + (j_wg < extra ? 1 : 0);
  if (R == 0) return;
  const int block0 = j_wg * base + min(j_wg, extra);
  const int NW = blockDim.x >> 6;
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int n = lane & 31, g = lane >> 5;
  // Which row block r of the workgroup the wave takes, as key group kg of that block's n_groups, and which 32-key blocks of
  // every staged tile: blocks kb0 .. kb0 + nkb - 1. The partial results of groups 1 .. n_groups - 1 go to LDS slots
  // slot0 + (kg - 1) * slot_step; group 0 folds them.
  int BT, r, kg, n_groups, kb0, nkb, slot0, slot_step;
  if (!mixed) {
    // the host launches R_max x KG waves; a workgroup with fewer row blocks may use more key groups or leave waves idle
    const int KG = min(min(NW / R, KG_MAX), kWideMaxSlots / R + 1);
    BT = 32 * KG;
    r = wave % R, kg = wave / R, n_groups = KG;
    kb0 = kg, nkb = 1, slot0 = r, slot_step = R;
  } else {
    // 16 waves on tiles of 128 keys: `heavy` row blocks are split between two waves (two 32-key blocks of a tile each), the
    // others between four (one block each). The heavy waves come first, so that dealt round-robin every SIMD gets the same
    // number of 32-key blocks per tile: R of them (R = 5: 2 + 1 + 1 + 1 against 4 x 1 per 96 keys with three key groups).
    BT = 128;
    const int heavy = max(2 * R - 8, 0), light = R - heavy;
    if (wave < 2 * heavy) {
      r = wave % heavy, kg = wave / heavy, n_groups = 2;
      kb0 = 2 * kg, nkb = 2, slot0 = r, slot_step = 0;
    } else {
      const int l = wave - 2 * heavy;
      r = heavy + l % light, kg = l / light, n_groups = 4;
      kb0 = kg, nkb = 1, slot0 = heavy + 3 * (l % light), slot_step = 1;
    }
  }
  const bool active = kg < n_groups;  // waves beyond the groups only help to stage
  const int qi = (block0 + r) * 32 + n;

  int n_keys = a.kv_len ? a.kv_len[b] : a.Sk;
  n_keys = min(max(n_keys, 0), a.Sk);
  const int n_kv_tiles = (n_keys + BT - 1) / BT;

  const uint16_t *qp = reinterpret_cast<const uint16_t *>(a.q) + b * a.qs[0] + hq * a.qs[1];
  const uint16_t *kp = reinterpret_cast<const uint16_t *>(a.k) + b * a.ks[0] + kvh * a.ks[1];
  const uint16_t *vp = reinterpret_cast<const uint16_t *>(a.v) + b * a.vs[0] + kvh * a.vs[1];

  vec8 qreg[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ks++) {
    uint4 raw = make_uint4(0, 0, 0, 0);
    if (active && qi < a.Sq && 16 * ks + 8 * g < a.D) raw = *reinterpret_cast<const uint4 *>(qp + (int64_t)qi * a.qs[2] + 16 * ks + 8 * g);
    qreg[ks] = __builtin_bit_cast(vec8, raw);
  }
  floatx16_t oacc[DB];
#pragma unroll
  for (int db = 0; db < DB; db++)
#pragma unroll
    for (int i = 0; i < 16; i++) oacc[db][i] = 0.f;
  float m_i = -INFINITY, l_i = 0.f;
  const float c = a.scale * kLog2e;

  // ---- staging, as in the kernel above: LDS-writing buffer loads, one tile ahead, wave w issues 1 KB blocks
  // w, w + NW, ...; the chunk -> (row, column) map does not depend on the tile height, rows past it are not fetched ----
  typedef int32_t i32x4_t __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) void lds_void_t;
  const int KI = (KC * BT + 63) / 64, VI = (VC * BT + 63) / 64;
  const int wave_u = __builtin_amdgcn_readfirstlane(wave);
  const int nw_u = __builtin_amdgcn_readfirstlane(NW);
  auto make_desc = [](const uint16_t *base_ptr, int bytes) {
    const uint64_t pp = (uint64_t)base_ptr;
    i32x4_t d;
    d[0] = __builtin_amdgcn_readfirstlane((int)(uint32_t)pp);
    d[1] = __builtin_amdgcn_readfirstlane((int)((pp >> 32) & 0xffff));
    d[2] = __builtin_amdgcn_readfirstlane(bytes);
    d[3] = 0x00020000;
    return d;
  };
  const i32x4_t k_desc = make_desc(kp, (int)((int64_t)n_keys * a.ks[2] * 2));
  const i32x4_t v_desc = make_desc(vp, (int)((int64_t)n_keys * a.vs[2] * 2));
  int k_voff[KJ], v_voff[VJ];
#pragma unroll
  for (int j = 0; j < KJ; j++) {
    const int ch = (wave + NW * j) * 64 + lane;
    const int row = ch / KC, col = ch % KC;
    k_voff[j] = (col < cpr && row < BT) ? (int)((row * a.ks[2] + col * 8) * 2) : kOutOfRange;
  }
#pragma unroll
  for (int j = 0; j < VJ; j++) {
    const int ch = (wave + NW * j) * 64 + lane;
    const int row = ch / VC, col = ch % VC;
    v_voff[j] = (col < cpr && row < BT) ? (int)((row * a.vs[2] + col * 8) * 2) : kOutOfRange;
  }
  const int k_tile_bytes = (int)(BT * a.ks[2] * 2), v_tile_bytes = (int)(BT * a.vs[2] * 2);
  const uint32_t k_lds0 = (uint32_t)(uintptr_t)(lds_void_t *)&lds[0] + wave_u * 1024;
  const uint32_t v_lds0 = (uint32_t)(uintptr_t)(lds_void_t *)&lds[NBUF * K_BUF] + wave_u * 1024;
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"  // m0 is a reserved register; it is only written here
  auto load_block = [](i32x4_t desc, uint32_t lds_addr, int voff, int soff) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 :: "s"(lds_addr), "v"(voff), "s"(desc), "s"(soff) : "memory", "m0");
  };
#pragma clang diagnostic pop
  auto load_tile = [&](int kt, int buf) {
#pragma unroll
    for (int j = 0; j < KJ; j++)
      if (wave_u + nw_u * j < KI)
        load_block(k_desc, k_lds0 + buf * (K_BUF * 2) + j * (nw_u * 1024), k_voff[j], kt * k_tile_bytes);
#pragma unroll
    for (int j = 0; j < VJ; j++)
      if (wave_u + nw_u * j < VI)
        load_block(v_desc, v_lds0 + buf * (V_BUF * 2) + j * (nw_u * 1024), v_voff[j], kt * v_tile_bytes);
  };

  const int k_frag_off = (kb0 * 32 + n) * LDK + 8 * g;  // + 32 LDK per further block
  const int i16 = lane & 15;
  const int v_frag_off = (kb0 * 32 + 4 * g + (i16 >> 2)) * LDV + 16 * ((lane >> 4) & 1) + 4 * (i16 & 3);

  if (n_kv_tiles > 0) load_tile(0, 0);
  if (a.q_rope) rotate_q_fragments<MT, D>(qreg, a, b, qi, g, reinterpret_cast<float *>(&lds[K_BUF]));
#pragma unroll
  for (int ks = 0; ks < KS; ks++) asm volatile("" :: "v"(qreg[ks]));

  for (int kt = 0; kt < n_kv_tiles; kt++) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's blocks of tile kt are in LDS
    __syncthreads();  // ... and everyone's; tile kt-1 has been consumed, its buffer is free
    if (kt + 1 < n_kv_tiles) load_tile(kt + 1, (kt + 1) & 1);
    for (int j = 0; j < nkb; j++) {
    const int k0 = kt * BT + (kb0 + j) * 32;  // this wave's 32 keys of the tile (nkb = 2: the second 32 follow)
    if (!active || k0 >= n_keys) break;
    const uint16_t *Ks = &lds[(kt & 1) * K_BUF + j * 32 * LDK];
    const uint16_t *Vs = &lds[NBUF * K_BUF + (kt & 1) * V_BUF + j * 32 * LDV];

    floatx16_t sacc;
#pragma unroll
    for (int i = 0; i < 16; i++) sacc[i] = 0.f;
    vec8 kf[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ks++) kf[ks] = *reinterpret_cast<const vec8 *>(&Ks[k_frag_off + 16 * ks]);
#pragma unroll
    for (int ks = 0; ks < KS; ks++) sacc = MT::mfma(kf[ks], qreg[ks], sacc);
    if (k0 + 32 > n_keys) {
#pragma unroll
      for (int i = 0; i < 16; i++)
        if (k0 + 8 * (i >> 2) + 4 * g + (i & 3) >= n_keys) sacc[i] = -INFINITY;
    }
    float mx = sacc[0];
#pragma unroll
    for (int i = 1; i < 16; i++) mx = fmaxf(mx, sacc[i]);
    mx = max_over_wave_halves(mx);
    if (__builtin_amdgcn_ballot_w64((mx - m_i) * c > kLazyRescale) != 0) {
      const float m_new = fmaxf(m_i, mx);
      const float alpha = __builtin_amdgcn_exp2f((m_i - m_new) * c);
      m_i = m_new;
      l_i *= alpha;
#pragma unroll
      for (int db = 0; db < DB; db++)
#pragma unroll
        for (int i = 0; i < 16; i++) oacc[db][i] *= alpha;
    }
    const float mc = m_i * c;
    vec8 pf[2], pf_lo[2];
#pragma unroll
    for (int t = 0; t < 2; t++) {
#pragma unroll
      for (int e = 0; e < 8; e++) {
        const float p = __builtin_amdgcn_exp2f(sacc[8 * t + e] * c - mc);
        pf[t][e] = MT::cvt(p);
        if (MT::kSplitP) pf_lo[t][e] = MT::cvt(p - (float)pf[t][e]);
      }
      l_i = MT::sum8(pf[t], l_i);
      if (MT::kSplitP) l_i = MT::sum8(pf_lo[t], l_i);
    }
#pragma unroll
    for (int t = 0; t < 2; t++) {
#pragma unroll
      for (int db = 0; db < DB; db++) {
        const uint16_t *vaddr = &Vs[v_frag_off + 16 * t * LDV + db * 32];
        const shortx4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_shortx4_t *)(vaddr));
        const shortx4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_shortx4_t *)(vaddr + 8 * LDV));
        const shortx8_t v8 = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
        oacc[db] = MT::mfma(__builtin_bit_cast(vec8, v8), pf[t], oacc[db]);
        if (MT::kSplitP) oacc[db] = MT::mfma(__builtin_bit_cast(vec8, v8), pf_lo[t], oacc[db]);
      }
    }
    }
  }

  // ---- fold the key groups of a row block: groups 1 .. KG-1 leave (m, l, O) in LDS, group 0 takes them in order ----
  float *xch = reinterpret_cast<float *>(&lds[0]) + lane;  // slot s at xch + s * NF * 64, [NF][64 lanes]
  __syncthreads();  // every wave has read its last tile
  if (active && kg > 0) {
    float *slot = xch + (slot0 + (kg - 1) * slot_step) * (NF * 64);
    slot[0] = m_i;
    slot[64] = l_i;
#pragma unroll
    for (int db = 0; db < DB; db++)
#pragma unroll
      for (int i = 0; i < 16; i++) slot[(2 + db * 16 + i) * 64] = oacc[db][i];
  }
  __syncthreads();
  if (!active || kg > 0) return;
  for (int k2 = 1; k2 < n_groups; k2++) {
    const float *slot = xch + (slot0 + (k2 - 1) * slot_step) * (NF * 64);
    const float m1 = slot[0], l1 = slot[64];
    const float m_new = fmaxf(m_i, m1);
    // a group that saw no key has m = -inf, l = 0, O = 0
    const float a0 = m_i == -INFINITY ? 0.f : __builtin_amdgcn_exp2f((m_i - m_new) * c);
    const float a1 = m1 == -INFINITY ? 0.f : __builtin_amdgcn_exp2f((m1 - m_new) * c);
    m_i = m_new;
    l_i = l_i * a0 + l1 * a1;
#pragma unroll
    for (int db = 0; db < DB; db++)
#pragma unroll
      for (int i = 0; i < 16; i++) oacc[db][i] = oacc[db][i] * a0 + slot[(2 + db * 16 + i) * 64] * a1;
  }

  const float l_tot = sum_over_wave_halves(l_i);
  const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
  if (qi < a.Sq) {
    const int64_t off = b * a.os[0] + hq * a.os[1] + (int64_t)qi * a.os[2];
    store_out_rows<MT, DB>(oacc, inv, a.out, off, g, a.D, a.out_f32);
  }
}

// ---------------------------------------------------------------------------------------------------------------
// Causal launches whose query tiles are few enough to matter one by one: a workgroup of 8 waves owns TWO 256-row query
// tiles of one (b, hq) — tile p and tile n - 1 - p — so that every workgroup of the launch walks the same number of keys
// (the short rows of the early tile plus the long rows of the late one), one workgroup per CU, no second round and no
// tail. Wave w carries rows 32 w .. of the early tile (row block 0) and rows 32 w .. of the late tile (row block 1).
// While the keys are visible to both tiles, every K and V^T fragment the wave reads from LDS feeds two MFMAs, one per
// row block (half the LDS reads per MFMA of the kernel above); past the early tile's diagonal the wave stores that
// tile's rows and goes on with the late tile alone. K/V tiles are staged once for both query tiles.
// Without a mask (CAUSAL = false) the two tiles are neighbours — a 512-row tile — and share every fragment to the end.
// ---------------------------------------------------------------------------------------------------------------
template <typename MT, int D, bool CAUSAL>
__global__ __launch_bounds__(512, 2) void prefill_mfma_pair_kernel(PrefillArgs a, Deal deal, int n_q_tiles, QueryCopy queries) {
  request_args(a);
  request_args(deal);
  request_arg(n_q_tiles);
  using vec8 = typename MT::vec8;
  static_assert(!MT::kSplitP && !MT::kConvertV, "one weight fragment per V fragment, V tiles staged as they are: fp16");
  constexpr int NW = 8, BM = 256;
  constexpr int BT = 2 * BN;        // 128 keys per staged tile
  constexpr int NKB = BT / 32;
  constexpr int KS = D / 16, DB = D / 32;
  const int cpr = a.D / 8;
  constexpr int LDK = D + kPadK, LDV = D + pad_v<D>();

  __shared__ __attribute__((aligned(16))) uint16_t Ks2[2][BT * LDK];
  __shared__ __attribute__((aligned(16))) uint16_t Vs2[2][BT * LDV];

  int bh, pair;
  if (!deal_tile(deal, blockIdx.x & 7, blockIdx.x >> 3, &bh, &pair)) return;
  const int b = (int)((uint32_t)bh / deal.hq), hq = bh - b * a.Hq;
  const int kvh = kv_head_of(hq, a.Hq, a.Hkv, a.head_map);
  // tile p with tile n - 1 - p; with an odd number of tiles the middle one is alone (its workgroup has no early tile)
  // (without a mask: two neighbouring tiles; the second one, row block 0 here, is missing at an odd end)
  const int t_late = CAUSAL ? n_q_tiles - 1 - pair : 2 * pair, t_early = CAUSAL ? pair : 2 * pair + 1;
  const bool has_early = CAUSAL ? t_early < t_late : t_early < n_q_tiles;

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int n = lane & 31, g = lane >> 5;
  // rows of this wave: qlo[rb] .. qlo[rb] + 31; without an early tile row block 0 lies past the last query
  const int shift = CAUSAL ? causal_shift(n_q_tiles, BM, a.Sq, BT) : 0;
  const int q0_early = t_early * BM - shift, q0_late = t_late * BM - shift;
  int qlo[2];
  qlo[0] = has_early ? q0_early + 32 * wave : a.Sq + 64;
  qlo[1] = q0_late + 32 * wave;

  int n_keys = a.kv_len ? a.kv_len[b] : a.Sk;
  n_keys = min(max(n_keys, 0), a.Sk);
  const int k_end_early = !has_early ? 0 : CAUSAL ? min(n_keys, q0_early + BM) : n_keys;   // keys the early tile can see
  const int k_end_late = CAUSAL ? min(n_keys, q0_late + BM) : n_keys;
  const int n_tiles_early = (k_end_early + BT - 1) / BT;
  const int n_tiles_late = (k_end_late + BT - 1) / BT;

  const uint16_t *qp = reinterpret_cast<const uint16_t *>(a.q) + b * a.qs[0] + hq * a.qs[1];
  const uint16_t *kp = reinterpret_cast<const uint16_t *>(a.k) + b * a.ks[0] + kvh * a.ks[1];
  const uint16_t *vp = reinterpret_cast<const uint16_t *>(a.v) + b * a.vs[0] + kvh * a.vs[1];

  vec8 qreg[2][KS];
#pragma unroll
  for (int rb = 0; rb < 2; rb++) {
    const int qi = qlo[rb] + n;
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
      uint4 raw = make_uint4(0, 0, 0, 0);
      if ((uint32_t)qi < (uint32_t)a.Sq && 16 * ks + 8 * g < a.D) raw = *reinterpret_cast<const uint4 *>(qp + (int64_t)qi * a.qs[2] + 16 * ks + 8 * g);
      qreg[rb][ks] = __builtin_bit_cast(vec8, raw);
    }
  }

  floatx16_t oacc[2][DB];
#pragma unroll
  for (int rb = 0; rb < 2; rb++)
#pragma unroll
    for (int db = 0; db < DB; db++)
#pragma unroll
      for (int i = 0; i < 16; i++) oacc[rb][db][i] = 0.f;
  float m_i[2] = {-INFINITY, -INFINITY}, l_i[2] = {0.f, 0.f};
  const float c = a.scale * kLog2e;

  // ---- tile staging, as in prefill_mfma_kernel ----
  typedef int32_t i32x4_t __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) void lds_void_t;
  constexpr int KC = LDK / 8, VC = LDV / 8;
  constexpr int KI = KC * BT / 64, VI = VC * BT / 64;
  constexpr int KJ = (KI + NW - 1) / NW, VJ = (VI + NW - 1) / NW;
  const int wave_u = __builtin_amdgcn_readfirstlane(wave);
  __builtin_assume(wave_u >= 0 && wave_u < NW);
  auto make_desc = [](const uint16_t *base, int bytes) {
    const uint64_t p = (uint64_t)base;
    i32x4_t d;
    d[0] = __builtin_amdgcn_readfirstlane((int)(uint32_t)p);
    d[1] = __builtin_amdgcn_readfirstlane((int)((p >> 32) & 0xffff));
    d[2] = __builtin_amdgcn_readfirstlane(bytes);
    d[3] = 0x00020000;
    return d;
  };
  const i32x4_t k_desc = make_desc(kp, (int)((int64_t)n_keys * a.ks[2] * 2));
  const i32x4_t v_desc = make_desc(vp, (int)((int64_t)n_keys * a.vs[2] * 2));
  int k_voff[KJ], v_voff[VJ];
#pragma unroll
  for (int j = 0; j < KJ; j++) {
    const int ch = (wave + NW * j) * 64 + lane;
    const int row = ch / KC, col = ch % KC;
    k_voff[j] = col < cpr ? (int)((row * a.ks[2] + col * 8) * 2) : kOutOfRange;
  }
#pragma unroll
  for (int j = 0; j < VJ; j++) {
    const int ch = (wave + NW * j) * 64 + lane;
    const int row = ch / VC, col = ch % VC;
    v_voff[j] = col < cpr ? (int)((row * a.vs[2] + col * 8) * 2) : kOutOfRange;
  }
  const int k_tile_bytes = (int)(BT * a.ks[2] * 2), v_tile_bytes = (int)(BT * a.vs[2] * 2);
  const uint32_t k_lds0 = (uint32_t)(uintptr_t)(lds_void_t *)&Ks2[0][0] + wave_u * 1024;
  const uint32_t v_lds0 = (uint32_t)(uintptr_t)(lds_void_t *)&Vs2[0][0] + wave_u * 1024;
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
  auto load_block = [](i32x4_t desc, uint32_t lds_addr, int voff, int soff) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 :: "s"(lds_addr), "v"(voff), "s"(desc), "s"(soff) : "memory", "m0");
  };
#pragma clang diagnostic pop
  auto load_tile = [&](int kt, int buf) {
#pragma unroll
    for (int j = 0; j < KJ; j++)
      if (wave_u + NW * j < KI)
        load_block(k_desc, k_lds0 + buf * (BT * LDK * 2) + j * (NW * 1024), k_voff[j], kt * k_tile_bytes);
#pragma unroll
    for (int j = 0; j < VJ; j++)
      if (wave_u + NW * j < VI)
        load_block(v_desc, v_lds0 + buf * (BT * LDV * 2) + j * (NW * 1024), v_voff[j], kt * v_tile_bytes);
  };

  const int k_frag_off = n * LDK + 8 * g;
  const int i16 = lane & 15;
  const int v_frag_off = (4 * g + (i16 >> 2)) * LDV + 16 * ((lane >> 4) & 1) + 4 * (i16 & 3);

  if (n_tiles_late > 0) load_tile(0, 0);
  if (a.q_rope) {
    float *table = reinterpret_cast<float *>(&Ks2[1][0]);
    if ((int)threadIdx.x < D / 2) table[threadIdx.x] = rope_inv_freq(threadIdx.x, D, a.q_log2_base);
    __syncthreads();
#pragma unroll
    for (int rb = 0; rb < 2; rb++) rotate_q_fragments_with_table<MT, D>(qreg[rb], a, b, qlo[rb] + n, g, table);
  }
#pragma unroll
  for (int rb = 0; rb < 2; rb++)
#pragma unroll
    for (int ks = 0; ks < KS; ks++) asm volatile("" :: "v"(qreg[rb][ks]));

  // One 32-key block at key k0 for row blocks RB0 .. 1 (RB0 = 0: both, every fragment read feeds two MFMAs; RB0 = 1: the
  // late tile alone). Online softmax per row block as in prefill_mfma_kernel.
  auto block = [&](auto rb0_c, auto nb_c, const uint16_t *Kb, const uint16_t *Vb, int k0) {
    constexpr int RB0 = decltype(rb0_c)::value;
    constexpr int NB = decltype(nb_c)::value;  // 32-key blocks taken together
    floatx16_t sacc[2][NB];
#pragma unroll
    for (int rb = RB0; rb < 2; rb++)
#pragma unroll
      for (int kb = 0; kb < NB; kb++)
#pragma unroll
        for (int i = 0; i < 16; i++) sacc[rb][kb][i] = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ks++)
#pragma unroll
      for (int kb = 0; kb < NB; kb++) {
        const vec8 kf = *reinterpret_cast<const vec8 *>(&Kb[k_frag_off + kb * 32 * LDK + 16 * ks]);
#pragma unroll
        for (int rb = RB0; rb < 2; rb++) sacc[rb][kb] = MT::mfma(kf, qreg[rb][ks], sacc[rb][kb]);
      }
    vec8 pf[2][NB][2];
#pragma unroll
    for (int rb = RB0; rb < 2; rb++) {
      if (k0 + 32 * NB > n_keys || (CAUSAL && k0 + 32 * NB - 1 > qlo[rb])) {  // the ragged last block, or a block on this row block's diagonal
        const int qi = qlo[rb] + n;
#pragma unroll
        for (int kb = 0; kb < NB; kb++)
#pragma unroll
          for (int i = 0; i < 16; i++) {
            const int key = k0 + 32 * kb + 8 * (i >> 2) + 4 * g + (i & 3);
            if (key >= n_keys || (CAUSAL && key > qi)) sacc[rb][kb][i] = -INFINITY;
          }
      }
      float mx = sacc[rb][0][0];
#pragma unroll
      for (int kb = 0; kb < NB; kb++)
#pragma unroll
        for (int i = 0; i < 16; i++) mx = fmaxf(mx, sacc[rb][kb][i]);
      mx = max_over_wave_halves(mx);
      // (key 0 is visible to every query, so m is finite after the first block)
      if (__builtin_amdgcn_ballot_w64((mx - m_i[rb]) * c > kLazyRescale) != 0) {
        const float m_new = fmaxf(m_i[rb], mx);
        const float alpha = __builtin_amdgcn_exp2f((m_i[rb] - m_new) * c);
        m_i[rb] = m_new;
        l_i[rb] *= alpha;
#pragma unroll
        for (int db = 0; db < DB; db++)
#pragma unroll
          for (int i = 0; i < 16; i++) oacc[rb][db][i] *= alpha;
      }
      const float mc = m_i[rb] * c;
#pragma unroll
      for (int kb = 0; kb < NB; kb++)
#pragma unroll
        for (int t = 0; t < 2; t++) {
#pragma unroll
          for (int e = 0; e < 8; e++) {
            const float p = __builtin_amdgcn_exp2f(sacc[rb][kb][8 * t + e] * c - mc);
            pf[rb][kb][t][e] = MT::cvt(p);
          }
          l_i[rb] = MT::sum8(pf[rb][kb][t], l_i[rb]);
        }
    }
#pragma unroll
    for (int kb = 0; kb < NB; kb++)
#pragma unroll
      for (int t = 0; t < 2; t++)
#pragma unroll
        for (int db = 0; db < DB; db++) {
          const uint16_t *vaddr = &Vb[v_frag_off + (32 * kb + 16 * t) * LDV + db * 32];
          const shortx4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_shortx4_t *)(vaddr));
          const shortx4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_shortx4_t *)(vaddr + 8 * LDV));
          const vec8 v8 = __builtin_bit_cast(vec8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
#pragma unroll
          for (int rb = RB0; rb < 2; rb++) {
            oacc[rb][db] = MT::mfma(v8, pf[rb][kb][t], oacc[rb][db]);
          }
        }
  };
  auto store_rows = [&](int rb) {
    const int qi = qlo[rb] + n;
    const float l_tot = sum_over_wave_halves(l_i[rb]);
    const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
    if ((uint32_t)qi < (uint32_t)a.Sq)
      store_out_rows<MT, DB>(oacc[rb], inv, a.out, b * a.os[0] + hq * a.os[1] + (int64_t)qi * a.os[2], g, a.D, a.out_f32);
  };
  // A whole 128-key tile for the late row block alone: the loop body of prefill_mfma_kernel (four 32-key blocks at a
  // time, their QK^T chains alternating two by two, one softmax pass over all 64 scores of a lane).
  auto tile_late = [&](const uint16_t *Ks, const uint16_t *Vs, int k0) {
    constexpr int rb = 1;
    if (CAUSAL && k0 > qlo[rb] + 31) return;  // the whole tile lies above this wave's rows
    floatx16_t sacc[NKB];
#pragma unroll
    for (int kb = 0; kb < NKB; kb++)
#pragma unroll
      for (int i = 0; i < 16; i++) sacc[kb][i] = 0.f;
#pragma unroll
    for (int kb0 = 0; kb0 < NKB; kb0 += 2) {
      vec8 kf[2][KS];
#pragma unroll
      for (int ks = 0; ks < KS; ks++)
#pragma unroll
        for (int kb = 0; kb < 2; kb++)
          kf[kb][ks] = *reinterpret_cast<const vec8 *>(&Ks[k_frag_off + (kb0 + kb) * 32 * LDK + 16 * ks]);
#pragma unroll
      for (int ks = 0; ks < KS; ks++)
#pragma unroll
        for (int kb = 0; kb < 2; kb++) sacc[kb0 + kb] = MT::mfma(kf[kb][ks], qreg[rb][ks], sacc[kb0 + kb]);
    }
    if (k0 + BT > n_keys || (CAUSAL && k0 + BT - 1 > qlo[rb])) {
      const int qi = qlo[rb] + n;
#pragma unroll
      for (int kb = 0; kb < NKB; kb++)
#pragma unroll
        for (int i = 0; i < 16; i++) {
          const int key = k0 + kb * 32 + 8 * (i >> 2) + 4 * g + (i & 3);
          if (key >= n_keys || (CAUSAL && key > qi)) sacc[kb][i] = -INFINITY;
        }
    }
    float mx = sacc[0][0];
#pragma unroll
    for (int kb = 0; kb < NKB; kb++)
#pragma unroll
      for (int i = 0; i < 16; i++) mx = fmaxf(mx, sacc[kb][i]);
    mx = max_over_wave_halves(mx);
    if (__builtin_amdgcn_ballot_w64((mx - m_i[rb]) * c > kLazyRescale) != 0) {
      const float m_new = fmaxf(m_i[rb], mx);
      const float alpha = __builtin_amdgcn_exp2f((m_i[rb] - m_new) * c);
      m_i[rb] = m_new;
      l_i[rb] *= alpha;
#pragma unroll
      for (int db = 0; db < DB; db++)
#pragma unroll
        for (int i = 0; i < 16; i++) oacc[rb][db][i] *= alpha;
    }
    const float mc = m_i[rb] * c;
    vec8 pf[NKB][2];
#pragma unroll
    for (int kb = 0; kb < NKB; kb++)
#pragma unroll
      for (int t = 0; t < 2; t++) {
#pragma unroll
        for (int e = 0; e < 8; e++) {
          const float p = __builtin_amdgcn_exp2f(sacc[kb][8 * t + e] * c - mc);
          pf[kb][t][e] = MT::cvt(p);
        }
        l_i[rb] = MT::sum8(pf[kb][t], l_i[rb]);
      }
#pragma unroll
    for (int kb = 0; kb < NKB; kb++)
#pragma unroll
      for (int t = 0; t < 2; t++)
#pragma unroll
        for (int db = 0; db < DB; db++) {
          const uint16_t *vaddr = &Vs[v_frag_off + (kb * 32 + 16 * t) * LDV + db * 32];
          const shortx4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_shortx4_t *)(vaddr));
          const shortx4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_shortx4_t *)(vaddr + 8 * LDV));
          const vec8 v8 = __builtin_bit_cast(vec8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
          oacc[rb][db] = MT::mfma(v8, pf[kb][t], oacc[rb][db]);
        }
  };
  const std::integral_constant<int, 0> kBoth{};
  const std::integral_constant<int, 1> kLate{};

  // ---- keys the early tile sees: both row blocks ----
  for (int kt = 0; kt < n_tiles_early; kt++) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (kt + 1 < n_tiles_late) load_tile(kt + 1, (kt + 1) & 1);
    const uint16_t *Ks = Ks2[kt & 1];
    const uint16_t *Vs = Vs2[kt & 1];
    constexpr int NB = 2;  // two 32-key blocks of both row blocks at a time: four score blocks in flight (fp16, D = 96: 244 registers)
    const std::integral_constant<int, NB> kNB{};
    const std::integral_constant<int, 1> kOne{};
#pragma unroll
    for (int kb = 0; kb < NKB; kb += NB) {
      const int k0 = kt * BT + kb * 32;
      if (k0 >= k_end_late) break;
      if (CAUSAL ? (k0 + 32 * NB - 1 <= qlo[0] && k0 + 32 * NB <= k_end_early) : true) {   // the whole group below the early rows' diagonal
        block(kBoth, kNB, Ks + kb * 32 * LDK, Vs + kb * 32 * LDV, k0);
      } else {
#pragma unroll
        for (int j = 0; j < NB; j++) {
          const int kj = k0 + 32 * j;
          if (kj >= k_end_late) break;
          if (kj <= qlo[0] + 31 && kj < k_end_early)
            block(kBoth, kOne, Ks + (kb + j) * 32 * LDK, Vs + (kb + j) * 32 * LDV, kj);
          else
            block(kLate, kOne, Ks + (kb + j) * 32 * LDK, Vs + (kb + j) * 32 * LDV, kj);
        }
      }
    }
  }
  if (has_early) store_rows(0);
  // ---- the rest: the late tile alone ----
  for (int kt = n_tiles_early; kt < n_tiles_late; kt++) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (kt + 1 < n_tiles_late) load_tile(kt + 1, (kt + 1) & 1);
    const uint16_t *Ks = Ks2[kt & 1];
    const uint16_t *Vs = Vs2[kt & 1];
    if (CAUSAL && kt * BT + BT - 1 > qlo[1]) {
      // a tile on the late rows' diagonal: block by block, so that blocks above the wave's rows are skipped (four at a
      // time they would be computed and masked: 109.9 -> 108.7 us on B=1 H=32 S=4096 D=96)
#pragma unroll
      for (int kb = 0; kb < NKB; kb++) {
        const int k0 = kt * BT + kb * 32;
        if (k0 > qlo[1] + 31 || k0 >= k_end_late) break;
        block(kLate, std::integral_constant<int, 1>{}, Ks + kb * 32 * LDK, Vs + kb * 32 * LDV, k0);
      }
    } else {
      tile_late(Ks, Vs, kt * BT);
    }
  }
  store_rows(1);
  if (CAUSAL && queries.dst) {
    for (int t = has_early ? 0 : 1; t < 2; t++) {
      const int q0 = t ? q0_late : q0_early, first = max(q0, 0);
      const int64_t at = ((int64_t)(b * a.Hq + hq) * a.Sq + first) * a.D * 2;
      copy_span<64 * NW, D / 16>((char *)queries.dst + at, (const char *)queries.src + at, (min(q0 + BM, a.Sq) - first) * a.D * 2, wave_u);
    }
  }
}

template <typename MT, int D>
int launch_pair(const PrefillArgs &a, const QueryCopy &queries, hipStream_t stream) {
  const int n_q_tiles = (a.Sq + 255) / 256;
  const int n_pairs = (n_q_tiles + 1) / 2;
  const int64_t wgs = deal_grid((int64_t)a.B * a.Hq, n_pairs);
  const int rc = check_grid(wgs, 512);
  if (rc != LMH_OK) return rc;
  dim3 grid((uint32_t)wgs), block(512);
  if (plan_only("prefill_mfma_pair_kernel<%s, D=%d, %s> query tiles=%d, workgroups=%u", MT::kName, D, a.causal ? "causal" : "full", n_q_tiles, grid.x)) return LMH_OK;
  const Deal deal = make_deal(a.B, a.Hq, n_pairs, 0, device_cu_count());
  if (a.causal)
    hipLaunchKernelGGL((prefill_mfma_pair_kernel<MT, D, true>), grid, block, 0, stream, a, deal, n_q_tiles, queries);
  else
    hipLaunchKernelGGL((prefill_mfma_pair_kernel<MT, D, false>), grid, block, 0, stream, a, deal, n_q_tiles, queries);
  LMH_HIP_TRY(hipGetLastError());
  return LMH_OK;
}

// The policy prefill_mfma_kernel runs a tensor type with. bf16 with V16: V rewritten as fp16 in the workgroups that own
// their query rows alone (B=1 H=32 S=4096 causal D=96 151 -> 122 us, D=128 202 -> 174, D=64 x 4 batches 443 -> 350; without
// a mask -15 ... -24 %); the small launches whose wave pairs split the keys keep head + remainder weights and LDS-direct V
// tiles (the rewrite sits on their critical path: 8 heads x 1024 rows 14.8 -> 20.6 us, 64 heads x 1024 rows 31.3 -> 35.6).
template <typename MT, bool V16, int KSPLIT> struct base_policy { using type = MT; };
template <> struct base_policy<MfmaBF16, true, 1> { using type = MfmaBF16V16; };

template <typename MT0, bool V16, int D, int KSPLIT, int NW, int WPS = default_wps<D, NW>(), bool AHEAD = false, int HEADS = 1>
int launch_split(const PrefillArgs &a, const QueryCopy &queries, hipStream_t stream) {
  using MT = typename base_policy<MT0, V16, KSPLIT>::type;
  constexpr int BM = 32 * NW / KSPLIT / HEADS;
  const int n_q_tiles = (a.Sq + BM - 1) / BM;
  const int64_t wgs = deal_grid((int64_t)a.B * a.Hq / HEADS, n_q_tiles);
  const int rc = check_grid(wgs, 64 * NW);
  if (rc != LMH_OK) return rc;
  dim3 grid((uint32_t)wgs), block(64 * NW);
  if (plan_only("prefill_mfma_kernel<%s, D=%d, %s, key groups=%d, waves=%d, waves per SIMD=%d> workgroups=%u%s%s%s", MT::kName, D,
                a.causal ? "causal" : "full", KSPLIT, NW, WPS, grid.x, HEADS == 2 ? ", two heads each" : "", MT::kConvertV ? ", V as fp16" : "", AHEAD ? ", a tile ahead" : ""))
    return LMH_OK;
  const Deal deal = make_deal(a.B, a.Hq / HEADS, n_q_tiles, a.causal ? 4 * WPS / NW : 0, device_cu_count());
  if (a.causal)
    hipLaunchKernelGGL((prefill_mfma_kernel<MT, D, true, KSPLIT, NW, WPS, AHEAD, HEADS>), grid, block, 0, stream, deal, a, queries);
  else if constexpr (HEADS == 1)
    hipLaunchKernelGGL((prefill_mfma_kernel<MT, D, false, KSPLIT, NW, WPS, AHEAD>), grid, block, 0, stream, deal, a, queries);
  LMH_HIP_TRY(hipGetLastError());
  return LMH_OK;
}

// Plan for the wide kernel: workgroups per head, waves per workgroup. Returns false where it does not apply or the
// equal 64-row workgroups are expected to do as well. `load` = the share of a 32-row block's keys that the busiest SIMD
// of the busiest CU walks, the quantity the launch time follows when the chip is not full. Measured (fp16, 1500 keys,
// wide against 64-row workgroups): load 1.33 vs 1.5 -12 % (D = 64), -14 % (D = 96); 0.75 vs 1.0 -7 ... -12 %; equal loads
// +-2 %, and +7 % at 1024 keys; under about 500 keys the single prologue per CU costs more than the balance wins.
inline bool wide_plan(const PrefillArgs &a, int n_cus, int *wgs_per_head, int *n_waves, int *mixed) {
  if ((int64_t)a.B * a.Hq > n_cus) return false;
  const int heads = a.B * a.Hq;
  const int n_blocks = (a.Sq + 31) / 32;
  if (a.causal || n_blocks < 2 || a.Sk < 640) return false;
  const int w = max(1, min(n_cus / heads, n_blocks / 2));
  const int r_max = (n_blocks + w - 1) / w;
  if (r_max > 8) return false;
  int best_kg = 0;
  double best = 1e30;
  for (int kg = 2; kg <= kWideMaxKeyGroups; kg++) {
    if (r_max * kg < 12 || r_max * kg > 16 || (kg - 1) * r_max > 12) continue;  // 12 to 16 waves, 12 partial results
    const double load = (double)((r_max * kg + 3) / 4) / kg;
    if (load <= best) best = load, best_kg = kg;  // on a tie, more waves
  }
  // two waves for some row blocks and four for the others (16 waves, tiles of 128 keys): every SIMD walks r_max / 4 of a
  // block's keys. Ahead of the equal key groups at five and seven row blocks (1.25 against 1.33, 1.75 against 2).
  *mixed = 0;
#ifndef LMH_NO_MIXED_KEY_GROUPS  // (a measurement build can keep equal key groups everywhere, for comparisons)
  if (r_max >= 5 && r_max <= 8 && r_max / 4.0 < best - 1e-9) best = r_max / 4.0, *mixed = 1;
#endif
  if (!best_kg && !*mixed) return false;
  // the equal 64-row workgroups, wave pairs splitting the keys: up to three resident on a CU, half a block's keys a wave
  const int64_t n64 = (int64_t)heads * ((a.Sq + 63) / 64);
  const double load_now = 0.5 * (double)((n64 + n_cus - 1) / n_cus);
  if (best > LMH_WIDE_MARGIN * load_now) return false;
  *wgs_per_head = w;
  *n_waves = *mixed ? 16 : r_max * best_kg;
  return true;
}

template <typename MT, int D>
int launch_wide(const PrefillArgs &a, int wgs_per_head, int n_waves, int mixed, hipStream_t stream) {
  dim3 grid((uint32_t)deal_grid(a.B * a.Hq, wgs_per_head)), block(64 * n_waves);
  if (plan_only("prefill_mfma_wide_kernel<%s, D=%d> workgroups per head=%d, waves=%d, workgroups=%u%s", MT::kName, D, wgs_per_head,
                n_waves, grid.x, mixed ? ", two and four key groups" : ""))
    return LMH_OK;
  hipLaunchKernelGGL((prefill_mfma_wide_kernel<MT, D>), grid, block, 0, stream, a, wgs_per_head, a.B * a.Hq / 8 * wgs_per_head, mixed);
  LMH_HIP_TRY(hipGetLastError());
  return LMH_OK;
}

// The forms of prefill_mfma_kernel and what a launch of each costs.
//
// A launch lasts as long as its busiest CU, and where the sizes leave a last row tile or a last round nearly empty the forms
// differ by up to 60 %: B=1 H=16 S=4501 D=96 causal bf16 is one and a half rounds of 128-row workgroups (173 us) or 1.1 rounds of
// 256-row ones (106). The thresholds of launch_for_d were measured at powers of two. Hence an estimate from the launch's tiles, in us:
//   fixed + longest row tile x alone       while every CU has at most one workgroup, or
//   the mean over the CUs x shared         when several share it (causal; the fourth powers blend the two), or
//   whole rounds of equal workgroups       (no mask), + per_wg for every workgroup that a CU starts.
// `alone` and `shared` are the times of a tile of 64 keys in a CU's only workgroup and in one of two or three (per tile, the
// others' tiles not counted). Fitted to 1916 launches, most of drawn sizes (16 to 8192 rows, 1 to 64 heads, batches to 16), some
// of powers of two, with every form timed on each: rms 5 to 13 %. The form of the rules by size is therefore left only for one
// that is estimated 8 % cheaper: 337 of those launches change their form, 296 of them gain more than 5 %, two lose more than 5 %
// (13 and 14 us), all 1916 together gain 2.5 % (with a margin of 4 % 2.9 %, and ten lose).
// The fit was made when causal tiles began at row 0, every workgroup took one head and 16-bit results were stored 8 bytes at a time, and the
// tiles are still counted so: the constants go with that count. Tiles counted as they are dealt now (causal_shift, two heads), with the
// constants as they are, change the form of 168 of 4000 drawn causal launches, to 0.75 to 1.44 of the time, 0.99 on average and half of them to more.
enum Form { kKeysSplit64, kRows128, kRows256, kRows256Pair };  // rows per workgroup; Pair: two 256-row workgroups on a CU
struct FormCost {
  float fixed, alone, per_wg, shared[2];  // shared by two and by three workgroups; with one per CU: in a later round
};
// [fp16, bf16 head + remainder, bf16 with V as fp16][head dims up to 64, 96, 128][form][causal]; fixed < 0: not built or never ahead
constexpr FormCost kFormCosts[3][3][4][2] = {
    {  // fp16
     {{{2.92f, 0.46f, 0.86f, 0.32f, 0.3f}, {2.75f, 0.49f, 0.91f, 0.31f, 0.31f}},
      {{2.6f, 0.75f, 1.2f, 0.55f, 0.54f}, {2.9f, 0.77f, 1.16f, 0.56f, 0.56f}},
      {{0.f, 1.01f, 4.8f, 1.01f, 1.01f}, {1.69f, 0.9f, 4.54f, 1.03f, 1.03f}},
      {{1.98f, 1.07f, 2.83f, 0.94f, 0.94f}, {3.44f, 1.02f, 2.09f, 1.05f, 1.05f}}},  // head dims up to 64
     {{{2.66f, 0.62f, 1.3f, 0.41f, 0.41f}, {2.55f, 0.61f, 1.47f, 0.43f, 0.43f}},
      {{2.18f, 0.9f, 2.07f, 0.7f, 0.7f}, {3.68f, 0.86f, 1.38f, 0.78f, 0.78f}},
      {{0.f, 1.29f, 5.74f, 1.29f, 1.29f}, {0.f, 1.11f, 6.8f, 1.36f, 1.36f}},
      {{1.12f, 1.34f, 4.16f, 1.23f, 1.23f}, {4.74f, 1.19f, 1.57f, 1.45f, 1.45f}}},  // head dims up to 96
     {{{1.97f, 0.79f, 2.58f, 0.53f, 0.53f}, {1.82f, 0.73f, 3.08f, 0.55f, 0.55f}},
      {{0.99f, 1.13f, 4.13f, 0.88f, 0.88f}, {2.55f, 1.06f, 3.23f, 0.99f, 0.99f}},
      {{0.f, 1.63f, 8.71f, 1.63f, 1.63f}, {0.19f, 1.41f, 8.29f, 1.77f, 1.77f}},
      {{-1.f}, {-1.f}}},  // head dims up to 128
    },
    {  // bf16, weights as head + remainder
     {{{3.3f, 0.59f, 0.74f, 0.46f, 0.42f}, {3.38f, 0.64f, 0.65f, 0.44f, 0.44f}},
      {{2.7f, 1.05f, 1.11f, 0.85f, 0.78f}, {4.61f, 1.01f, 0.24f, 0.86f, 0.86f}},
      {{1.28f, 1.55f, 3.98f, 1.55f, 1.55f}, {1.58f, 1.45f, 3.93f, 1.53f, 1.53f}},
      {{2.2f, 1.62f, 2.77f, 1.4f, 1.4f}, {4.8f, 1.55f, 0.22f, 1.58f, 1.58f}}},  // head dims up to 64
     {{{2.9f, 0.76f, 1.25f, 0.55f, 0.55f}, {3.1f, 0.75f, 1.17f, 0.58f, 0.58f}},
      {{2.65f, 1.21f, 1.79f, 1.f, 1.f}, {4.61f, 1.17f, 0.69f, 1.1f, 1.1f}},
      {{0.f, 1.8f, 6.79f, 1.8f, 1.8f}, {0.15f, 1.66f, 6.72f, 1.88f, 1.88f}},
      {{3.04f, 2.f, 4.23f, 1.81f, 1.81f}, {4.45f, 2.24f, 1.47f, 2.04f, 2.04f}}},  // head dims up to 96
     {{{2.96f, 0.92f, 2.21f, 0.71f, 0.71f}, {2.48f, 0.93f, 2.75f, 0.72f, 0.72f}},
      {{1.99f, 1.49f, 3.51f, 1.23f, 1.23f}, {3.23f, 1.43f, 2.58f, 1.34f, 1.34f}},
      {{-1.f}, {-1.f}},
      {{-1.f}, {-1.f}}},  // head dims up to 128
    },
    {  // bf16, V as fp16
     {{{-1.f}, {-1.f}},
      {{4.03f, 0.97f, 2.01f, 0.66f, 0.57f}, {4.68f, 0.98f, 1.59f, 0.64f, 0.64f}},
      {{0.98f, 1.11f, 6.96f, 1.11f, 1.11f}, {0.99f, 1.04f, 7.51f, 1.14f, 1.14f}},
      {{3.86f, 1.16f, 3.91f, 0.97f, 0.97f}, {6.18f, 1.17f, 1.98f, 1.13f, 1.13f}}},  // head dims up to 64
     {{{-1.f}, {-1.f}},
      {{4.55f, 1.5f, 3.45f, 0.88f, 0.84f}, {1.55f, 1.88f, 4.44f, 1.59f, 0.87f}},
      {{0.f, 1.33f, 9.72f, 1.33f, 1.33f}, {0.8f, 1.22f, 9.79f, 1.35f, 1.35f}},
      {{-1.f}, {-1.f}}},  // head dims up to 96
     {{{-1.f}, {-1.f}},
      {{3.81f, 1.36f, 4.9f, 0.97f, 0.97f}, {3.82f, 1.3f, 4.58f, 1.f, 1.f}},
      {{0.07f, 1.71f, 11.89f, 1.71f, 1.71f}, {0.f, 1.54f, 12.61f, 1.7f, 1.7f}},
      {{-1.f}, {-1.f}}},  // head dims up to 128
    },
};

inline double form_cost(const FormCost &f, const PrefillArgs &a, int form, int per_cu, int n_cus) {
  const int64_t heads = (int64_t)a.B * a.Hq, rows = form == kKeysSplit64 ? 64 : form == kRows128 ? 128 : 256;
  const int64_t n = (a.Sq + rows - 1) / rows, step = rows / BN, row_tiles = (a.Sk + BN - 1) / BN;
  const double wgs = (double)(heads * n) / n_cus;
  const int64_t rounds = (heads * n + n_cus - 1) / n_cus;
  const int on_cu = (int)std::min<int64_t>(rounds, per_cu);
  if (!a.causal) {
    auto batch = [&](int64_t k) -> double { return k < 1 ? 0. : k < 2 ? f.alone : std::max<double>(f.alone, k * f.shared[k - 2]); };
    return f.fixed + row_tiles * (rounds / per_cu * batch(per_cu) + batch(rounds % per_cu)) + f.per_wg * rounds;
  }
  const int64_t ramp = std::min(n, row_tiles / step);  // workgroups r < ramp walk (r + 1) step tiles, the others all of them
  const double longest = (double)std::min(row_tiles, n * step) * f.alone;
  if (wgs <= 1) return f.fixed + longest + f.per_wg;
  const double mean = (double)heads * (step * ramp * (ramp + 1) / 2 + (n - ramp) * row_tiles) / n_cus * f.shared[on_cu > 1 ? on_cu - 2 : 0];
  return f.fixed + sqrt(sqrt(longest * longest * longest * longest + mean * mean * mean * mean)) + f.per_wg * wgs;
}

// Whether a causal launch of 128-row workgroups at head dim 128 takes two query heads of one KV head in eight waves instead (HEADS = 2). By 230 launches of drawn sizes, both ways timed on each (104 to 128 elements, 1 to 64 heads, 200 to 4096 rows): from 1.5 to 2.1
// of the doubled workgroups per CU, of at least eight row tiles (bf16) or five (fp16), it takes 0.89 to 0.98 of the time, 0.93 on average,
// the worst 1.00. Up to 1.5 per CU 1.05 on average (0.92 to 1.12: the longest workgroup decides, and is longer), beyond 2.1 0.93 to 1.1, with
// fewer row tiles 0.94 to 1.1 (the two smaller workgroups of a CU are at different places of their tiles).
inline bool two_heads_ahead(const PrefillArgs &a, bool v16, int n_cus) {
  const int64_t tiles = (a.Sq + 127) / 128, wgs = (int64_t)a.B * a.Hq / 2 * tiles;
  return tiles >= (v16 ? 8 : 5) && 2 * wgs > 3 * n_cus && 10 * wgs <= 21 * n_cus;
}

// The forms of four and eight key groups (KSPLIT), by what they cost, in us, as above with their own tiles of 128 and 256 keys: a launch
// part, a tile of a CU's only workgroup, a part per workgroup on a CU, a tile of one of several. Without a mask with a CU for every
// workgroup only (two on a CU come out even). Fitted to 1260 launches of drawn sizes (1 to 128 heads, 16 to 8192 rows, 100 to
// 8192 keys, up to 2.5 workgroups per CU, fp16 and bf16, every form timed on each), rms 2 to 9 %. A launch goes over
// where the estimate is 5 % below that of the form it leaves: the 1260 gain 13 % together, half of what is over 12 us more than 15 %;
// 5 lose more than 4 %, the worst 8 % (bf16 60 heads 278 x 1233 D=64 20.1 and 21.7; the wide kernel is asked first). Below 256 keys they
// stay: 5.4 and 7.3 us (bf16 2 heads 258 x 164 D=64).
enum ManyGroups { k64RowsBy4, k32RowsBy4, k32RowsBy8 };
struct ManyGroupsCost {
  float fixed, alone, per_wg, shared;
};
// [fp16, bf16 head + remainder][head dims up to 64, 96, 128][form][causal]
constexpr ManyGroupsCost kManyGroupsCosts[2][3][3][2] = {
    {{{{3.31f, 0.675f, 1.10f, 0.f}, {3.01f, 0.685f, 1.63f, 0.450f}},
      {{2.46f, 0.585f, 1.58f, 0.f}, {2.77f, 0.556f, 1.48f, 0.298f}},
      {{2.94f, 0.832f, 1.99f, 0.f}, {0.f, 0.680f, 5.74f, 0.682f}}},
     {{{3.05f, 0.854f, 2.09f, 0.f}, {0.f, 0.840f, 5.29f, 0.867f}}, {}, {}},
     {{{3.32f, 1.091f, 2.66f, 0.f}, {0.f, 1.026f, 6.29f, 1.292f}}, {}, {}}},
    {{{{3.00f, 0.928f, 1.39f, 0.f}, {3.81f, 0.935f, 0.64f, 0.963f}},
      {{3.53f, 0.736f, 0.61f, 0.f}, {2.68f, 0.721f, 1.59f, 0.434f}},
      {{3.70f, 1.088f, 1.16f, 0.f}, {0.f, 1.010f, 5.22f, 0.866f}}},
     {{{3.89f, 1.113f, 1.13f, 0.f}, {0.f, 1.083f, 5.29f, 1.157f}}, {}, {}},
     {{{4.76f, 1.360f, 1.46f, 0.f}, {0.f, 1.325f, 6.33f, 1.548f}}, {}, {}}},
};

inline double many_groups_cost(const ManyGroupsCost &f, const PrefillArgs &a, int form, int n_cus) {
  const int64_t heads = (int64_t)a.B * a.Hq, rows = form == k64RowsBy4 ? 64 : 32, keys = form == k32RowsBy8 ? 256 : 128;
  const int64_t n = (a.Sq + rows - 1) / rows, row_tiles = (a.Sk + keys - 1) / keys;
  const double wgs = (double)(heads * n) / n_cus;
  // Beyond what the fit has seen: B=9 H=8 S=3885 D=32 143 -> 174 us. With lengths, of which only the largest possible one is known here, a walk is
  // shorter and the turning over of several workgroups on a CU weighs more (bf16 1 x 6 heads S=4527 D=96 causal at 0.6 of the length 39.8 -> 46.7).
  if (wgs > (a.kv_len ? 1. : 2.5)) return INFINITY;
  if (!a.causal) return wgs > 1 ? INFINITY : f.fixed + row_tiles * f.alone + f.per_wg;
  // step workgroups of a head end in the same key tile
  const int64_t step = keys / rows, whole = std::min(n / step, row_tiles), rest = n - whole * step;
  const double longest = (double)std::min(row_tiles, (n + step - 1) / step) * f.alone;
  if (wgs <= 1) return f.fixed + longest + f.per_wg;
  const double mean = (double)heads * (step * whole * (whole + 1) / 2 + rest * std::min(row_tiles, whole + 1)) / n_cus * f.shared;
  return f.fixed + sqrt(sqrt(longest * longest * longest * longest + mean * mean * mean * mean)) + f.per_wg * wgs;
}

// Launch the cheapest form, in favour of the one that the rules by size chose. bf16 launches whose weights are head + remainder
// by those rules stay so: V as fp16 goes with weights of 11 bits.
template <typename MT, int D, bool V16>
int launch_cheapest(const PrefillArgs &a, const QueryCopy &queries, int by_size, hipStream_t stream) {
  constexpr int tiling = D / 32 - 2;
  const int n_cus = device_cu_count();
  const bool v16 = V16 && by_size != kKeysSplit64;
  auto cost = [&](bool v, int form) {
    const FormCost &f = kFormCosts[!MT::kSplitP ? 0 : v ? 2 : 1][tiling][form][a.causal != 0];
    if (f.fixed < 0 || (form >= kRows256 && a.Sq <= 128)) return 1e30;
    // one row tile and one key tile in fp16 are as many workgroups either way, and no fold (recorded back to back, H=2 S=45 D=128
    // 5.15 against 5.34 us, D=64 3.68 and 3.72; on two key tiles 64 rows are ahead, 5.08 and 5.27)
    if (form == kKeysSplit64 && by_size != form && !MT::kSplitP && a.Sq <= 64 && a.Sk <= BN) return 1e30;
    return form_cost(f, a, form, form == kRows256 ? 1 : form == kRows256Pair || D > 96 ? 2 : 3, n_cus);
  };
  int best = by_size;
  bool best_v = v16;
  const double now = cost(v16, by_size);
  double least = now < 1e30 ? 0.92 * now : 0.;  // (a form without an estimate stays)
  for (int v = 0; v <= (int)v16; v++)
    for (int form = v ? (int)kRows128 : (int)kKeysSplit64; form <= kRows256Pair; form++) {
      const double t = cost(v, form);
      if (t < least) least = t, best = form, best_v = v;
    }
  int many = -1;  // of ManyGroups
  if (now < 1e30 && a.Sk >= 4 * BN) {
    least = best == by_size ? (a.kv_len ? 0.88 : 0.95) * now : least;  // (3 x 2 heads S=452 D=128 with lengths 11.0 -> 11.8 at 0.95)
    for (int form = k64RowsBy4; form <= (D == 64 ? k32RowsBy8 : k64RowsBy4); form++) {
      const double t = many_groups_cost(kManyGroupsCosts[MT::kSplitP][tiling][form][a.causal != 0], a, form, n_cus);
      if (t < least) least = t, many = form;
    }
  }
  if (many == k64RowsBy4) return launch_split<MT, false, D, 4, 8, D == 64 ? 4 : 2>(a, queries, stream);
  if constexpr (D == 64) {
    if (many == k32RowsBy4) return launch_split<MT, false, D, 4, 4, 2>(a, queries, stream);
    if (many == k32RowsBy8) return launch_split<MT, false, D, 8, 8, 2>(a, queries, stream);
  }
  auto launch = [&](auto with_v) {
    constexpr bool V = decltype(with_v)::value;
    if (best == kKeysSplit64) return launch_split<MT, V, D, 2, 4>(a, queries, stream);
    // Causal launches that eight waves of 256 rows would serve take two query heads of a KV head instead, 128 rows of each: as much shared,
    // and half a tile less on the diagonal and past the last row. 128 drawn launches of 256 to 8192 rows, time against 256 rows: head dim
    // 128 0.96 on average (0.88 to 1.01), up to 96 two workgroups on a CU 0.98 (0.90 to 1.01), one 0.98 in bf16 (0.94 to 1.01); one in fp16
    // 1.00 (to 1.02), which stays.
    const bool two = a.causal && a.Hq / a.Hkv % 2 == 0;
    if constexpr (D <= 96) {
      if constexpr (MT::kSplitP)
        if (best == kRows256 && two) return launch_split<MT, V, D, 1, 8, 2, false, 2>(a, queries, stream);
      if (best == kRows256) return launch_split<MT, V, D, 1, 8, 2>(a, queries, stream);
      if constexpr (!(D == 96 && V))  // (its registers spill at four waves per SIMD)
        if (best == kRows256Pair) return two ? launch_split<MT, V, D, 1, 8, 4, false, 2>(a, queries, stream) : launch_split<MT, V, D, 1, 8>(a, queries, stream);
    } else if constexpr (!MT::kSplitP || V) {
      if (best == kRows256 ? two : best == kRows128 && two && two_heads_ahead(a, V, n_cus))
        return launch_split<MT, V, D, 1, 8, 2, false, 2>(a, queries, stream);
      if (best == kRows256) return launch_split<MT, V, D, 1, 8>(a, queries, stream);
    }
    return launch_split<MT, V, D, 1, 4>(a, queries, stream);
  };
  if constexpr (V16)
    if (best_v) return launch(std::true_type{});
  return launch(std::false_type{});
}

// V16 (bf16 only): the launches of one key group hand V to the matrix cores as fp16 (base_policy above). The rules by size of
// this function hold where the sizes fill whole tiles and rounds; launch_cheapest looks at the others.
template <typename MT, int D, bool V16>
int launch_for_d(const PrefillArgs &a, const QueryCopy &queries, hipStream_t stream) {
  static_assert(!V16 || MT::kSplitP, "V16 is a form of the bf16 kernels");
  const auto launch = [&](int by_size) { return launch_cheapest<MT, D, V16>(a, queries, by_size, stream); };
  // With fewer than two 128-row workgroups per CU the launch is bound by how long one workgroup
  // takes to walk its keys, not by the matrix pipes: split the keys of a tile between wave pairs.
  // Measured on 256 CUs: at exactly two per CU the split still wins for causal launches (41.8 vs
  // 46.7 us at B=1 H=32 S=2048 D=96) and loses for non-causal ones (79.8 vs 66.6 us); at three per
  // CU it loses for both.
  const int n_cus = device_cu_count();
  // Causal launches that are exactly one round of paired 256-row tiles (tile p with tile n - 1 - p: equal work in every
  // workgroup, one per CU): the Phi-3 prompt, 32 heads x 16 tiles = 256 pairs. Measured against the kernels below on
  // 256 CUs, fp16: B=1 H=32 S=4096 D=96 -3.2 %, D=64 -6 %, D=80 -3 %; B=2 H=32 S=2048 -5 %; H=8 S=16384 -4.6 %;
  // S=3900 -2 %. With the chip not exactly full it loses (1.25 rounds +23 %, 1.5 rounds +10 %, half a round +30 %),
  // at exactly two rounds it ties (-1.4 ... +7 %).
  // bf16 stays on the kernels below: the fp16 rewrite of V that prefill_mfma_kernel does gains more than the pairing did
  // with bf16 weights as head + remainder (B=1 H=32 S=4096 D=64 causal: 117.7 us here, 99.8 us there), and two row blocks
  // plus the rewrite's registers do not fit; this kernel is built for fp16 only.
#ifndef LMH_NO_PAIR_KERNEL  // (measurement builds can keep these launches on the kernels below, for comparisons with them)
  if constexpr (D <= 96 && !MT::kSplitP) {
    const int64_t wgs_pair = (int64_t)a.B * a.Hq * (((a.Sq + 255) / 256 + 1) / 2);
    if (a.causal && a.Sq > 256 && wgs_pair <= n_cus && 16 * wgs_pair >= 15 * n_cus) return launch_pair<MT, D>(a, queries, stream);
    // Without a mask the same kernel takes two neighbouring tiles (512 rows, every fragment read shared all the way);
    // its workgroups are equal, so it wants whole rounds: B=1 H=32 S=4096 D=96 (one round) -5.9 %, S=8192 (two) -3.5 %,
    // B=4 (four) -1.1 %; D=64 one round -2.4 %, two rounds +2.5 %; 1.25 rounds +20 %.
    if (!a.causal && a.Sq > 256) {
      const int64_t rounds = (wgs_pair + n_cus - 1) / n_cus, last = wgs_pair - (rounds - 1) * n_cus;
      if (16 * last >= 15 * n_cus && (rounds == 1 || (D > 64 && rounds <= 2))) return launch_pair<MT, D>(a, queries, stream);
    }
  }
#endif
  const int64_t wgs = (int64_t)a.B * a.Hq * ((a.Sq + 127) / 128);
  const int64_t limit = a.causal ? 2 * n_cus : 2 * n_cus - 1;
  if (wgs <= limit && a.Sk >= 4 * BN) {
    if constexpr (D <= 96) {
      int wgs_per_head, n_waves, mixed;
      if (wide_plan(a, n_cus, &wgs_per_head, &n_waves, &mixed)) return launch_wide<MT, D>(a, wgs_per_head, n_waves, mixed, stream);
    }
    return launch(kKeysSplit64);
  }
  // Large launches: 256-row workgroups of eight waves. Measured against the 128-row ones at D = 96, fp16:
  // non-causal 512 / 768 / 1024 / 1536 / 2048 workgroups +3 / +2 / +2 / +6 / +5 %, causal 512 -7 %
  // (too few to balance their unequal lengths), 1024 +3 %, 1536 +4..7 %, 2048 +5 %.
  // D = 128 does not fit the 128 registers that four waves per SIMD leave: one 256-row workgroup per CU there,
  // which turns over in rounds and balances earlier. fp16: non-causal 256 / 512 / 2048 workgroups +5 / +3 / +6 %,
  // causal 256 / 384 -8 / -5 %, 512 / 1024 / 2048 +8 / +3 / +4 %; bf16 (V rewritten as fp16) 512 workgroups causal
  // +8 %, without a mask +5 %, 2048 causal +5 %.
  const int64_t wgs256 = (int64_t)a.B * a.Hq * ((a.Sq + 255) / 256);
  if (a.Sq <= 128) return launch(kRows128);  // nothing for waves 4-7 to own
  if constexpr (D <= 96) {
    // Causal launches of 1.5 to 3 rounds of one 256-row workgroup per CU (the Phi-3 prompt, 32 heads x 4096 rows,
    // is exactly two): the workgroups turn over heaviest first, so every CU ends up with about the same number
    // of key tiles; K/V tiles are staged once per 256 rows, and with the CU to itself the workgroup stages 128
    // keys at a time. Against the 128-row workgroups at D = 96: 1.5 rounds +2 %, 2 rounds +6 % (120.4 -> 112 us;
    // bf16 164 -> 153 us), 2.25 / 2.5 rounds +1 %, 3 and 3.5 rounds +-0; one round -20 %; D = 64 (2 rounds) -5 %.
    // Non-causal workgroups are all equally long and a part-filled round is lost time: from two rounds on only
    // (2 rounds +1 %, bf16 +4 %; 2.5 rounds +3 %; 1.5 rounds -11 %).
    // bf16 (V rewritten as fp16 through registers) spills at four waves per SIMD and stays on this form however many
    // rounds there are: B=4 H=32 S=4096 causal 583 -> 507 us, without a mask 946 -> 892 us. At D = 64 it takes this form for
    // causal launches of 1.5 to 3 rounds (the rewrite is shared by eight waves instead of four: B=1 H=32 S=4096 100.1 -> 96.5
    // us, H=64 S=2048 60.3 -> 58.6); from three rounds on and without a mask two workgroups per CU are 6-10 % ahead there.
    if constexpr (D == 96 || V16)
      if ((D == 96 || a.causal) && ((D == 96 && V16) || wgs256 < 3 * n_cus) &&
          (a.causal ? 2 * wgs256 >= 3 * n_cus : wgs256 >= 2 * n_cus))
        return launch(kRows256);
    if constexpr (!(D == 96 && V16))  // (with V16, D = 96 never gets here with that many workgroups)
      if (wgs256 >= (a.causal ? 4 * n_cus : 2 * n_cus)) return launch(kRows256Pair);
  } else if constexpr (!MT::kSplitP || V16) {  // (bf16 with head + remainder weights: 0 / -2 %, stays on 128 rows)
    if (wgs256 >= (a.causal ? 2 * n_cus : n_cus)) return launch(kRows256);
  }
  return launch(kRows128);
}

// Head dims above 128: Q and the accumulators of 32 rows take up to 192 registers and a tile buffer pair up to 141 KB, so a
// workgroup has the CU to itself. The vector-ALU kernel that took these launches reaches 8 TFLOP/s. Four forms:
//   64 rows, four waves in two key groups: one wave per SIMD, as many workgroups as there can be;
//   128 rows, four waves: no fold at the end, one wave per SIMD;
//   128 rows, eight waves in two key groups: two waves per SIMD, which fit with 256 registers each when K fragments are
//     fetched four k-steps at a time. The second wave computes while the first waits for LDS;
//   fp16: 64 rows, eight waves in four key groups, one tile of 128 keys (IN_TURN above).
// The first two work a tile ahead (AHEAD) from three key tiles a row on; on one or two the shorter loop is 3 to 9 % faster (B=1
// H=8 S=83 D=256 bf16 11.0 against 11.5 us, B=3 H=12 Sq=5675 Sk=43 D=192 fp16 65 against 72).
// A launch lasts as long as its busiest CU: the key tiles it walks (its longest workgroup or the mean over the CUs with a causal
// mask, whole rounds without one) and the workgroups it starts, each worth five tiles of the first form. A tile takes 1.4 and 1.2
// times as long in the other two, a start of the third six tiles. Fitted to 386 drawn launches (fp16 and bf16, head dims 160 to
// 256, 16 to 8192 rows, 1 to 64 heads, with every form timed on each): within 0.7 % of the best form on average, where the
// comparison of the tiles alone is 5 % behind it. (fp16 launches whose 64-row and 128-row workgroups walk the same 12 tiles or more are
// in it too: of 60 such the 46 with a mask, up to 50 workgroups, take 19 to 37 % less time in the 64-row form than on eight waves, H=2/1
// S=1537 D=208 44.4 and 31.2 us; the 14 without one from -5 to +11 %.) That comparison, in which 64 rows have to be 10 % cheaper to be
// left (fp16 from 12 tiles on takes 128), was measured with the shorter loop and still chooses for it.
// The fourth form walks a tile of 128 keys in 1.5 to 1.9 us, what the CU's fetch of it takes (65 to 70 bytes a ns), where the first takes two of
// 64 in 2.1 to 2.4; folding four groups costs it 3 to 5 us a workgroup. fp16, us in the form of before and in it: 16 heads 548 x 5273 D=160 88.1 and 64.7, H=6
// S=2255 causal 42.6 and 32.7, H=2 S=6502 D=192 causal 109.8 and 82.5, H=1 S=5850 D=256 causal 108.3 and 89.0, H=3 S=2389 51.0 and 45.1, H=6 110 x 2476
// 52.9 and 46.9. Fitted to 64 launches of 500 to 8192 keys that one or two of the others were best for: 29 go over, none loses more than 2.6 % (H=2 S=1739 D=256
// 22.4 and 24.1 stays). Launches of more workgroups than CUs, whose K and V the 64-row tiles read more often, go over from 15 % on (H=6 S=7218 D=256
// causal with lengths 144.5 and 168.5, B=5 H=4 S=961 D=192 causal 22.0 and 24.7, 160 heads 252 x 4832 D=176 242 and 354 stay): of 3000 drawn launches 527 go over,
// 1.17 times as fast in the geometric mean, none loses more than 5 %; from 0 % on 611 did, 13 of them lost that, up to 30 %. bf16, with twice the second products, comes out even (H=8 S=3130 D=256 causal 71.4 and 73.3, 16/8 heads S=1500 45.7 and 52.3). With the
// second half's waves a barrier behind, so that one half's softmax stands beside the other's second product, it took 2 to 10 % longer (H=3 3451 keys D=160
// 45.4 and 48.1): the phases are as long as the fetches then.
// B=1 H=32 S=4096 D=256 causal fp16 takes 292 us = 940 TFLOP/s (363 with 128 rows on four waves as the only form).
// bf16 keeps head + remainder weights at every length: the registers of the fp16 rewrite of V spill here (S=4096: 633 us).
// The head dims that are odd multiples of 8 stay on the vector-ALU kernel.
template <typename MT, int D>
int launch_wide_heads(const PrefillArgs &a, const QueryCopy &queries, hipStream_t stream) {
  const int64_t heads = (int64_t)a.B * a.Hq, cus = device_cu_count();
  const int64_t row_tiles = (a.Sk + BN - 1) / BN;  // key tiles of a whole row
  auto cost = [&](int rows, double tile, double start, int64_t step = 1) -> double {  // workgroups of `rows` query rows that take `step` key tiles at a time
    const int64_t n = (a.Sq + rows - 1) / rows, s = rows / BN, row = (row_tiles + step - 1) / step * step;
    if (!a.causal) return (double)((heads * n + cus - 1) / cus) * (row * tile + start);
    const int64_t ramp = std::min(n, row / s);  // workgroups r < ramp walk (r + 1) s tiles, the others all of them
    const double longest = (double)((std::min(row, n * s) + step - 1) / step * step);
    const double mean = heads * (s * ramp * (ramp + 1) / 2 + (n - ramp) * row + ramp * (step - 1) / 2.) / cus;
    return std::max(longest, mean) * tile + std::max(1., (double)(heads * n) / cus) * start;
  };
  if (row_tiles <= 2) {
    const double s64 = cost(64, 1., 0.), s128 = cost(128, 1., 0.);
    if (s128 > 0.9 * s64 && (MT::kSplitP || s128 < 12)) return launch_split<MT, false, D, 2, 4>(a, queries, stream);
    return launch_split<MT, false, D, 1, 4>(a, queries, stream);
  }
  const double rows64 = cost(64, 1., 5.), rows128 = cost(128, 1.4, 5.), eight = cost(128, 1.2, 6.);
  if constexpr (!MT::kSplitP)
    if (cost(64, 0.68, D <= 192 ? 9. : 15., 2) < (heads * ((a.Sq + 63) / 64) > cus ? 0.85 : 1.) * std::min(rows64, std::min(rows128, eight))) return launch_split<MT, false, D, 4, 8, 2>(a, queries, stream);
  if (rows64 <= std::min(rows128, eight)) return launch_split<MT, false, D, 2, 4, 1, true>(a, queries, stream);
  if (rows128 < 0.98 * eight) return launch_split<MT, false, D, 1, 4, 1, true>(a, queries, stream);
  return launch_split<MT, false, D, 2, 8, 2>(a, queries, stream);
}

template <typename MT>
int launch_for_type(const PrefillArgs &a, const QueryCopy &queries, hipStream_t stream) {
  if (a.D > 256) return fail(LMH_E_UNSUPPORTED, "MFMA flash attention: head dim %d not tiled", a.D);
#ifndef LMH_BF16_SPLIT_P
  if constexpr (MT::kSplitP) {
    // bf16: V as fp16 pays from about 512 keys per query row on. Its prologue (the first V tile through registers before
    // the first barrier) and one workgroup per CU cost short rows more than the second MFMA per fragment does: 512 heads,
    // fp16 rewrite against head + remainder, causal S=128 +15 ... +35 %, S=256 +7 ... +44 %, S=512 -3 ... +18 %, S=1024
    // -13 ... 0 %; without a mask S=128 0 ... +30 %, S=256 -7 ... -1 %, S=512 -13 ... +5 %, S=1024 -5 ... -19 %. (The
    // D = 96 tiling, one workgroup per CU in this form, is the one that ties or loses at 512 keys per row: 1024 there.)
    const int64_t keys_per_row = a.causal ? (a.Sq < a.Sk ? a.Sq : a.Sk) / 2 : a.Sk;
    if (a.D <= 128 && keys_per_row >= (a.D > 64 && a.D <= 96 ? 1024 : 512)) {
      if (a.D <= 64) return launch_for_d<MT, 64, true>(a, queries, stream);
      if (a.D <= 96) return launch_for_d<MT, 96, true>(a, queries, stream);
      return launch_for_d<MT, 128, true>(a, queries, stream);
    }
  }
#endif
  // the smallest tiling that holds the head dim; the padding costs its share of the MFMAs
  if (a.D <= 64) return launch_for_d<MT, 64, false>(a, queries, stream);
  if (a.D <= 96) return launch_for_d<MT, 96, false>(a, queries, stream);
  if (a.D <= 128) return launch_for_d<MT, 128, false>(a, queries, stream);
  if (a.D <= 192) return launch_wide_heads<MT, 192>(a, queries, stream);
  return launch_wide_heads<MT, 256>(a, queries, stream);
}

}  // namespace

bool prefill_mfma_supported(int dtype, int D) {
  return (dtype == LMH_F16 || dtype == LMH_BF16) && D >= 8 && (D <= 128 ? D % 8 == 0 : D <= 256 && D % 16 == 0);
}

int launch_prefill_mfma(const PrefillArgs &a, int dtype, hipStream_t stream, const QueryCopy &queries) {
#ifdef LMH_W64_KERNEL
  if (prefill_w64_takes(a, dtype)) return launch_prefill_w64(a, stream);
#endif
  if (dtype == LMH_F16) return launch_for_type<MfmaF16>(a, queries, stream);
  if (dtype == LMH_BF16) return launch_for_type<MfmaBF16>(a, queries, stream);
  return fail(LMH_E_UNSUPPORTED, "MFMA flash attention: dtype %d has no matrix-core path", dtype);
}

}  // namespace lmh
