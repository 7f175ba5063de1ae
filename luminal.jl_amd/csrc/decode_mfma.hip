// Single-token GQA decode attention on the matrix cores (fp16 / bf16 caches).
//
// Decode is HBM-bound: the only thing that matters is keeping >= 6 TB/s of K/V reads in flight.
// On the vector ALUs the 2*G flops per cache element (plus 16-bit unpacking and the cross-lane
// dot-product reductions) keep the VALUs ~60 % busy at 5 TB/s, which caps the kernel below the
// memory roofline. The matrix cores are otherwise idle, so the G query heads of a KV head are
// padded to a 16-wide MFMA operand and both products run as v_mfma_f32_16x16x32: per 32 keys of
// head dim 128 a wave then issues 16 MFMAs and ~200 VALU instructions instead of ~900, and the
// kernel is left waiting on memory only. (Same semantics as decode.hip: reference src/Whisper.jl:584-620 with the
// GQA head sharing of src/NN.jl:305-317.)
//
// Data flow per wave, 32 keys at a time (each wave owns a private LDS region, so the loop has no
// workgroup barrier):
//   global --128-bit coalesced loads (16 lanes per 256-byte row)--> registers (prefetched one
//   block ahead) --> LDS, row-major, padded rows
//   S^T[key, head] = K Q^T : A = K fragment (plain 128-bit LDS read), B = Q^T (registers, loaded once)
//   online softmax on the accumulator: lane (head n, g) holds keys 4g..4g+3 of each 16-key half; the
//   4 lanes of a head agree on the max through two lane exchanges
//   O^T[d, head] += V^T P^T : A = V^T fragment via the transposing LDS read ds_read_b64_tr_b16,
//   B = P^T = the softmax registers converted to 16 bit (never leaves the register file), as two (fp16)
//   or three (bf16) pieces so that P keeps 22 or 24 significant bits. Up to 8 (5) query heads per KV head
//   the pieces are columns of one product (COLUMNS); as products of their own the third took a walk of 512
//   keys from 10.5 to 11.2 us. Error of fp32 results against 64 bits (2-norm), L = 512 D = 128: bf16
//   1.6e-7 (two pieces: 1.9e-6), fp16 1.9e-7
//
// Scheduling: a rectangular (split, kv head, batch) grid wastes a ragged batch twice — workgroups
// whose split lies past kv_len[b] still have to be dispatched (≈40 % of the grid for lengths spread
// over [Lmax/4, Lmax]), and every workgroup pays its own ramp-up. Instead the kernel is persistent:
// the launch has as many workgroups as fit on the chip, every workgroup builds the prefix sum of
// ceil(kv_len[b] / chunk) over the batch in LDS, and takes an equal, contiguous share of the
// existing (b, kv head, chunk) units. Inside its share it streams through maximal runs of chunks of
// one (b, kv head) with a single softmax state, so partials are written once per run, not once per
// chunk (the other chunk slots of the run get an "empty" marker the merge kernel skips).
// Split-KV partial layout and the merge kernel are shared with decode.hip.
#include <algorithm>
#include <utility>

#include "common.hpp"
#include "copy.hpp"
#include "dtypes.hpp"
#include "rope.hpp"

namespace lmh {
namespace {

constexpr int kWaves = 4;
constexpr int kBlk = 32;  // keys per wave per step
constexpr float kLog2e = 1.4426950408889634f;

typedef short shortx8_t __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) shortx4_t lds_shortx4_t;

struct Mfma16F16Full;
struct Mfma16F16 {
  using full = Mfma16F16Full;
  static constexpr int kPieces = 2;
  static constexpr float kScale = 16384.f;  // of the weights: the second piece of one below 2^-3 would be subnormal
  using vec8 = half8_t;
  using elem = F16;
  __device__ static floatx4_t mfma(vec8 a, vec8 b, floatx4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
  __device__ static _Float16 cvt(float x) { return (_Float16)x; }
  __device__ static uint16_t cvt_bits(float x) { return __builtin_bit_cast(uint16_t, (_Float16)x); }
};
// Three pieces, 33 bits, at the head dims whose weights stayed in fp32 before this kernel took them (two: 2 to 5 % further from 64 bits).
struct Mfma16F16Full : Mfma16F16 {
  static constexpr int kPieces = 3;
};
struct Mfma16BF16 {
  using full = Mfma16BF16;
  static constexpr int kPieces = 3;
  static constexpr float kScale = 1.f;
  using vec8 = bf16x8_t;
  using elem = BF16;
  __device__ static floatx4_t mfma(vec8 a, vec8 b, floatx4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
  __device__ static __bf16 cvt(float x) { return (__bf16)x; }
  __device__ static uint16_t cvt_bits(float x) { return f32_to_bf16_bits(x); }
};

// Compiler-level ordering of one wave's LDS writes against its later LDS reads by other lanes.
// The hardware executes a wave's LDS instructions in order; this only pins the program order.
__device__ inline void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

constexpr int kMaxBatchPersistent = 1024;  // prefix sums live in LDS

// COLUMNS: the pieces of a head's weights are columns of one product. The 16 columns hold the heads of a slice kPieces times, so
// that their scores come out once per copy; the lanes of copy x take piece x, and the copies of O are added where the waves' are.
// Softmax and second product of a wave's 32 keys from key0 on, whose raw scores of head n are in sacc: lane (n, g) holds keys
// 4 g .. 4 g + 3 of each 16. `end`: the first key that does not exist; v_xor: how the lane's rows of V are swizzled; GB: row blocks
// whose products are on their way together.
template <typename MT, int D, bool COLUMNS, int GB, int LDV>
__device__ __forceinline__ void attend_block(floatx4_t (&sacc)[2], int key0, int end, int g, int copy, float c, const uint16_t *v_frag, int v_xor, float &m_i,
                                             float &l_i, floatx4_t (&oacc)[D / 16]) {
  using vec8 = typename MT::vec8;
  constexpr int DB = D / 16;
  if (key0 + kBlk > end) {  // ragged last block
#pragma unroll
    for (int hb = 0; hb < 2; hb++)
#pragma unroll
      for (int i = 0; i < 4; i++)
        if (key0 + 16 * hb + 4 * g + i >= end) sacc[hb][i] = -INFINITY;
  }

  // ---- online softmax; lane (n, g) owns head n ----
  float mx = fmaxf(fmaxf(fmaxf(sacc[0][0], sacc[0][1]), fmaxf(sacc[0][2], sacc[0][3])),
                   fmaxf(fmaxf(sacc[1][0], sacc[1][1]), fmaxf(sacc[1][2], sacc[1][3])));
  mx = max_over_wave_rows(mx);
  // (finite: key0 < end, so every head sees a key in this block.) The product is rounded before anything is subtracted from it:
  // old and new weights then differ by exactly the factor alpha, whatever the rounding
  const float mc = fmaxf(m_i, mx * c);
  const float alpha = __builtin_amdgcn_exp2f(m_i - mc);
  m_i = mc;
  // P is split into 16-bit pieces that hold all of it that fp32 sums see (two of fp16, 22 bits, or three of bf16, 24), and each is
  // multiplied with V: the matrix cores have time to spare here, and the result depends on where the split boundaries fall by
  // fp32 roundings only.
  float psum = 0.f;
  vec8 pf[COLUMNS ? 1 : MT::kPieces];
#pragma unroll
  for (int hb = 0; hb < 2; hb++)
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const float p = __builtin_amdgcn_exp2f(sacc[hb][i] * c - mc);
      psum += p;
      float rest = p * MT::kScale;
#pragma unroll
      for (int x = 0; x < MT::kPieces; x++) {
        const auto piece = MT::cvt(rest);
        rest -= (float)piece;
        if (!COLUMNS || x == 0 || copy >= x) pf[COLUMNS ? 0 : x][4 * hb + i] = piece;
      }
    }
  l_i = l_i * alpha + psum;
#pragma unroll
  for (int db = 0; db < DB; db++) oacc[db] *= alpha;

  // ---- O^T += V^T P^T: a block's share from zero, the first pieces apart from the others, added once ----
#pragma unroll
  for (int b0 = 0; b0 < DB; b0 += GB) {
    floatx4_t o[GB], rest[GB];
#pragma unroll
    for (int i = 0; i < GB; i++) {
      const uint16_t *vaddr = v_frag + ((16 * (b0 + i)) ^ v_xor);
      const shortx4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_shortx4_t *)(vaddr));
      const shortx4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_shortx4_t *)(vaddr + 16 * LDV));
      const vec8 v8 = __builtin_bit_cast(vec8, (shortx8_t)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
      o[i] = MT::mfma(v8, pf[0], floatx4_t{0.f, 0.f, 0.f, 0.f});
      if constexpr (!COLUMNS) {
        rest[i] = MT::mfma(v8, pf[MT::kPieces - 1], floatx4_t{0.f, 0.f, 0.f, 0.f});
        if (MT::kPieces == 3) rest[i] = MT::mfma(v8, pf[1], rest[i]);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < GB; i++)
#pragma unroll
      for (int e = 0; e < 4; e++) oacc[b0 + i][e] += COLUMNS ? o[i][e] : o[i][e] + rest[i][e];
  }
}

// What the split kernel divides by in front of its first load. Five divisions of 25 to 40 instructions, one behind the other, went with
// it, and with the branches around the loads of q the wait for all of them: steps of fp16 B=4 L=4096 D=128 17.5 -> 16.7 us, bf16 B=1 L=8192
// 16.0 -> 15.2, decodes of B=4 L=4096 16.3 -> 16.0, B=64 L=512 ragged 16.8 -> 16.3.
struct DecodeDeal {
  int32_t group, g_chunks;  // query heads of a KV head, and in slices of 16
  FastDiv by_chunk, by_g_chunks, by_grid;
};

template <typename MT, int D, bool COLUMNS>
__global__ __launch_bounds__(kWaves * 64) void decode_mfma_kernel(DecodeDeal deal, DecodeArgs a) {
  request_arg(deal.group);
  request_args(a);
  using vec8 = typename MT::vec8;
  static_assert(D % 16 == 0 && D <= 256, "whole row blocks of O^T, whole loads of a tile");
  constexpr int KS = (D + 31) / 32;      // k-steps of S^T = K Q^T
  constexpr bool kHalfStep = D % 32 != 0;  // half of the last one is zeros
  constexpr int DB = D / 16;             // 16-row blocks of O^T
  constexpr int CPR = D / 8;             // 16-byte chunks per cache row
  constexpr int NL = kBlk * CPR / 64;    // 128-bit loads per lane per 32-key tile
  constexpr int LDK = D + 8;             // LDS row strides (elements): chosen so that the 16 rows a
  constexpr int LDV = D % 32 ? D : D + 16;  // fragment read touches fall on different banks
  constexpr int kTileBytes = kBlk * (LDK + LDV) * 2;
  // rows of the waves' sums, in floats: as rows of D the sixteen heads fall on the same banks (D=256 B=2 Hkv=2 L=3000 fp16 20.8 -> 19.2
  // us, D=128 B=64 Hkv=8 L=512 ragged 19.4 -> 18.6, B=16 L=4096 49.4 -> 48.8)
  constexpr int LDO = D + 4;
  constexpr int kMergeBytes = kWaves * 16 * (LDO + 2) * 4;
  constexpr int kSmemBytes = kWaves * kTileBytes > kMergeBytes ? kWaves * kTileBytes : kMergeBytes;
  __shared__ __attribute__((aligned(16))) unsigned char smem[kSmemBytes];
  __shared__ int s_pref[kMaxBatchPersistent + 1];  // s_pref[b] = chunks of sequences 0..b-1
  __shared__ int s_len[kMaxBatchPersistent];       // keys of sequence b

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int n = lane & 15, g = lane >> 4;
  const int group = deal.group, g_chunks = deal.g_chunks;
  const int kv_slots = a.Hkv * g_chunks;  // (kv head, slice of <= 16 group members) pairs

  // ---- this workgroup's share of the (b, kv slot, chunk) units ----
  // s_pref = exclusive prefix sum of the chunks per sequence. Without kv_len it is a closed form; with it, the
  // first wave scans 64 sequences at a time with lane shifts (a serial loop over B = 64 by one thread was 3 us).
  if (!a.kv_len) {
    const int per_seq = (int)((uint32_t)(a.Lmax + a.chunk - 1) / deal.by_chunk);
    for (int i = tid; i <= a.B; i += kWaves * 64) {
      s_pref[i] = i * per_seq;
      if (i < a.B) s_len[i] = a.Lmax;
    }
  } else if (wave == 0) {
    int carry = 0;
    for (int base = 0; base < a.B; base += 64) {
      const int i = base + lane;
      int v = 0;
      if (i < a.B) {
        const int len = min(max(a.kv_len[i], 0), a.Lmax);
        s_len[i] = len;
        v = (int)((uint32_t)(len + a.chunk - 1) / deal.by_chunk);
      }
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const int up = __shfl_up(v, off);
        if (lane >= off) v += up;
      }
      if (i < a.B) s_pref[i + 1] = carry + v;
      carry += __shfl(v, 63);
    }
    if (lane == 0) s_pref[0] = 0;
  }
  __syncthreads();
  // Equal contiguous shares of the units, in 32-bit arithmetic (the launcher routes batches with 2^31 units or more to
  // the other kernel): the first total % grid workgroups take one unit more. 64-bit divisions are ~100 scalar
  // instructions each on this hardware, and five of them stood between a workgroup's start and its first load.
  const uint32_t total_units = (uint32_t)s_pref[a.B] * (uint32_t)kv_slots;
  const uint32_t share = total_units / deal.by_grid, extra = total_units - share * gridDim.x;
  uint32_t u = blockIdx.x * share + min((uint32_t)blockIdx.x, extra);
  const uint32_t u_end = u + share + (blockIdx.x < extra ? 1u : 0u);

  // Per-lane byte offsets of the NL 16-byte loads of a 32-key block, relative to the block's first row: load r of lane l
  // fetches chunk (r * 64 + l) of the block, i.e. row (r * 64 + l) / CPR, 16-byte column (r * 64 + l) % CPR. They do not
  // depend on the block, so they are computed once; a block's own position goes into the scalar offset of the load.
  int k_voff[NL], v_voff[NL];
#pragma unroll
  for (int r = 0; r < NL; r++) {
    const int id = r * 64 + lane;
    k_voff[r] = (int)(((id / CPR) * a.ks[2] + (id % CPR) * 8) * 2);
    v_voff[r] = (int)(((id / CPR) * a.vs[2] + (id % CPR) * 8) * 2);
  }
  const int k_row_bytes = (int)(a.ks[2] * 2), v_row_bytes = (int)(a.vs[2] * 2);

  uint16_t *Ks = reinterpret_cast<uint16_t *>(smem + wave * kTileBytes);
  uint16_t *Vs = Ks + kBlk * LDK;
  const float c = a.scale * kLog2e;
  const int k_frag_off = n * LDK + 8 * g;                             // + 16*hb*LDK + 32*ks
  const int v_frag_off = (4 * g + (n >> 2)) * LDV + 4 * (n & 3);      // + 16*hb*LDV + 16*db

  // A segment = the maximal run of units of one (b, kv slot) inside [u, u_end).
  struct Segment { int b, kvh, g0, n_heads, c0, c1, L, start, end, n_blocks; };
  auto next_segment = [&]() {
    Segment s;
    // largest b with s_pref[b] * kv_slots <= u, 64 sequences at a time (halving the range, one LDS read after the other, and
    // kv_len[b] from memory once more, stood in front of a segment's first load: steps of B=16 L=4096 D=128 50.3 -> 49.8 us, decodes of
    // B=64 L=512 ragged 18.6 -> 17.9, L=3000 93.5 -> 91.9)
    int b = -1;
    for (int base = 0; base < a.B; base += 64) {
      const int i = base + lane;
      b += __builtin_popcountll(__builtin_amdgcn_ballot_w64(i < a.B && (uint32_t)s_pref[i] * (uint32_t)kv_slots <= u));
    }
    s.b = b = __builtin_amdgcn_readfirstlane(b);
    const int n_chunks = s_pref[b + 1] - s_pref[b];
    const uint32_t rem = u - (uint32_t)s_pref[b] * (uint32_t)kv_slots;
    const int slot_id = (int)(rem / (uint32_t)n_chunks);
    s.c0 = (int)rem - slot_id * n_chunks;
    s.c1 = (int)min((uint32_t)n_chunks, s.c0 + (u_end - u));
    u += (uint32_t)(s.c1 - s.c0);
    s.kvh = (int)((uint32_t)slot_id / deal.by_g_chunks);
    s.g0 = (slot_id - s.kvh * g_chunks) * 16;  // first group member handled here
    s.n_heads = min(16, group - s.g0);
    s.L = s_len[b];
    s.start = s.c0 * a.chunk;
    s.end = min(s.L, s.c1 * a.chunk);
    s.n_blocks = (s.end - s.start + kBlk - 1) / kBlk;
    return s;
  };

  // Q^T fragments (B operand): lane (head n, g) holds q[head][32*ks + 8*g .. +7], the first head's for padding columns, which nothing
  // reads (no branch: with one, the wait for q is a wait for all loads)
  vec8 qreg[KS];
  int copy;
  // Raw buffer descriptors over the valid rows [0, end) of this (b, kv head) slice: a load past `end` returns zeros
  // without a branch, so the loads of a block are NL back-to-back instructions (address = lane-invariant offset +
  // scalar block offset). Non-temporal, like every cache stream of this library.
  __amdgpu_buffer_rsrc_t k_rsrc, v_rsrc;
  uint4 kreg[NL], vreg[NL];
  auto load_tile = [&](int key0) {
    const int k_soff = __builtin_amdgcn_readfirstlane(key0 * k_row_bytes);
    const int v_soff = __builtin_amdgcn_readfirstlane(key0 * v_row_bytes);
#pragma unroll
    for (int r = 0; r < NL; r++) {
      kreg[r] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(k_rsrc, k_voff[r], k_soff, 2));
      vreg[r] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(v_rsrc, v_voff[r], v_soff, 2));
    }
  };
  auto store_tile = [&]() {
#pragma unroll
    for (int r = 0; r < NL; r++) {
      const int id = r * 64 + lane;
      const int row = id / CPR, col = id % CPR;
      *reinterpret_cast<uint4 *>(&Ks[row * LDK + col * 8]) = kreg[r];
      *reinterpret_cast<uint4 *>(&Vs[row * LDV + col * 8]) = vreg[r];
    }
  };

  // q and the wave's first block of a segment on their way
  auto begin = [&](const Segment &s) {
    copy = COLUMNS ? n / s.n_heads : 0;
    const int head = n - copy * s.n_heads;
    const bool head_ok = COLUMNS ? copy < MT::kPieces : n < s.n_heads;
    const int hq = q_head_of(s.kvh, head_ok ? s.g0 + head : 0, a.Hq, a.Hkv, a.head_map);
    const uint16_t *qp = reinterpret_cast<const uint16_t *>(a.q) + s.b * a.qs[0] + hq * a.qs[1];
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
      const bool in = !kHalfStep || ks < KS - 1 || g < 2;
      uint4 x = *reinterpret_cast<const uint4 *>(qp + (in ? 32 * ks + 8 * g : 0));
      if (kHalfStep) x = make_uint4(in ? x.x : 0, in ? x.y : 0, in ? x.z : 0, in ? x.w : 0);
      qreg[ks] = __builtin_bit_cast(vec8, x);
    }
    const uint16_t *kbase = reinterpret_cast<const uint16_t *>(a.k) + s.b * a.ks[0] + s.kvh * a.ks[1];
    const uint16_t *vbase = reinterpret_cast<const uint16_t *>(a.v) + s.b * a.vs[0] + s.kvh * a.vs[1];
    k_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t *>(kbase), 0, __builtin_amdgcn_readfirstlane(s.end * k_row_bytes), 0x00020000);
    v_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t *>(vbase), 0, __builtin_amdgcn_readfirstlane(s.end * v_row_bytes), 0x00020000);
    load_tile(wave < s.n_blocks ? s.start + wave * kBlk : s.end);  // (behind the end: zeros, without a branch)
  };

  auto rotate_q = [&](int L) {
    // lmh_decode_step: this step's query is rotated at the position of the row the step appends, kv_len[b], as it is
    // loaded (apply_rotary_embeddings on the queries, reference src/NN.jl:356). Lane (n, g) holds elements
    // 32 ks + 8 g + e: the partner j + D/2 sits in fragment ks + KS/2 of the same lane when KS is even (the launcher
    // sends other head dims elsewhere), interleaved partners are neighbours inside a fragment.
    // The position is the sequence's, so a lane evaluates pair `lane` (and lane + 64) and the others fetch it from there. With every
    // pair of its own evaluated by each lane, 16 to 64 sines in a row, steps of B=16 L=4096 D=128 took 48.1 us instead of 47.0, B=4
    // 18.5 instead of 17.3 (17.9 and 16.8 without a rotation: a tenth of the kernel's code), B=4 Hkv=4 L=3000 D=256 22.1 instead of 20.1.
    if (a.q_rope) {
      float sn[(D + 127) / 128], cs[(D + 127) / 128];
#pragma unroll
      for (int i = 0; i < (D + 127) / 128; i++) {
        int j = 64 * i + lane;
        asm volatile("" : "+v"(j));  // (the frequency stays here and is not evaluated in front of everything, also where nothing rotates)
        sincos_angle((float)L * rope_inv_freq(j, D, a.rope_log2_base), &sn[i], &cs[i]);
      }
      auto from = [&](const float *x, int j0, int j) { return __int_as_float(__builtin_amdgcn_ds_bpermute(4 * (j0 % 64 + j), __float_as_int(x[j0 / 64]))); };
      if (!a.rope_interleaved) {
        if constexpr (KS % 2 == 0) {
          constexpr int HK = KS / 2;
#pragma unroll
          for (int ks = 0; ks < HK; ks++)
#pragma unroll
            for (int e = 0; e < 8; e++) {
              float o0, o1;
              rope_rotate((float)qreg[ks][e], (float)qreg[ks + HK][e], from(sn, 32 * ks, 8 * g + e), from(cs, 32 * ks, 8 * g + e), &o0, &o1);
              qreg[ks][e] = MT::cvt(o0);
              qreg[ks + HK][e] = MT::cvt(o1);
            }
        }
      } else {
#pragma unroll
        for (int ks = 0; ks < KS; ks++)
#pragma unroll
          for (int e = 0; e < 8; e += 2) {
            float o0, o1;
            rope_rotate((float)qreg[ks][e], (float)qreg[ks][e + 1], from(sn, 16 * ks, (8 * g + e) / 2), from(cs, 16 * ks, (8 * g + e) / 2), &o0, &o1);
            qreg[ks][e] = MT::cvt(o0);
            qreg[ks][e + 1] = MT::cvt(o1);
          }
      }
    }
  };

  Segment seg = {};
  bool more = u < u_end;
  if (more) {
    seg = next_segment();
    begin(seg);
  }
  while (more) {
  rotate_q(seg.L);  // (after the first loads are on their way: the rotation is in front of the first score)
  floatx4_t oacc[DB];
#pragma unroll
  for (int db = 0; db < DB; db++) oacc[db] = floatx4_t{0.f, 0.f, 0.f, 0.f};
  float m_i = -INFINITY;  // running max of the scores of head n in log2 units, as the weights have it (same in the 4 lanes of a head)
  float l_i = 0.f;        // this lane's share of the running sum

  for (int blk = wave; blk < seg.n_blocks; blk += kWaves) {
    const int key0 = seg.start + blk * kBlk;
    wave_lds_fence();  // the previous block's fragment reads precede these writes
    store_tile();
    wave_lds_fence();
    if (blk + kWaves < seg.n_blocks) load_tile(key0 + kWaves * kBlk);  // in flight during the math below

    // ---- S^T = K Q^T for the two 16-key halves ----
    floatx4_t sacc[2];
#pragma unroll
    for (int hb = 0; hb < 2; hb++) {
      sacc[hb] = floatx4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KS; ks++) {
        vec8 kf = *reinterpret_cast<const vec8 *>(&Ks[k_frag_off + 16 * hb * LDK + 32 * ks]);
        if (kHalfStep && ks == KS - 1) {  // (behind the row lies the next one, or V: zero times what they hold could be NaN)
          const uint4 x = __builtin_bit_cast(uint4, kf);
          kf = __builtin_bit_cast(vec8, make_uint4(g < 2 ? x.x : 0, g < 2 ? x.y : 0, g < 2 ? x.z : 0, g < 2 ? x.w : 0));
        }
        sacc[hb] = MT::mfma(kf, qreg[ks], sacc[hb]);
      }
    }
    attend_block<MT, D, COLUMNS, DB % 8 == 0 ? 8 : DB, LDV>(sacc, key0, seg.end, g, copy, c, Vs + v_frag_off, 0, m_i, l_i, oacc);
  }

  // The next segment's first blocks travel while this one's sums are folded (asked for behind them: decodes of B=64 H=32/8 L=3000 ragged
  // D=128 88.9 us instead of 87.4, B=100 L=1000 52.8 instead of 52.0, B=64 L=2000 D=64 28.8 instead of 28.4).
  const int b = seg.b, kvh = seg.kvh, g0 = seg.g0, n_heads = seg.n_heads, c0 = seg.c0, c1 = seg.c1;
  more = u < u_end;
  if (more) {
    seg = next_segment();
    begin(seg);
  }

  // ---- merge the 4 waves, then write the split partial (or the final output) ----
  l_i = sum_over_wave_rows(l_i);
  __syncthreads();  // all waves are done with their tiles: the memory is reused for the merge
  float *sm_o = reinterpret_cast<float *>(smem);              // [kWaves][16][LDO]
  float *sm_m = sm_o + kWaves * 16 * LDO;                       // [kWaves][16]
  float *sm_l = sm_m + kWaves * 16;                           // [kWaves][16]
#pragma unroll
  for (int db = 0; db < DB; db++)
#pragma unroll
    for (int i = 0; i < 4; i++) sm_o[(wave * 16 + n) * LDO + 16 * db + 4 * g + i] = oacc[db][i] * (1.f / MT::kScale);
  if (g == 0) {
    sm_m[wave * 16 + n] = m_i;
    sm_l[wave * 16 + n] = l_i;
  }
  __syncthreads();

  auto store = [&](int h, int d, float o, float M, float lsum) __attribute__((always_inline)) {
    const int hq = q_head_of(kvh, g0 + h, a.Hq, a.Hkv, a.head_map);
    if (a.num_splits == 1) {
      const int64_t off = b * a.os[0] + hq * a.os[1] + d;
      if (a.out_f32) reinterpret_cast<float *>(a.out)[off] = o / lsum;
      else reinterpret_cast<uint16_t *>(a.out)[off] = MT::cvt_bits(o / lsum);
    } else {
      const int64_t row = ((int64_t)b * a.Hq + hq) * a.num_splits + c0;
      a.ws_o[row * D + d] = o;
      if (d == 0) {
        a.ws_ml[row * 2 + 0] = M;
        a.ws_ml[row * 2 + 1] = lsum;
      }
    }
  };
  float finite = 0.f;  // no longer zero where a sum is infinite or no number
  for (int idx = tid; idx < n_heads * D; idx += kWaves * 64) {
    const int h = idx / D, d = idx % D;
    float M = -INFINITY;
#pragma unroll
    for (int w = 0; w < kWaves; w++) M = fmaxf(M, sm_m[w * 16 + h]);
    float lsum = 0.f, o = 0.f;
#pragma unroll
    for (int w = 0; w < kWaves; w++) {
      const float mw = sm_m[w * 16 + h];
      const float f = (mw == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f(mw - M);
      lsum += sm_l[w * 16 + h] * f;
      float x = sm_o[(w * 16 + h) * LDO + d];
      if constexpr (COLUMNS) {
        float rest = sm_o[(w * 16 + (MT::kPieces - 1) * n_heads + h) * LDO + d];
        if (MT::kPieces == 3) rest += sm_o[(w * 16 + n_heads + h) * LDO + d];
        x += rest;
      }
      o += x * f;
    }
    store(h, d, o, M, lsum);
    if (kHalfStep) finite = fmaf(o, 0.f, finite);
  }
  // An infinite value of V times pieces of a weight, some of them negative or zero, is no number; times the weight it is infinite, and
  // was so where the vector ALUs took this head dim. A wave takes a head's keys again, 64 at a time, with the weights in fp32.
  if constexpr (kHalfStep) {
    if (__syncthreads_or(finite != 0.f)) {
      const int start = c0 * a.chunk, end = min(s_len[b], c1 * a.chunk);
      const uint16_t *kbase = reinterpret_cast<const uint16_t *>(a.k) + b * a.ks[0] + kvh * a.ks[1];
      const uint16_t *vbase = reinterpret_cast<const uint16_t *>(a.v) + b * a.vs[0] + kvh * a.vs[1];
      using E = typename MT::elem;
      using raw = typename E::raw;
      for (int h = wave; h < n_heads; h += kWaves) {
        const raw *qp = reinterpret_cast<const raw *>(a.q) + b * a.qs[0] + q_head_of(kvh, g0 + h, a.Hq, a.Hkv, a.head_map) * a.qs[1];
        float M = -INFINITY, lsum = 0.f, o[(D + 63) / 64] = {};
#pragma unroll
        for (int w = 0; w < kWaves; w++) M = fmaxf(M, sm_m[w * 16 + h]);
#pragma unroll
        for (int w = 0; w < kWaves; w++) lsum += sm_m[w * 16 + h] == -INFINITY ? 0.f : sm_l[w * 16 + h] * __builtin_amdgcn_exp2f(sm_m[w * 16 + h] - M);
        for (int key0 = start; key0 < end; key0 += 64) {
          const int n_keys = min(64, end - key0);
          float dot = 0.f;
          if (lane < n_keys) {
            const raw *kp = reinterpret_cast<const raw *>(kbase) + (int64_t)(key0 + lane) * a.ks[2];
            for (int d = 0; d < D; d++) dot = fmaf(E::ld(qp[d]), E::ld(kp[d]), dot);
          }
          const float p = __builtin_amdgcn_exp2f(fmaf(dot, c, -M));
          for (int j = 0; j < n_keys; j++) {
            const float pj = __shfl(p, j);
            const raw *vp = reinterpret_cast<const raw *>(vbase) + (int64_t)(key0 + j) * a.vs[2];
#pragma unroll
            for (int i = 0; i < (D + 63) / 64; i++)
              if (64 * i + lane < D) o[i] = fmaf(pj, E::ld(vp[64 * i + lane]), o[i]);
          }
        }
#pragma unroll
        for (int i = 0; i < (D + 63) / 64; i++)
          if (64 * i + lane < D) store(h, 64 * i + lane, o[i], M, lsum);
      }
    }
  }
  // the other chunk slots of this run hold nothing: mark them so the merge kernel skips them
  if (a.num_splits > 1) {
    for (int idx = tid; idx < n_heads * (c1 - c0 - 1); idx += kWaves * 64) {
      const int h = idx / (c1 - c0 - 1), cs = c0 + 1 + idx % (c1 - c0 - 1);
      const int hq = q_head_of(kvh, g0 + h, a.Hq, a.Hkv, a.head_map);
      const int64_t row = ((int64_t)b * a.Hq + hq) * a.num_splits + cs;
      a.ws_ml[row * 2 + 0] = -INFINITY;
      a.ws_ml[row * 2 + 1] = 0.f;
    }
  }
  __syncthreads();  // the merge buffers are tile memory again in the next segment
  }  // while (more)

  // A sequence without keys has no unit. With several splits the merge kernel writes its zeros; with one split
  // nothing else would write its output rows.
  if (a.num_splits == 1) {
    for (int b = blockIdx.x; b < a.B; b += gridDim.x) {
      if (s_pref[b + 1] != s_pref[b]) continue;
      for (int idx = tid; idx < a.Hq * D; idx += kWaves * 64) {
        const int64_t off = b * a.os[0] + (idx / D) * a.os[1] + idx % D;
        if (a.out_f32) reinterpret_cast<float *>(a.out)[off] = 0.f;
        else reinterpret_cast<uint16_t *>(a.out)[off] = 0;
      }
    }
  }
}

// A (b, kv head slice) pair's whole walk in one workgroup, for the launches that decode_by_pairs names: no partials in memory and no
// second launch. What bounds these launches is latency: the kernel's chain of round trips and barriers, and the start
// of a second kernel behind it. So as many waves as LDS holds take a 32-key block each (256 keys at once at D = 128), straight into LDS
// in whole rows (K into the MFMA's layout, 16 rows x 64 bytes a load, reads every line twice: a step of 512 keys 12.6 us, 10.5 this
// way), and q, which every wave needs, is rotated once by the whole workgroup. Bank conflicts of the sums' rows and of V's transposing
// read were 2.4 of those 10.5 us. A step's new row is one more partial of the merge of the waves, as in decode_merge_kernel, and the
// copies of a fed step are further workgroups.
template <int D> constexpr int pair_waves() { return D > 128 ? 4 : D > 96 ? 8 : D > 64 ? 12 : 16; }
template <typename MT, int D, bool COLUMNS>
__global__ __launch_bounds__(64 * pair_waves<D>()) void decode_pair_kernel(DecodeArgs a, int group, CopyManyArgs fed, int n_copies) {
  constexpr int NW = pair_waves<D>(), NT = 64 * NW;
  if ((int)blockIdx.z >= a.B) {
    constexpr int CT = NT >= 1024 ? 1024 : NT >= 512 ? 512 : 256;  // threads that divide a chunk of the copies
    const int block = ((blockIdx.z - a.B) * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x;
    if (block < n_copies && threadIdx.x < CT) copy_block<CT>(fed, block);
    return;
  }
  request_args(a);
  request_arg(group);
  using vec8 = typename MT::vec8;
  using E = typename MT::elem;
  using raw = typename E::raw;
  constexpr int KS = D / 32, DB = D / 16, CPR = D / 8, NL = kBlk * CPR / 64;
  constexpr int LDQ = D + 8;
  constexpr int kTile = NW * 2 * kBlk * D * 2, LDO = D + 4, kMerge = NW * 16 * LDO * 4;
  __shared__ __attribute__((aligned(16))) unsigned char smem[kTile > kMerge ? kTile : kMerge];  // K and V tiles, then the waves' sums
  __shared__ __attribute__((aligned(16))) raw q_s[16 * LDQ], k_s[D], v_s[D], row_s[NW][D];
  __shared__ float sm_m[NW * 16], sm_l[NW * 16], sm_f[NW * 16], new_s[16], total_s[16], new_w[16];

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15, g = lane >> 4;
  const int b = blockIdx.z, kvh = blockIdx.x, g0 = 16 * blockIdx.y, n_heads = min(16, group - g0);
  // (a scalar load, which is not counted with the loads of the tiles, and no branch, which would wait for it; without kv_len any word)
  typedef const __attribute__((address_space(4))) int32_t constant_int_t;
  const int length = *(constant_int_t *)(a.kv_len ? (uintptr_t)(a.kv_len + b) : (uintptr_t)a.q);
  const int head0 = a.head_map == LMH_HEADMAP_BLOCKED ? kvh * group + g0 : kvh + a.Hkv * g0, head_step = a.head_map == LMH_HEADMAP_BLOCKED ? 1 : a.Hkv;
  auto head_at = [&](int h) { return head0 + h * head_step; };  // q_head_of

  // ---- tiles: global memory -> LDS directly, in whole rows (see prefill_mfma.hip for the asm). Load r of a block fetches its chunks
  // r * 64 .. + 63; the descriptor ends with the cache, past it zeros arrive. The first block is fetched without waiting for kv_len:
  // rows past it are masked (K) and cleared (V) below. Chunk j of row i of K lies at j ^ (i % 16) (of a
  // row of 8 or 16 chunks or more), so that a fragment read, 16 rows x 64 bytes, falls on all banks; V's likewise in pairs. ----
  typedef int32_t i32x4_t __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) void lds_void_t;
  constexpr int kSwizzle = CPR == 8 ? 7 : CPR % 16 == 0 ? 15 : 0, kSwizzleV = kSwizzle & ~1;
  const int k_row_bytes = (int)(a.ks[2] * 2), v_row_bytes = (int)(a.vs[2] * 2);
  auto make_desc = [](const void *base, int64_t offset, int bytes) {
    const uint64_t p = (uint64_t)base + 2 * offset;
    i32x4_t d;
    d[0] = __builtin_amdgcn_readfirstlane((int)(uint32_t)p);
    d[1] = __builtin_amdgcn_readfirstlane((int)((p >> 32) & 0xffff));
    d[2] = __builtin_amdgcn_readfirstlane(bytes);
    d[3] = 0x00020000;
    return d;
  };
  const i32x4_t k_desc = make_desc(a.k, b * a.ks[0] + kvh * a.ks[1], a.Lmax * k_row_bytes), v_desc = make_desc(a.v, b * a.vs[0] + kvh * a.vs[1], a.Lmax * v_row_bytes);
  // (where a load is whole rows, its lanes' rows are the first load's and a scalar more: no product each)
  constexpr bool kWhole = 64 % CPR == 0;
  constexpr int kRows = kWhole ? 64 / CPR : 0;
  int k_voff[NL], v_voff[NL];
#pragma unroll
  for (int r = 0; r < NL; r++) {
    const int id = kWhole ? lane : r * 64 + lane, row = id / CPR, col = id % CPR, at = row + kRows * r;
    k_voff[r] = row * k_row_bytes + ((col ^ (at & kSwizzle)) * 16 + kRows * r * k_row_bytes);
    v_voff[r] = row * v_row_bytes + ((col ^ (2 * at & kSwizzleV)) * 16 + kRows * r * v_row_bytes);
  }
  const uint32_t k_lds = (uint32_t)(uintptr_t)(lds_void_t *)smem + wave * (2 * kBlk * D * 2), v_lds = k_lds + kBlk * D * 2;
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"  // m0 is a reserved register; it is only written here
  auto load_1k = [](i32x4_t desc, uint32_t lds, int voff, int soff) __attribute__((always_inline)) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen nt lds" :: "s"(lds), "v"(voff), "s"(desc), "s"(soff) : "memory", "m0");
  };
#pragma clang diagnostic pop
  auto load = [&](i32x4_t desc, uint32_t lds, const int (&voff)[NL], int soff) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < NL; r++) load_1k(desc, lds + r * 1024, voff[r], soff);
  };
  auto load_k = [&](int key0) __attribute__((always_inline)) { load(k_desc, k_lds, k_voff, key0 * k_row_bytes); };
  auto load_v = [&](int key0) __attribute__((always_inline)) { load(v_desc, v_lds, v_voff, key0 * v_row_bytes); };

  // ---- q and, for a step, its new key, rotated at position L and rounded to the element type, and the new value, through LDS: a
  // wave per row, whose elements arrive in front of the wave's keys. (Loaded behind those they were waited for with the keys and then
  // once more: with the branches of the merge below that was 8.4 us for a step of 512 keys, H=32/8 D=128, which takes 7.5, and 7.2 for a
  // decode of 322 keys, which takes 6.7.) ----
  const int rows = n_heads + (a.step ? 2 : 0);
  const int64_t new_row = ((int64_t)b * a.Hkv + kvh) * D;
  auto row_at = [&](int h) {
    const void *base = h < n_heads ? a.q : h == n_heads ? a.k_new : a.v_new;
    return reinterpret_cast<const raw *>(base) + (h < n_heads ? b * a.qs[0] + head_at(h) * a.qs[1] : new_row);
  };
  bool own_direct = false;
  const int own = NW - 1 - wave;  // (the last waves are the first to be left without keys)
  if (own < rows) {
    const raw *from = row_at(own);
    own_direct = ((uint64_t)from & 15) == 0;
    if (own_direct && lane < CPR) load_1k(make_desc(from, 0, D * 2), (uint32_t)(uintptr_t)(lds_void_t *)row_s[wave], lane * 16, 0);
  }
  if (wave * kBlk < a.Lmax) {
    load_k(wave * kBlk);
    load_v(wave * kBlk);
    asm volatile("s_waitcnt vmcnt(%0)" :: "n"(2 * NL) : "memory");  // the row is in LDS
  } else {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }
  const int L = a.kv_len ? min(max(length, 0), a.Lmax) : a.Lmax;
  const int n_blocks = (L + kBlk - 1) / kBlk;
  const bool append = a.step && L < a.Lmax;
  auto place = [&](int h, auto element) __attribute__((always_inline)) {
    raw *to = h < n_heads ? q_s + h * LDQ : h == n_heads ? k_s : v_s;
#pragma unroll 1
    for (int j = lane; j < D / 2; j += 64) {
      const int d0 = a.rope_interleaved ? 2 * j : j, d1 = a.rope_interleaved ? 2 * j + 1 : j + D / 2;
      raw x0 = element(d0), x1 = element(d1);
      if (a.q_rope && h <= n_heads) {
        float o0, o1;
        rope_pair(E::ld(x0), E::ld(x1), (float)L, j, D, a.rope_log2_base, &o0, &o1);
        x0 = E::st(o0);
        x1 = E::st(o1);
      }
      to[d0] = x0;
      to[d1] = x1;
    }
  };
  const int n_rows = n_heads + (append ? 2 : 0);
  if (own_direct && own < n_rows) place(own, [&](int d) { return row_s[wave][d]; });
#pragma unroll 1
  for (int h = own_direct ? own + NW : own; h < n_rows; h += NW) {
    const raw *from = row_at(h);
    place(h, [&](int d) { return from[d]; });
  }
  __syncthreads();
  const int copy = !COLUMNS ? 0 : (n >= n_heads) + (n >= 2 * n_heads) + (MT::kPieces > 2 && n >= 3 * n_heads), head = n - copy * n_heads;
  const bool head_ok = COLUMNS ? copy < MT::kPieces : n < n_heads;
  vec8 qreg[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ks++) {
    uint4 x = make_uint4(0, 0, 0, 0);
    if (head_ok) x = *reinterpret_cast<const uint4 *>(&q_s[head * LDQ + 32 * ks + 8 * g]);
    qreg[ks] = __builtin_bit_cast(vec8, x);
  }
  const float c = a.scale * kLog2e;
  if (append) {  // the new row's scores, a head per wave
    for (int h = wave; h < n_heads; h += NW) {
      float dot = 0.f;
      for (int d = lane; d < D; d += 64) dot += E::ld(q_s[h * LDQ + d]) * E::ld(k_s[d]);
#pragma unroll
      for (int o = 32; o >= 1; o >>= 1) dot += __shfl_xor(dot, o);
      if (lane == 0) new_s[h] = dot * a.scale * kLog2e;
    }
  }

  floatx4_t oacc[DB];
#pragma unroll
  for (int db = 0; db < DB; db++) oacc[db] = floatx4_t{0.f, 0.f, 0.f, 0.f};
  float m_i = -INFINITY, l_i = 0.f;
  uint16_t *const k_tile = reinterpret_cast<uint16_t *>(smem) + wave * (2 * kBlk * D);
  const int v_row = 4 * g + (n >> 2), v_xor = (2 * v_row & kSwizzleV) * 8;  // (and row v_row + 16)
  const uint16_t *v_frag = k_tile + kBlk * D + v_row * D + 4 * (n & 3);
  for (int blk = wave; blk < n_blocks; blk += NW) {
    const int key0 = blk * kBlk;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the block is in LDS
    floatx4_t sacc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int ks = 0; ks < KS; ks++)
#pragma unroll
      for (int hb = 0; hb < 2; hb++) {
        const vec8 kf = *reinterpret_cast<const vec8 *>(k_tile + (16 * hb + n) * D + ((4 * ks + g) ^ (n & kSwizzle)) * 8);
        sacc[hb] = MT::mfma(kf, qreg[ks], sacc[hb]);
      }
    if (blk + NW < n_blocks) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // every read of this block's K has returned
      load_k(key0 + NW * kBlk);
    }
    if (key0 + kBlk > L) {  // (zero times what lies past the last row could be NaN)
#pragma unroll
      for (int r = 0; r < NL; r++)
        if (r * 64 + lane >= (L - key0) * CPR) *reinterpret_cast<uint4 *>(k_tile + kBlk * D + (r * 64 + lane) * 8) = make_uint4(0, 0, 0, 0);
      wave_lds_fence();
    }
    attend_block<MT, D, COLUMNS, DB % 4 == 0 ? 4 : DB, D>(sacc, key0, L, g, copy, c, v_frag, v_xor, m_i, l_i, oacc);
    if (blk + NW < n_blocks) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // every read of this block's V has returned
      load_v(key0 + NW * kBlk);
    }
  }

  // ---- merge the waves and the new row: the waves' factors against the common maximum first ----
  l_i = sum_over_wave_rows(l_i);
  if (g == 0) {
    sm_m[wave * 16 + n] = m_i;
    sm_l[wave * 16 + n] = l_i;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (blocks fetched for nobody)
  __syncthreads();  // all waves are done with their tiles: the memory is reused for the merge
  float *sm_o = reinterpret_cast<float *>(smem);  // [NW][16][LDO]
  const int used = min(NW, n_blocks);
  {
    const float m_new = append && head_ok ? new_s[head] : -INFINITY;
    float M = m_new, tops[NW];
#pragma unroll
    for (int w = 0; w < NW; w++) M = fmaxf(M, tops[w] = sm_m[w * 16 + n]);
    if (wave < used) {
      if (g == 0) sm_f[wave * 16 + n] = __builtin_amdgcn_exp2f(m_i - M);
#pragma unroll
      for (int db = 0; db < DB; db++)
#pragma unroll
        for (int i = 0; i < 4; i++) sm_o[(wave * 16 + n) * LDO + 16 * db + 4 * g + i] = oacc[db][i] * (1.f / MT::kScale);
    }
    if (wave == NW - 1 && g == 0 && n < n_heads) {
      const float w_new = append ? __builtin_amdgcn_exp2f(m_new - M) : 0.f;  // the new row's sum is 1
      float part[4] = {0.f, 0.f, 0.f, 0.f};  // (four shorter sums are rounded less than one)
      // (waves without keys add zeros; branches around them, here and below, would make a round trip to LDS of each)
#pragma unroll
      for (int w = 0; w < NW; w++) part[w & 3] += sm_l[w * 16 + n] * __builtin_amdgcn_exp2f(tops[w] - M);
      total_s[n] = used == 0 && !append ? 1.f : (part[0] + part[1]) + (part[2] + part[3]) + w_new;  // no key: zeros
      new_w[n] = w_new;
    }
  }
  __syncthreads();
  // the new row's place in the caches (in front of the keys, the wait for them would be one for these stores)
  if (append && g0 == 0) {
    raw *k_dst = const_cast<raw *>(reinterpret_cast<const raw *>(a.k)) + b * a.ks[0] + kvh * a.ks[1] + (int64_t)L * a.ks[2];
    raw *v_dst = const_cast<raw *>(reinterpret_cast<const raw *>(a.v)) + b * a.vs[0] + kvh * a.vs[1] + (int64_t)L * a.vs[2];
    for (int d = tid; d < D; d += NT) {
      k_dst[d] = k_s[d];
      v_dst[d] = v_s[d];
    }
  }
  for (int idx = tid; idx < n_heads * D; idx += NT) {
    const int h = idx / D, d = idx % D;
    float part[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w0 = 0; w0 < NW; w0 += 4) {
      if (w0 >= used) break;
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int w = w0 + u;
        float x = sm_o[(w * 16 + h) * LDO + d];
        if constexpr (COLUMNS) {
          float rest = sm_o[(w * 16 + (MT::kPieces - 1) * n_heads + h) * LDO + d];
          if (MT::kPieces == 3) rest += sm_o[(w * 16 + n_heads + h) * LDO + d];
          x += rest;
        }
        x *= sm_f[w * 16 + h];
        part[u] += w < used ? x : 0.f;  // (what lies in LDS for waves without keys is read and thrown away)
      }
    }
    float o = (part[0] + part[1]) + (part[2] + part[3]);
    if (append) o += new_w[h] * E::ld(v_s[d]);
    const float out = o / total_s[h];
    const int64_t off = b * a.os[0] + head_at(h) * a.os[1] + d;
    if (a.out_f32) reinterpret_cast<float *>(a.out)[off] = out;
    else reinterpret_cast<uint16_t *>(a.out)[off] = MT::cvt_bits(out);
  }
}

template <typename MT, int D, bool COLUMNS>
int launch_form(const DecodeArgs &a, hipStream_t stream) {
  // Persistent launch: as many workgroups as the chip holds at once (never more than there are units). Same for every device this
  // library runs on (gfx950 only); initialised once, thread-safely.
  static const int per_cu = [] {
    int n = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, decode_mfma_kernel<MT, D, COLUMNS>, kWaves * 64, 0) != hipSuccess) {
      (void)hipGetLastError();
      return 1;  // correct for any value, only the balance changes
    }
    return n < 1 ? 1 : n;
  }();
  // With several splits every further workgroup is a further partial row for the merge to read: one per CU, two up to head dim 96
  // (bf16 steps D = 128 B=32 L=1024: 30.8 us, 32.2 with two). With one split, as many as fit (fp16 B=64 L=512 ragged 20.1 and 22.4).
  const int wgs_per_device = device_cu_count() * (a.num_splits > 1 ? std::min(per_cu, D > 96 ? 1 : 2) : per_cu);
  const int group = a.Hq / a.Hkv;
  const int g_chunks = (group + 15) / 16;
  const int64_t max_units = (int64_t)a.B * a.Hkv * g_chunks * a.num_splits;
  if (max_units >= (int64_t(1) << 31)) return fail(LMH_E_UNSUPPORTED, "MFMA decode: %lld units do not fit 32 bits", (long long)max_units);
  const int n_wgs = (int)(max_units < wgs_per_device ? max_units : wgs_per_device);
  const DecodeDeal deal = {group, g_chunks, fast_div(a.chunk), fast_div(g_chunks), fast_div(n_wgs)};
  hipLaunchKernelGGL((decode_mfma_kernel<MT, D, COLUMNS>), dim3(n_wgs), dim3(kWaves * 64), 0, stream, deal, a);
  LMH_HIP_TRY(hipGetLastError());
  return LMH_OK;
}

template <typename MT, int D, bool COLUMNS>
int launch_pair(const DecodeArgs &a, const CopyManyArgs *fed, int n_copies, hipStream_t stream) {
  const int group = a.Hq / a.Hkv, g_chunks = (group + 15) / 16, per = a.Hkv * g_chunks;
  const CopyManyArgs copies = n_copies ? *fed : CopyManyArgs{};
  hipLaunchKernelGGL((decode_pair_kernel<MT, D, COLUMNS>), dim3(a.Hkv, g_chunks, a.B + (n_copies + per - 1) / per), dim3(64 * pair_waves<D>()), 0,
                     stream, a, group, copies, n_copies);
  LMH_HIP_TRY(hipGetLastError());
  return LMH_OK;
}

template <typename MT, int D>
int launch_for_d(const DecodeArgs &a, const CopyManyArgs *fed, int n_copies, hipStream_t stream) {
  const bool columns = a.Hq / a.Hkv * MT::kPieces <= 16;
  if constexpr (D % 32 == 0)
    if (a.num_splits == 1 && (a.step || decode_by_pairs(a))) return columns ? launch_pair<MT, D, true>(a, fed, n_copies, stream) : launch_pair<MT, D, false>(a, fed, n_copies, stream);
  return columns ? launch_form<MT, D, true>(a, stream) : launch_form<MT, D, false>(a, stream);
}

template <typename MT>
int launch_for_type(const DecodeArgs &a, const CopyManyArgs *fed, int n_copies, hipStream_t stream) {
  switch (a.D) {
    case 64: return launch_for_d<MT, 64>(a, fed, n_copies, stream);
    case 80: return launch_for_d<typename MT::full, 80>(a, fed, n_copies, stream);
    case 96: return launch_for_d<MT, 96>(a, fed, n_copies, stream);
    case 128: return launch_for_d<MT, 128>(a, fed, n_copies, stream);
    case 256: return launch_for_d<MT, 256>(a, fed, n_copies, stream);
  }
  return fail(LMH_E_UNSUPPORTED, "MFMA decode: head dim %d not tiled", a.D);
}

}  // namespace

// The query rotation of lmh_decode_step happens in registers: the partner of every element must be in the same lane.
bool decode_mfma_rope_ok(int D, int interleaved) { return interleaved || (D / 32) % 2 == 0; }

// Whether no two rows of a cache with these strides (batch, KV head, row) have an element in common.
static bool rows_apart(const int64_t (&stride)[3], const DecodeArgs &a) {
  std::pair<int64_t, int64_t> dims[3] = {{stride[0], a.B}, {stride[1], a.Hkv}, {stride[2], a.Lmax}};
  std::sort(dims, dims + 3);
  int64_t span = a.D;  // of what lies inside of a step along the next dimension
  for (const auto &[step, n] : dims) {
    if (n == 1) continue;
    if (step < span) return false;
    span += (n - 1) * step;
  }
  return true;
}

// Whether a pair's whole walk in one workgroup (decode_pair_kernel, with one split) is taken. A launch of it lasts as long as its longest
// pair, and the host knows the caches' length, not the sequences': of lengths that differ, one long sequence may stand beside many short
// ones, whose keys the split kernel deals to all CUs. So wherever lengths are given (steps always) the line lies where one sequence
// as long as the cache beside others of one key takes no longer than it did in the two launches before this kernel, and where the others gain.
// Measured on 2150 calls one behind the other, host and launches together (G = 1 to 4, D = 64 to 256, 2 to 2048 pairs), time against the split
// kernel (and the merge) of today with all lengths full / uniform in the upper three quarters / one full beside single keys, and the last
// also against the two launches before this kernel:
//   steps, few pairs: D=64 80 thousand elements a walk 0.76 to 0.90 / 0.73 to 0.88 / 0.87 to 0.91, 110 0.88 to 1.07 / 0.72 to 0.96 / 0.97 to 1.08;
//     D=128 110 0.70 to 0.96 / 0.54 to 0.82 / 0.81 to 0.94, 130 up to 1.11; D=256 130 0.78 to 0.91 / 0.60 to 0.86 / 0.78 to 0.91, 150 up to 1.05
//   steps on three eighths of the CUs and more: D=64 85 0.73 to 0.80 / 0.72 to 0.82 / 1.03 to 1.09 (0.85 to 0.90), 110 (0.99 to 1.08); D=128
//     140 0.76 to 0.87 / 0.65 to 0.87 / 1.00 to 1.29 (0.80 to 1.03), 180 from seven eighths on 0.84 to 0.87 / 0.78 to 0.81 / 1.23 to 1.30 (0.95 to 0.99), on fewer (0.92
//     to 1.21); D=256 180 0.73 to 0.92 / 0.68 to 0.85 / 0.87 to 1.18 (0.72 to 0.96), 250 from seven eighths on (0.93), on fewer (1.14 to 1.17)
//   steps of several rounds: D=128 170 0.86 to 1.01 / 0.78 to 1.02 / 0.93 to 1.39 (0.80 to 1.05), 300 (up to 1.32); D=256 300 nearly full rounds 0.91 to
//     0.93 / 0.74 to 0.92 / 0.77 to 1.32 (0.73 to 1.10); two rounds D=64 and 96 50 0.78 to 0.98 / 0.85 to 0.97 / 1.08 to 1.28 (0.87 to 1.01), 100 (up to 1.14); three
//     rounds D=64 8 0.86 / 0.82 / 0.91, 16 1.07 / 1.09 / 1.28, D=96 16 0.95 / 0.96 / 1.16 (0.94), 50 (1.29); four D=64 8 1.20, D=96 8 0.93, 16 1.23: a workgroup has the
//     CU, its prologue and fold nothing beside them
//   decodes, few pairs: D=64 80 0.83 to 0.94 / 0.77 to 0.90 / 0.88 to 0.94, 95 0.94 to 1.07; D=96 95 0.86 to 1.03; D=128 110 0.75 to 1.02 / 0.70 to 0.91 / 0.91 to 1.07, 130 0.95 to
//     1.19; D=256 95 0.79 to 0.86 / 0.59 to 0.82 / 0.80 to 0.85, 110 0.87 to 1.09. On three eighths of the CUs and more D=64 85 0.88 / 0.88 / 1.12 (0.92), 110
//     (1.20); D=128 110 0.78 to 0.99 / 0.88 to 0.99 / 1.00 to 1.17 (0.82 to 0.95), 140 (up to 1.17); D=256 140 0.77 to 0.94 / 0.76 to 0.96 / 0.98 to 1.29 (0.77 to 0.95), 180 (up to
//     1.10). From half the CUs on the split kernel takes walks up to 131 thousand in one split too: D=64 and 96 0.96 to 1.08, D=128 and 256 0.91 to 1.01
//   decodes without lengths (all as long as the cache), 112 to 256 pairs: 0.73 to 0.97 of two launches up to 160 thousand, from three quarters
//     of the CUs on 0.82 to 0.96 up to 440. With lengths 300 thousand on 256 pairs took 1.32, D=64 on 224 1.93 (one beside sixteenths).
//
// A step whose sequences share rows of a cache (windows of one buffer) stays on two launches: there every row is read before one is written.
bool decode_by_pairs(const DecodeArgs &a) {
  if (a.D % 32 != 0) return false;  // not built
  if (a.step && !(rows_apart(a.ks, a) && rows_apart(a.vs, a))) return false;
  const int64_t cus = device_cu_count(), pairs = (int64_t)a.B * a.Hkv * ((a.Hq / a.Hkv + 15) / 16), walk = (int64_t)a.Lmax * a.D;
  const int d = a.D > 128 ? 3 : a.D > 96 ? 2 : a.D > 64 ? 1 : 0;
  const bool many = pairs * 8 >= cus * 3;
  if (a.step) {
    constexpr int32_t kFew[4] = {100000, 100000, 120000, 140000}, kMany[4] = {100000, 100000, 140000, 200000}, kAll[4] = {100000, 100000, 180000, 280000};
    if (pairs <= cus) return walk <= (pairs * 8 >= cus * 7 ? kAll : many ? kMany : kFew)[d];
    const int64_t rounds = (pairs + cus - 1) / cus;
    if (d >= 2) return walk <= (d == 3 && pairs * 20 >= rounds * cus * 17 ? 300000 : 170000);
    return walk <= (rounds == 2 ? 50000 : rounds == 3 ? (d ? 16384 : 8192) : rounds == 4 && d ? 8192 : 0);
  }
  constexpr int32_t kFew[4] = {90000, 92000, 110000, 105000}, kMany[4] = {90000, 92000, 110000, 150000};
  if (d < 2 && pairs * 2 >= cus && walk <= 131072) return false;
  if (pairs > cus || (d == 0 && pairs * 20 > cus * 19)) return false;
  if (!a.kv_len && pairs * 16 >= cus * 7) return walk <= (pairs * 4 >= cus * 3 ? 450000 : 160000);
  return walk <= (many ? kMany : kFew)[d];
}

bool decode_mfma_supported(int dtype, int D, int B) {
  return (dtype == LMH_F16 || dtype == LMH_BF16) && (D == 64 || D == 96 || D == 128 || D == 256) &&
         B <= kMaxBatchPersistent;
}

// Whether a call's rows go to the split kernel here: the head dims above, and 80 where it is ahead of the vector ALUs. Those are busy with
// the products from three query heads a KV head on: us there and here, bf16, every sequence Lmax long, B=33 64/8 heads L=682 49.3 and 15.4, B=31 64/8 L=12366 409
// and 162 (981 MB; with lengths from a quarter of it up 293 and 113), B=34 8/1 L=5052 44.7 and 16.3, B=57 16/4 L=1315 34.0 and 18.3, B=7 4/1 L=3337 12.7 and 10.7;
// walks of up to 160 keys of up to four heads stay (B=13 32/8 L=152 8.7 and 10.2). Of two heads it takes the longer walks (B=1 40/20 L=12138 26.3 and 17.2, B=11
// 12/6 L=1269 12.2 and 11.1; B=7 12/6 L=484 9.0 and 9.2) and what goes round (B=113 12/6 L=498 26.1 and 19.9; not more than four times: B=120 64/32 L=231 48.7
// and 47.6, with lengths 36.4 and 41.5). Of one it takes what goes round, for the lengths' sake (fp16 B=50 Hkv=12 L=844 30.7 and 29.4, with lengths 28.2 and 21.6,
// B=37 Hkv=16 L=1487 50.0 and 49.4, 41.6 and 39.2); a round or less comes out even, and behind with lengths (bf16 B=2 Hkv=20 L=2714 12.4 and 12.0, 9.4 and 11.2).
bool decode_mfma_takes(const DecodeArgs &a, int dtype) {
  if (!a.mfma_ok) return false;
  if (decode_mfma_supported(dtype, a.D, a.B)) return true;
  if (dtype == LMH_F32 || a.D != 80 || a.B > kMaxBatchPersistent || a.step) return false;
  const int64_t cus = device_cu_count(), pairs = (int64_t)a.B * a.Hkv, group = a.Hq / a.Hkv;
  if (group > 2) return group > 4 || a.Lmax > 160;
  if (group == 2 && a.Lmax >= 560) return true;
  return pairs > cus && pairs <= 4 * cus && a.Lmax >= (group == 2 ? 224 : 384);
}

// Enqueues only the split kernel; the caller adds the merge kernel when num_splits > 1. With one split, everything (the copies
// only of a step).
int launch_decode_mfma_split(const DecodeArgs &a, int dtype, hipStream_t stream, const CopyManyArgs *fed, int n_copies) {
  if (dtype == LMH_F16) return launch_for_type<Mfma16F16>(a, fed, n_copies, stream);
  if (dtype == LMH_BF16) return launch_for_type<Mfma16BF16>(a, fed, n_copies, stream);
  return fail(LMH_E_UNSUPPORTED, "MFMA decode: dtype %d has no matrix-core path", dtype);
}

}  // namespace lmh
