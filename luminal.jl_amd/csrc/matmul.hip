// The matrix products of a model graph's projections in fp32 on the gfx950 matrix cores (v_mfma_f32_32x32x2_f32):
// c = a b (+ bias), batched, up to kMatmulGroup products in one launch. Semantics: batch_matmul of the reference
// (src/Execution.jl:12-90) and its Linear layer (src/NN.jl:11-38); operands of any element type are taken to fp32 as they
// are loaded, sums are fp32, the result is rounded once to c's type.
//
// Bound: the fp32 matrix pipe (157 TFLOP/s, 64 flops per cycle and SIMD). A wave owns a 32 x 32 block of c: one 128-bit
// LDS read of each operand feeds four MFMAs of 64 cycles, so LDS (two reads, 16 of 256 cycles) and the vector ALUs are idle
// most of the time and what decides is how evenly the blocks fall on the 1024 SIMDs:
//   * a workgroup is WM x WN blocks, and WK waves share a block by taking every WK-th 32 elements of the contraction
//     (folded through LDS at the end): the launcher takes the form whose last round is fullest (launch_matmul below);
//   * several products that run at the same time in a model (the q, k and v projections of a layer, which share a) go into
//     one launch, so their rounds are filled together;
//   * blockIdx -> tile hands every XCD a contiguous range of tiles, rows of c fastest: its L2 holds a slice of b's columns.
// Tiles of 32 contraction elements go to double-buffered LDS rows of eight 16-byte chunks; chunk j of row r lies at
// j ^ (r & 7), which spreads the eight rows that a fragment read's quarter-wave touches over all banks without padding.
// fp32 operands that are contiguous along the contraction (VEC) are fetched with buffer loads that write straight into LDS,
// each lane asking for the chunk whose swizzled place it fills; everything else passes through registers, where any element
// type and layout becomes fp32.
// The contraction runs in the order 8 j + e, 8 j + 4 + e (e = 0..3): the MFMA takes its two elements from the two halves
// of the wave, which read neighbouring chunks.
#include <limits.h>

#include <algorithm>

#include "common.hpp"
#include "copy.hpp"
#include "dtypes.hpp"
#include "split.hpp"

namespace lmh {
namespace {

constexpr int BK = 32;  // contraction elements a wave takes per staged tile
// Byte offset no operand reaches (the host routes larger ones to the other form): a buffer load there returns zeros.
constexpr int kOutOfRange = 0x7ffffff0;

__device__ inline float load_as_f32(const void *p, int64_t i, int dtype) {
  switch (dtype) {
    case LMH_F16: return (float)reinterpret_cast<const _Float16 *>(p)[i];
    case LMH_BF16: return bf16_bits_to_f32(reinterpret_cast<const uint16_t *>(p)[i]);
    case LMH_I32: return (float)reinterpret_cast<const int32_t *>(p)[i];
    default: return reinterpret_cast<const float *>(p)[i];
  }
}
// Column j of c is column `b_column` of b: the same, or, where c is split into heads, column h + heads * d for j = h D + d
// (the reference's column-major reshape of hidden into (heads, D) makes the head index the fast one).
__device__ inline int b_column(const MatmulProblem &p, int D, int j) { return p.heads ? j / D + p.heads * (j % D) : j; }

// Store a wave's 32 x 32 block: lane (n, h) holds column j, register i row mw + 8 (i / 4) + 4 h + i % 4.
__device__ inline void store_block(const MatmulProblem &p, const floatx16_t &acc, int mw, int j, int h, int batch) {
  if (j >= p.N || mw >= p.M) return;
  const int D = p.heads ? p.N / p.heads : 1;
  const float bias = p.bias ? load_as_f32(p.bias, b_column(p, D, j), p.bias_dtype) : 0.f;
  // Offsets by addition: a division per row and lane made the epilogue a tenth of the launch at K = 2048.
  int64_t base, wrap = 0;          // offset of row mw; what a step to the next sequence adds beyond a row step
  int row_step, s0 = 0, seq = INT_MAX;
  if (p.heads) {  // c[b, head, s, d], rows m = b S + s
    const int head = j / D, b = mw / p.seq;
    seq = p.seq;
    s0 = mw - b * seq;
    row_step = D;
    base = (((int64_t)b * p.heads + head) * seq + s0) * D + (j - head * D);
    wrap = (int64_t)(p.heads - 1) * seq * D;
  } else {
    row_step = p.N;
    base = ((int64_t)batch * p.M + mw) * p.N + j;
  }
  auto store_rows = [&](auto store) {
#pragma unroll
    for (int i = 0; i < 16; i++) {
      const int r = 8 * (i >> 2) + 4 * h + (i & 3);
      if (mw + r >= p.M) break;  // rows ascend with i
      int64_t off = base + (int64_t)r * row_step;
      for (int s = s0 + r; s >= seq; s -= seq) off += wrap;
      store(off, acc[i] + bias);
    }
  };
  if (p.c_dtype == LMH_F32) store_rows([&](int64_t off, float x) { reinterpret_cast<float *>(p.c)[off] = x; });
  else if (p.c_dtype == LMH_F16) store_rows([&](int64_t off, float x) { reinterpret_cast<_Float16 *>(p.c)[off] = (_Float16)x; });
  else store_rows([&](int64_t off, float x) { reinterpret_cast<uint16_t *>(p.c)[off] = f32_to_bf16_bits(x); });
}

// VEC: every operand is fp32, contiguous along the contraction and 16-byte aligned, K a multiple of 4.
template <int WM, int WN, int WK, bool VEC>
__global__ __launch_bounds__(64 * WM * WN * WK, 2) void matmul_f32_kernel(MatmulArgs args, CopyManyArgs fed, int n_copies) {
  constexpr int NT = 64 * WM * WN * WK;
  constexpr int BM = 32 * WM, BN = 32 * WN, BKT = BK * WK;
  constexpr int CA = BM * BKT / 4, CB = BN * BKT / 4;  // 16-byte chunks of a tile
  constexpr int RA = CA / NT, RB = CB / NT;
  static_assert(CA % NT == 0 && CB % NT == 0, "whole chunks per thread");
  __shared__ __attribute__((aligned(16))) float As[2][BM * BKT];
  __shared__ __attribute__((aligned(16))) float Bs[2][BN * BKT];

  // ---- which tile of which product ----
  const int per_xcd = (args.n_tiles + 7) / 8;
  int t = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per_xcd) {  // copies beside the products
    if ((int)blockIdx.x - 8 * per_xcd < n_copies) copy_block<64 * WM * WN * WK>(fed, blockIdx.x - 8 * per_xcd);
    return;
  }
  if (t >= args.n_tiles) return;
  int g = 0;
#pragma unroll
  for (int i = 1; i < kMatmulGroup; i++)
    if (t >= args.first_tile[i]) g = i;
  const MatmulProblem p = args.p[g];
  t -= args.first_tile[g];
  const int m_tiles = (p.M + BM - 1) / BM;
  const int tm = t % m_tiles;
  t /= m_tiles;
  const int n_tiles = (p.N + BN - 1) / BN;
  const int tn = t % n_tiles, batch = t / n_tiles;
  const int m0 = tm * BM, n0 = tn * BN;

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int n = lane & 31, h = lane >> 5;
  const int wk = wave / (WM * WN), wm = (wave % (WM * WN)) / WN, wn = wave % WN;

  const int D = p.heads ? p.N / p.heads : 1;
  auto b_col = [&](int j) { return b_column(p, D, j); };

  floatx16_t acc;
#pragma unroll
  for (int i = 0; i < 16; i++) acc[i] = 0.f;
  const int n_k = (p.K + BKT - 1) / BKT;
  // Fragments of the wave's block from a staged tile, and their 16 MFMAs. All eight reads are issued first.
  auto multiply = [&](int buf) {
    const int arow = 32 * wm + n, brow = 32 * wn + n;
    const float *Aw = &As[buf][32 * BM * wk], *Bw = &Bs[buf][32 * BN * wk];
    floatx4_t af[4], bf[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
      af[j] = *reinterpret_cast<const floatx4_t *>(&Aw[4 * (arow * 8 + ((2 * j + h) ^ (arow & 7)))]);
      bf[j] = *reinterpret_cast<const floatx4_t *>(&Bw[4 * (brow * 8 + ((2 * j + h) ^ (brow & 7)))]);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < 4; j++)
#pragma unroll
      for (int e = 0; e < 4; e++) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(af[j][e], bf[j][e], acc, 0, 0, 0);
  };

  if constexpr (VEC) {
    // A tile of `rows` rows is WK slices of rows / 8 blocks of 1 KB; wave w issues blocks w, w + NW, ... of a, then of b.
    typedef int32_t i32x4_t __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) void lds_void_t;
    constexpr int NW = WM * WN * WK;
    constexpr int KA = BM * WK / 8 / NW, KB = BN * WK / 8 / NW;  // blocks per wave
    const int wave_u = __builtin_amdgcn_readfirstlane(wave);
    auto make_desc = [](const float *base, int64_t elements) {
      const uint64_t q = (uint64_t)base;
      i32x4_t d;
      d[0] = __builtin_amdgcn_readfirstlane((int)(uint32_t)q);
      d[1] = __builtin_amdgcn_readfirstlane((int)((q >> 32) & 0xffff));  // stride 0: raw buffer
      d[2] = __builtin_amdgcn_readfirstlane((int)(elements * 4));
      d[3] = 0x00020000;
      return d;
    };
    const i32x4_t a_desc = make_desc(reinterpret_cast<const float *>(p.a) + batch * p.as[0] + m0 * p.as[1], (min(p.M - m0, BM) - 1) * p.as[1] + p.K);
    const i32x4_t b_desc = make_desc(reinterpret_cast<const float *>(p.b) + batch * p.bs[0], (int64_t)(p.N - 1) * p.bs[2] + p.K);
    int a_voff[KA], b_voff[KB], a_k[KA], b_k[KB];  // byte offset of the lane's chunk in k-tile 0; its first k
#pragma unroll
    for (int j = 0; j < KA; j++) {
      const int q = wave + NW * j, row = (q % (BM / 8)) * 8 + (lane >> 3);
      a_k[j] = (q / (BM / 8)) * BK + 4 * ((lane & 7) ^ (row & 7));
      a_voff[j] = m0 + row < p.M ? (int)((row * p.as[1] + a_k[j]) * 4) : kOutOfRange;
    }
#pragma unroll
    for (int j = 0; j < KB; j++) {
      const int q = wave + NW * j, row = (q % (BN / 8)) * 8 + (lane >> 3);
      b_k[j] = (q / (BN / 8)) * BK + 4 * ((lane & 7) ^ (row & 7));
      b_voff[j] = n0 + row < p.N ? (int)((b_col(n0 + row) * p.bs[2] + b_k[j]) * 4) : kOutOfRange;
    }
    const uint32_t a_lds = (uint32_t)(uintptr_t)(lds_void_t *)&As[0][0] + wave_u * 1024;
    const uint32_t b_lds = (uint32_t)(uintptr_t)(lds_void_t *)&Bs[0][0] + wave_u * 1024;
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"  // m0 is a reserved register; it is only written here
    // (in asm for the reason prefill_mfma.hip gives: the compiler would wait for the load before the next LDS read)
    auto load_block = [](i32x4_t desc, uint32_t lds_addr, int voff, int soff) {
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                   :: "s"(lds_addr), "v"(voff), "s"(desc), "s"(soff) : "memory", "m0");
    };
#pragma clang diagnostic pop
    auto load_tile = [&](int kt) {
      const int buf = kt & 1, k0 = kt * BKT;
      const bool tail = k0 + BKT > p.K;  // chunks past the contraction's end are fetched out of range: zeros
#pragma unroll
      for (int j = 0; j < KA; j++)
        load_block(a_desc, a_lds + buf * (BM * BKT * 4) + j * (NW * 1024), tail && k0 + a_k[j] >= p.K ? kOutOfRange : a_voff[j], k0 * 4);
#pragma unroll
      for (int j = 0; j < KB; j++)
        load_block(b_desc, b_lds + buf * (BN * BKT * 4) + j * (NW * 1024), tail && k0 + b_k[j] >= p.K ? kOutOfRange : b_voff[j], k0 * 4);
    };
    load_tile(0);
    for (int kt = 0; kt < n_k; kt++) {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's blocks of tile kt are in LDS
      __syncthreads();  // ... and everyone's; tile kt - 1 has been consumed, its buffer is free
      if (kt + 1 < n_k) load_tile(kt + 1);  // in flight while tile kt is multiplied
      multiply(kt & 1);
    }
  } else {
    // chunk ch of a tile = row ch / (8 WK), 16-byte chunk ch % (8 WK) of it; where b is contiguous along its columns,
    // neighbouring threads take neighbouring columns instead
    const bool b_by_column = p.b_by_column;
    int64_t a_off[RA], b_off[RB];  // negative: a row past the operand's end
#pragma unroll
    for (int r = 0; r < RA; r++) {
      const int m = m0 + (tid + r * NT) / (8 * WK);
      a_off[r] = m < p.M ? batch * p.as[0] + m * p.as[1] : -1;
    }
#pragma unroll
    for (int r = 0; r < RB; r++) {
      const int j = n0 + (b_by_column ? (tid + r * NT) % BN : (tid + r * NT) / (8 * WK));
      b_off[r] = j < p.N ? batch * p.bs[0] + b_col(j) * p.bs[2] : -1;
    }
    floatx4_t a_reg[RA], b_reg[RB];
    auto fetch = [&](const void *base, int dtype, int64_t off, int64_t ks, int k) {
      floatx4_t x = {0.f, 0.f, 0.f, 0.f};
      if (off < 0) return x;
#pragma unroll
      for (int e = 0; e < 4; e++)
        if (k + e < p.K) x[e] = load_as_f32(base, off + (k + e) * ks, dtype);
      return x;
    };
    auto load_tile = [&](int k0) {
#pragma unroll
      for (int r = 0; r < RA; r++) a_reg[r] = fetch(p.a, p.a_dtype, a_off[r], p.as[2], k0 + 4 * ((tid + r * NT) % (8 * WK)));
#pragma unroll
      for (int r = 0; r < RB; r++) {
        const int c = b_by_column ? (tid + r * NT) / BN : (tid + r * NT) % (8 * WK);
        b_reg[r] = fetch(p.b, p.b_dtype, b_off[r], p.bs[1], k0 + 4 * c);
      }
    };
    auto lds_chunk = [](int rows, int row, int c) { return ((c >> 3) * rows + row) * 8 + ((c & 7) ^ (row & 7)); };
    auto store_tile = [&](int buf) {
#pragma unroll
      for (int r = 0; r < RA; r++) {
        const int ch = tid + r * NT;
        *reinterpret_cast<floatx4_t *>(&As[buf][4 * lds_chunk(BM, ch / (8 * WK), ch % (8 * WK))]) = a_reg[r];
      }
#pragma unroll
      for (int r = 0; r < RB; r++) {
        const int ch = tid + r * NT;
        const int row = b_by_column ? ch % BN : ch / (8 * WK), c = b_by_column ? ch / BN : ch % (8 * WK);
        *reinterpret_cast<floatx4_t *>(&Bs[buf][4 * lds_chunk(BN, row, c)]) = b_reg[r];
      }
    };
    load_tile(0);
    store_tile(0);
    for (int kt = 0; kt < n_k; kt++) {
      __syncthreads();  // tile kt is in LDS; everyone is done with tile kt - 1, whose buffer is written below
      if (kt + 1 < n_k) load_tile((kt + 1) * BKT);
      multiply(kt & 1);
      if (kt + 1 < n_k) store_tile((kt + 1) & 1);
    }
  }

  // ---- fold the WK shares of a block, first share first ----
  if constexpr (WK > 1) {
    static_assert((WK - 1) * WM * WN * 16 * 64 <= 2 * BM * BKT, "the folded shares fit the tiles of a");
    float *xch = &As[0][0];
    __syncthreads();
    if (wk > 0) {
      float *w = xch + ((wk - 1) * (WM * WN) + wave % (WM * WN)) * (16 * 64) + lane;
#pragma unroll
      for (int i = 0; i < 16; i++) w[i * 64] = acc[i];
    }
    __syncthreads();
    if (wk > 0) return;
#pragma unroll
    for (int o = 0; o < WK - 1; o++) {
      const float *r = xch + (o * (WM * WN) + wave) * (16 * 64) + lane;
#pragma unroll
      for (int i = 0; i < 16; i++) acc[i] += r[i * 64];
    }
  }

  store_block(p, acc, m0 + 32 * wm, n0 + 32 * wn + n, h, batch);
}

// The same products for fp32 operands that are contiguous along the contraction, on the bf16 matrix pipe (16 times the rate).
// Every operand is split into three bf16 pieces (split.hpp); of the nine products of pieces the six with x_i y_j, i + j <= 4, are
// summed, the other three are below 2^-25 of x y. Error against 64 bits (2-norm): 3.6e-7 where the fp32 product has 5.7e-7 (K =
// 2048; fewer roundings), 9.2e-8 and 1.07e-7 (K = 64). A workgroup with a sum that is not finite (an operand that the pieces do not
// hold, or a sum beyond 2^80 before the scale comes off) takes its block again with the fp32 product; a launch all of whose blocks are
// repeated takes twice as long (700 x 2048 x 2048: 44 and 103 us).
//
// Bound: the vector ALUs beside the matrix pipe. Splitting takes 6.5 instructions an element, 6.5 a MFMA at 64 x 128 and 8.7 at
// 64 x 64, where the chip holds 1590 TFLOP/s of bare MFMAs and 1280 with six vector instructions each. So:
//   * a wave multiplies blocks as large as its registers hold (MB x NB of 32 x 32, up to nine or eight), and the four
//     waves of a workgroup each take all of its tile for every fourth 16 elements of the contraction; the shares are folded
//     through LDS at the end;
//   * a wave fetches its own operands and shares nothing until then, so there is no barrier in the loop: buffer loads write fp32
//     rows of 64 bytes straight into the wave's two stages in LDS, the wave reads them in the MFMA's layout (chunk j of row r
//     lies at j ^ f(r): all banks) and splits them in registers one step ahead of the MFMAs, five to ten instructions between
//     every two of those. (Planes of pieces in LDS, split once per workgroup with a barrier per 64 elements, take 50 us in place
//     of 46.5 on 700 x 2560 x 2048: the waves of a SIMD then do the same thing at the same time.)
__device__ inline int swizzle16(int row) { return ((row >> 1 ^ row >> 3) & 1) | (row >> 1 & 2); }

template <int MB, int NB>
__global__ __launch_bounds__(256, 1) void matmul_split_kernel(MatmulArgs args, CopyManyArgs fed, int n_copies) {
  constexpr int BM = 32 * MB, BN = 32 * NB, WK = 4;
  constexpr int L = 2 * (MB + NB);              // loads of 1 KB (16 rows) per stage: a, then b
  constexpr int kStage = 16 * 16 * L;           // floats
  constexpr int LDC = BN + 8;                   // row of a wave's sums: the rows r and r + 4 of a store fall on different banks
  constexpr int kShare = BM * LDC;              // floats of a wave's sums
  __shared__ __attribute__((aligned(16))) float bias_s[BN];
  __shared__ __attribute__((aligned(16))) float lds[WK * (2 * kStage > kShare ? 2 * kStage : kShare)];

  const int per_xcd = (args.n_tiles + 7) / 8;
  int t = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per_xcd) {
    if ((int)blockIdx.x - 8 * per_xcd < n_copies) copy_block<256>(fed, blockIdx.x - 8 * per_xcd);
    return;
  }
  if (t >= args.n_tiles) return;
  int g = 0;
#pragma unroll
  for (int i = 1; i < kMatmulGroup; i++)
    if (t >= args.first_tile[i]) g = i;
  const MatmulProblem p = args.p[g];
  t -= args.first_tile[g];
  const int m_tiles = (p.M + BM - 1) / BM, n_tiles = (p.N + BN - 1) / BN;
  const int tm_row = (uint32_t)t / p.by_m_tiles, tm = t - tm_row * m_tiles;
  const int batch = (uint32_t)tm_row / p.by_n_tiles, tn = tm_row - batch * n_tiles;
  const int m0 = tm * BM, n0 = tn * BN;
  const int wk = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

  const int lane = threadIdx.x & 63;
  const int n = lane & 31, h = lane >> 5;
  const int D = p.heads ? p.N / p.heads : 1;
  auto b_col = [&](int j) {  // b_column
    const int head = (uint32_t)j / p.by_D;
    return p.heads ? head + p.heads * (j - head * D) : j;
  };
  // the bias of column n0 + thread, fetched ahead of everything
  const float bias = p.bias && (int)threadIdx.x < BN && n0 + (int)threadIdx.x < p.N ? load_as_f32(p.bias, b_col(n0 + threadIdx.x), p.bias_dtype) : 0.f;
  const int steps = ((p.K + 15) / 16 - wk + WK - 1) / WK;  // of this wave (may be none)

  typedef int32_t i32x4_t __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) void lds_void_t;
  auto make_desc = [](const float *base, int64_t elements) {
    const uint64_t q = (uint64_t)base;
    i32x4_t d;
    d[0] = __builtin_amdgcn_readfirstlane((int)(uint32_t)q);
    d[1] = __builtin_amdgcn_readfirstlane((int)((q >> 32) & 0xffff));  // stride 0: raw buffer
    d[2] = __builtin_amdgcn_readfirstlane((int)(elements * 4));
    d[3] = 0x00020000;
    return d;
  };
  const float *a_base = reinterpret_cast<const float *>(p.a) + batch * p.as[0] + m0 * p.as[1];
  const float *b_base = reinterpret_cast<const float *>(p.b) + batch * p.bs[0];
  const i32x4_t a_desc = make_desc(a_base, (min(p.M - m0, BM) - 1) * p.as[1] + p.K);
  const i32x4_t b_desc = make_desc(b_base, (int64_t)(p.N - 1) * p.bs[2] + p.K);
  int voff[L], k_of[2];  // byte offset of the lane's chunk of each load at k = 0; its first k, by the parity of the load
#pragma unroll
  for (int l = 0; l < L; l++) {
    const int row = 16 * l + (lane >> 2), chunk = (lane & 3) ^ swizzle16(row), col = n0 + row - BM;
    if (l < 2) k_of[l] = 4 * chunk;
    if (l < 2 * MB) voff[l] = m0 + row < p.M ? (int)((row * p.as[1] + 4 * chunk) * 4) : kOutOfRange;
    else voff[l] = col < p.N ? (int)((b_col(col) * p.bs[2] + 4 * chunk) * 4) : kOutOfRange;
  }
  const uint32_t ring = (uint32_t)(uintptr_t)(lds_void_t *)&lds[wk * 2 * kStage];
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"  // m0 is a reserved register; it is only written here
  auto load_block = [](i32x4_t desc, uint32_t lds_addr, int off, int soff) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 :: "s"(lds_addr), "v"(off), "s"(desc), "s"(soff) : "memory", "m0");
  };
#pragma clang diagnostic pop
  // Past the wave's last step every lane is out of range and zeros arrive; the scalar offset stays inside the operand (one beyond
  // its end would defeat the range check).
  auto load_stage = [&](int i) {
    const int k0 = 16 * (wk + WK * i), soff = min(k0, p.K - 4) * 4;
    const bool tail = k0 + 16 > p.K;
#pragma unroll
    for (int l = 0; l < L; l++)
      load_block(l < 2 * MB ? a_desc : b_desc, ring + (i & 1) * (kStage * 4) + l * 1024, tail && k0 + k_of[l & 1] >= p.K ? kOutOfRange : voff[l], soff);
  };

  // 32 rows of a stage in the MFMA's layout: lane (n, h) takes elements 8 h .. 8 h + 7 of row n. Blocks: MB of a, then NB of b.
  const int frag0 = n * 16 + 4 * ((2 * h) ^ swizzle16(n)), frag1 = n * 16 + 4 * ((2 * h + 1) ^ swizzle16(n));
  const float *own = &lds[wk * 2 * kStage];
  struct Raw { floatx4_t lo, hi; };
  auto split = [](const Raw &r) { return split_8(r.lo * kPieceScale, r.hi * kPieceScale); };
  auto read_stage = [&](int i, Raw (&raw)[MB + NB]) {
#pragma unroll
    for (int b = 0; b < MB + NB; b++) {
      const float *q = own + (i & 1) * kStage + b * 512;
      raw[b].lo = *reinterpret_cast<const floatx4_t *>(q + frag0);
      raw[b].hi = *reinterpret_cast<const floatx4_t *>(q + frag1);
    }
  };

  floatx16_t acc[MB][NB];
  auto clear = [&]() {
#pragma unroll
    for (int i = 0; i < MB; i++)
#pragma unroll
      for (int j = 0; j < NB; j++)
#pragma unroll
        for (int e = 0; e < 16; e++) acc[i][j][e] = 0.f;
  };
  clear();

  // Step i multiplies stage i while stage i + 1 is split and stages i + 2 and i + 3 are on their way.
  Pieces even[MB + NB], odd[MB + NB];
  Raw raw[MB + NB];
  load_stage(0);
  load_stage(1);
  asm volatile("s_waitcnt vmcnt(%0)" :: "n"(L) : "memory");
  read_stage(0, raw);
#pragma unroll
  for (int b = 0; b < MB + NB; b++) even[b] = split(raw[b]);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  load_stage(2);
  constexpr int kA[6] = {0, 0, 1, 1, 0, 2}, kB[6] = {0, 1, 0, 1, 2, 0};
  auto step = [&](int i, const Pieces (&cur)[MB + NB], Pieces (&nxt)[MB + NB]) {
    asm volatile("s_waitcnt vmcnt(%0)" :: "n"(L) : "memory");  // stage i + 1 has landed
    read_stage(i + 1, raw);
#pragma unroll
    for (int r = 0; r < MB; r++)
#pragma unroll
      for (int j = 0; j < NB; j++) acc[r][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(cur[r].p[0], cur[MB + j].p[0], acc[r][j], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // every read of that stage has returned
    load_stage(i + 3);
#pragma unroll
    for (int b = 0; b < MB + NB; b++) nxt[b] = split(raw[b]);  // (past the last step: zeros)
#pragma unroll
    for (int q = 1; q < 6; q++)
#pragma unroll
      for (int r = 0; r < MB; r++)
#pragma unroll
        for (int j = 0; j < NB; j++) acc[r][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(cur[r].p[kA[q]], cur[MB + j].p[kB[q]], acc[r][j], 0, 0, 0);
    constexpr int kValu = (52 * (MB + NB) + 5 * MB * NB) / (5 * MB * NB);
#pragma unroll
    for (int q = 0; q < 5 * MB * NB; q++) {
      __builtin_amdgcn_sched_group_barrier(0x002, kValu, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    }
  };
  int i = 0;
  for (; i + 1 < steps; i += 2) {  // (two steps a turn: no copies of the fragments)
    step(i, even, odd);
    step(i + 1, odd, even);
  }
  if (i < steps) step(i, even, odd);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // nothing arrives in the ring any more

  // ---- fold the shares, four columns of a row a thread, and look whether the sums are finite ----
  // Through LDS in rows, so that a wave stores whole rows of c: as a lane holds them, a column each, they are stores of 64 to 128
  // bytes a row, 2.2 to 4.4 us of a launch. us a layer, before and now: 700 rows, hidden 2048, 32 heads of 64 111.1 and 108.7 (32 KV heads
  // 178.8 and 173.5), 2 x 1000 rows, 12 heads of 128 302 and 283, 4 x 400 rows, 16 heads of 96 167 and 160, with biases 144.8 and 137.8
  constexpr int Q = BM * BN / 1024;  // fours of a thread
  if ((int)threadIdx.x < BN) bias_s[threadIdx.x] = bias;
  floatx4_t sum[Q];
  bool redone = false;
  for (int pass = 0;; pass++) {
    redone = pass > 0;
    const float unscale = pass ? 1.f : kPieceUnscale * kPieceUnscale;
    if (pass) {
      // the workgroup's block again with the fp32 product, the operands straight from memory
      clear();
      const __amdgpu_buffer_rsrc_t a_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(a_base), 0, a_desc[2], 0x00020000);
      const __amdgpu_buffer_rsrc_t b_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(b_base), 0, b_desc[2], 0x00020000);
      int off[MB + NB];
#pragma unroll
      for (int i = 0; i < MB + NB; i++) {
        const int row = 32 * i + n, col = n0 + row - BM;
        if (i < MB) off[i] = m0 + row < p.M ? (int)(row * p.as[1] * 4) : -1;
        else off[i] = col < p.N ? (int)(b_col(col) * p.bs[2] * 4) : -1;
      }
      for (int i = 0; i < 2 * steps; i++) {
        const int k = 16 * (wk + WK * (i >> 1)) + 8 * (i & 1) + 4 * h;
        floatx4_t x[MB + NB];
#pragma unroll
        for (int r = 0; r < MB + NB; r++)
          x[r] = __builtin_bit_cast(floatx4_t, __builtin_amdgcn_raw_buffer_load_b128(r < MB ? a_rsrc : b_rsrc, k < p.K && off[r] >= 0 ? off[r] + 4 * k : kOutOfRange, 0, 0));
#pragma unroll
        for (int e = 0; e < 4; e++)
#pragma unroll
          for (int r = 0; r < MB; r++)
#pragma unroll
            for (int j = 0; j < NB; j++) acc[r][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(x[r][e], x[MB + j][e], acc[r][j], 0, 0, 0);
      }
    }
    __syncthreads();
    float *w = &lds[wk * kShare + 4 * h * LDC + n];
#pragma unroll
    for (int r = 0; r < MB; r++)
#pragma unroll
      for (int j = 0; j < NB; j++)
#pragma unroll
        for (int i = 0; i < 16; i++) w[(32 * r + 8 * (i >> 2) + (i & 3)) * LDC + 32 * j] = acc[r][j][i];
    __syncthreads();
    float finite = 0.f;
#pragma unroll
    for (int q = 0; q < Q; q++) {
      const int at = threadIdx.x + 256 * q;
      const float *s = &lds[at / (BN / 4) * LDC + at % (BN / 4) * 4];
      floatx4_t x = *reinterpret_cast<const floatx4_t *>(s);
#pragma unroll
      for (int o = 1; o < WK; o++) x += *reinterpret_cast<const floatx4_t *>(s + o * kShare);
#pragma unroll
      for (int e = 0; e < 4; e++) finite = fmaf(x[e], 0.f, finite);
      sum[q] = x * unscale;
    }
    if (pass || !__syncthreads_or(finite != 0.f || finite != finite)) break;
  }
  auto place = [&](int m, int j) -> int64_t {
    if (!p.heads) return ((int64_t)batch * p.M + m) * p.N + j;
    const int b = (uint32_t)m / p.by_seq, head = (uint32_t)j / p.by_D;  // c[b, head, s, d], rows m = b S + s
    return (((int64_t)b * p.heads + head) * p.seq + (m - b * p.seq)) * D + (j - head * D);
  };
  if (!p.c_vec) {  // columns that do not come in fours: element by element, from the shares in LDS
    const float unscale = redone ? 1.f : kPieceUnscale * kPieceUnscale;
#pragma unroll 1
    for (int at = threadIdx.x; at < BM * BN; at += 256) {
      const int m = m0 + at / BN, j = n0 + at % BN;
      if (m >= p.M || j >= p.N) continue;
      const float *s = &lds[at / BN * LDC + at % BN];
      float x = s[0];
#pragma unroll
      for (int o = 1; o < WK; o++) x += s[o * kShare];
      x = x * unscale + bias_s[at % BN];
      const int64_t off = place(m, j);
      if (p.c_dtype == LMH_F32) reinterpret_cast<float *>(p.c)[off] = x;
      else if (p.c_dtype == LMH_F16) reinterpret_cast<_Float16 *>(p.c)[off] = (_Float16)x;
      else reinterpret_cast<uint16_t *>(p.c)[off] = f32_to_bf16_bits(x);
    }
    return;
  }
#pragma unroll
  for (int q = 0; q < Q; q++) {
    const int at = threadIdx.x + 256 * q, m = m0 + at / (BN / 4), j = n0 + at % (BN / 4) * 4;
    if (m >= p.M || j >= p.N) continue;
    const floatx4_t x = sum[q] + *reinterpret_cast<const floatx4_t *>(&bias_s[j - n0]);
    const int64_t off = place(m, j);
    if (p.c_dtype == LMH_F32) {
      *reinterpret_cast<floatx4_t *>(reinterpret_cast<float *>(p.c) + off) = x;
      continue;
    }
    uint16_t y[4];
#pragma unroll
    for (int e = 0; e < 4; e++) y[e] = p.c_dtype == LMH_F16 ? __builtin_bit_cast(uint16_t, (_Float16)x[e]) : f32_to_bf16_bits(x[e]);
    *reinterpret_cast<uint2 *>(reinterpret_cast<uint16_t *>(p.c) + off) = make_uint2((uint32_t)y[0] | (uint32_t)y[1] << 16, (uint32_t)y[2] | (uint32_t)y[3] << 16);
  }
}

// The tiles of the products of a launch, numbered one product after the other; negative where there are too many.
int64_t number_tiles(MatmulArgs &args, int n, int bm, int bn) {
  int64_t tiles = 0;
  for (int i = 0; i < kMatmulGroup; i++) {
    args.first_tile[i] = (int)tiles;
    if (i < n) tiles += (int64_t)args.p[i].batch * ((args.p[i].M + bm - 1) / bm) * ((args.p[i].N + bn - 1) / bn);
    if (tiles >= (int64_t(1) << 31) - 65536) return -1;  // (with room for the copies)
  }
  args.n_tiles = (int)tiles;
  return tiles;
}

template <int WM, int WN, int WK>
int launch_form(MatmulArgs &args, int n, hipStream_t stream, const CopyManyArgs &fed, int n_copies) {
  const int64_t tiles = number_tiles(args, n, 32 * WM, 32 * WN);
  if (tiles < 0) return fail(LMH_E_UNSUPPORTED, "matmul: too many tiles");
  bool vec = true;
  for (int i = 0; i < n; i++) vec = vec && args.p[i].a_vec && args.p[i].b_vec;
  const dim3 grid((unsigned)((tiles + 7) / 8 * 8 + n_copies)), block(64 * WM * WN * WK);
  if (vec) hipLaunchKernelGGL((matmul_f32_kernel<WM, WN, WK, true>), grid, block, 0, stream, args, fed, n_copies);
  else hipLaunchKernelGGL((matmul_f32_kernel<WM, WN, WK, false>), grid, block, 0, stream, args, fed, n_copies);
  LMH_HIP_TRY(hipGetLastError());
  return LMH_OK;
}

template <int MB, int NB>
int launch_split_form(MatmulArgs &args, int n, hipStream_t stream, const CopyManyArgs &fed, int n_copies) {
  const int64_t tiles = number_tiles(args, n, 32 * MB, 32 * NB);
  if (tiles < 0) return fail(LMH_E_UNSUPPORTED, "matmul: too many tiles");
  for (int i = 0; i < n; i++) {
    MatmulProblem &p = args.p[i];
    const int D = p.heads ? p.N / p.heads : 1;
    p.by_m_tiles = fast_div((p.M + 32 * MB - 1) / (32 * MB));
    p.by_n_tiles = fast_div((p.N + 32 * NB - 1) / (32 * NB));
    p.by_D = fast_div(D);
    p.by_seq = fast_div(p.heads ? p.seq : 1);
    p.c_vec = p.N % 4 == 0 && (!p.heads || D % 4 == 0) && (reinterpret_cast<uintptr_t>(p.c) & 15u) == 0;
  }
  hipLaunchKernelGGL((matmul_split_kernel<MB, NB>), dim3((unsigned)((tiles + 7) / 8 * 8 + n_copies)), dim3(256), 0, stream, args, fed, n_copies);
  LMH_HIP_TRY(hipGetLastError());
  return LMH_OK;
}

}  // namespace

int launch_matmul(MatmulArgs &args, int n, hipStream_t stream, CopyManyArgs *fed, int n_fed) {
  const int n_copies = n_fed ? (int)number_copy_blocks(*fed, n_fed) : 0;
  const CopyManyArgs copies = n_copies ? *fed : CopyManyArgs{};
  // Both kernels by what their forms cost, in us: a part per launch, a part per round of the CUs, and one per round and
  // contraction element.
  // fp32 product: rounds times the 32 x 32 blocks of a workgroup, with a weight for what the smaller workgroups pay in loads and
  // fixed costs per block. Measured, us for (64 x 64, eight waves) / (32 x 64) / (32 x 32): 700 x 2560 x 2048 82 / 90 / 99,
  // 700 x 2048 x 2048 73 / 62 / 73, 606 x 1536 x 1536 33 / 35 / 39, 1446 x 768 x 384 18.5 / 16.1 / 19.5,
  // 690 x 384 x 384 10.9 / 8.5 / 8.5, 164 x 1280 x 1280 26 / 18 / 11.
  const int64_t cus = device_cu_count();
  auto rounds = [&](int bm, int bn) {
    int64_t tiles = 0;
    for (int i = 0; i < n; i++) tiles += (int64_t)args.p[i].batch * ((args.p[i].M + bm - 1) / bm) * ((args.p[i].N + bn - 1) / bn);
    return (tiles + cus - 1) / cus;
  };
  const int64_t r64 = rounds(64, 64);
  const double c64 = 4.0 * r64, c32x64 = 2.2 * rounds(32, 64), c32 = 1.5 * rounds(32, 32);
  // Split product: fitted to 160 launches of drawn projections (16 to 4000 rows, 256 to 4096 columns and elements, one to three
  // products, every form timed on each); the choice is 0.8 % from the best form on average (three forms, of 64 x 128, 64 x 64 and
  // 32 x 64, with constants from nine sizes: 4 %). us fp32 product / 96 x 96 / 64 x 128 / 64 x 96 / 64 x 64 / 32 x 64:
  // 700 x 2048 x 2048 67 / 44 / 46 / 40 / 47 / 51, 1374 x 1536 x 1536 80 / 42 / 69 / 56 / 56 / 62, 700 x 2560 x 2048 70 / 49 / 48 /
  // 69 / 49 / 63, 1248 x 1024 x 512 19 / 19 / 17 / 15 / 17 / 16. A launch of few tiles stays with the fp32 product, whose waves
  // share the contraction of smaller blocks (100 x 768 x 768 8.1 -> 18.6 on 64 x 128, 9.6 on 32 x 64).
  bool vec = true, near96 = true;  // 96 rows of every a within 32-bit offsets; a_vec has looked at 64
  int64_t K = 0;
  for (int i = 0; i < n; i++) {
    vec = vec && args.p[i].a_vec && args.p[i].b_vec;
    near96 = near96 && (96 * args.p[i].as[1] + args.p[i].K) * 4 < kOutOfRange;
    K = std::max<int64_t>(K, args.p[i].K);
  }
  if (vec) {
    const double fp32 = 0.95 * (3.3 + 0.0045 * K * std::min(c64, std::min(c32x64, c32)));
    const double s96 = near96 ? rounds(96, 96) * (10.0 + 0.0160 * K) : INFINITY, s64x128 = rounds(64, 128) * (7.5 + 0.0165 * K);
    const double s64x96 = rounds(64, 96) * (7.0 + 0.0129 * K), s64 = 2.9 + r64 * (2.6 + 0.0096 * K), s32x64 = 3.7 + rounds(32, 64) * (0.9 + 0.0068 * K);
    const double split = std::min({s96, s64x128, s64x96, s64, s32x64});
    if (split < fp32) {
      if (split == s64) return launch_split_form<2, 2>(args, n, stream, copies, n_copies);
      if (split == s32x64) return launch_split_form<1, 2>(args, n, stream, copies, n_copies);
      if (split == s64x96) return launch_split_form<2, 3>(args, n, stream, copies, n_copies);
      if (split == s64x128) return launch_split_form<2, 4>(args, n, stream, copies, n_copies);
      return launch_split_form<3, 3>(args, n, stream, copies, n_copies);
    }
  }
  if (c64 <= c32x64 && c64 <= c32) {
    // with several rounds the other workgroups on a CU cover what eight waves on one block cover in a single round
    // (4096^3: 1062 against 1086 us = 129 TFLOP/s, 82 % of the fp32 matrix peak)
    if (r64 > 4) return launch_form<2, 2, 1>(args, n, stream, copies, n_copies);
    return launch_form<2, 2, 2>(args, n, stream, copies, n_copies);
  }
  if (c32x64 <= c32) return launch_form<1, 2, 2>(args, n, stream, copies, n_copies);
  return launch_form<1, 1, 4>(args, n, stream, copies, n_copies);
}

}  // namespace lmh
