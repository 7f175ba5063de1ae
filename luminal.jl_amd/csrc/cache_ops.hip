// The two operators that sit directly in front of attention on the decode path:
//
//   rotary embedding   apply_rotary_embeddings, reference src/NN.jl:253-303. The reference reshapes
//     the head dim to (D/2, 2) on a column-major array, so the rotated pairs are (j, j + D/2), the
//     "half-split" convention; inv_freq[j] = base^(-2j/D), angle = (prev_seq + s) * inv_freq[j],
//     x0' = x0 cos - x1 sin, x1' = x0 sin + x1 cos. The interleaved pairing (2j, 2j+1) is offered too.
//   KV-cache append    _kv_scatter, reference src/Whisper.jl:552-570, which rebuilds the whole
//     (B, H, max_seq, D) cache by slice + concat to insert one row at step_pos. Here the new rows
//     are written in place at pos[b] .. pos[b]+T-1 (per-sequence positions, device int32[B]), with
//     the rotary embedding of K optionally fused into the same pass.
//
// Both are a few bytes of traffic per element and HBM-bound. The kernels that run for the usual head
// dims move 16-byte chunks: a thread owns the chunk of pairs (j .. j+V-1) — chunk c of the first half
// of the row and chunk c of the second half, or one chunk of interleaved pairs — and, for the
// standalone rotary embedding, evaluates its sin / cos once and walks the heads with them (the angle
// does not depend on the head). Rows whose head dim or alignment does not allow 16-byte chunks take
// the one-element-per-thread kernels.
#include "common.hpp"
#include "copy.hpp"
#include "dtypes.hpp"
#include "rope.hpp"

namespace lmh {
namespace {

template <typename E>
__global__ __launch_bounds__(256) void rope_kernel(RopeArgs a) {
  request_args(a);
  using raw = typename E::raw;
  const int half = a.D / 2;
  const int64_t total = (int64_t)a.B * a.H * a.S * half;
  for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total; idx += (int64_t)gridDim.x * blockDim.x) {
    const int j = (int)(idx % half);
    const int s = (int)((idx / half) % a.S);
    const int h = (int)((idx / ((int64_t)half * a.S)) % a.H);
    const int b = (int)(idx / ((int64_t)half * a.S * a.H));
    const int d0 = a.interleaved ? 2 * j : j;
    const int d1 = a.interleaved ? 2 * j + 1 : j + half;
    const float pos = (float)((a.pos0 ? a.pos0[b] : a.prev_seq) + s);
    const raw *xp = reinterpret_cast<const raw *>(a.x) + b * a.xs[0] + h * a.xs[1] + (int64_t)s * a.xs[2];
    raw *op = reinterpret_cast<raw *>(a.out) + b * a.os[0] + h * a.os[1] + (int64_t)s * a.os[2];
    float o0, o1;
    rope_pair(E::ld(xp[d0]), E::ld(xp[d1]), pos, j, a.D, a.log2_base, &o0, &o1);
    op[d0] = E::st(o0);
    op[d1] = E::st(o1);
  }
}

template <typename E>
__device__ __forceinline__ void append_elements(const KvAppendArgs &a, unsigned n_blocks) {
  using raw = typename E::raw;
  const int64_t total = (int64_t)a.B * a.Hkv * a.T * a.D;
  const int half = a.D / 2;
  const int64_t total_q = a.q ? (int64_t)a.B * a.Hq * a.T * half : 0;  // pairs of this step's queries to rotate in place
  for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total + total_q; idx += (int64_t)n_blocks * blockDim.x) {
    if (idx >= total) {
      const int64_t r = idx - total;
      const int j = (int)(r % half);
      const int t = (int)((r / half) % a.T);
      const int64_t bh = r / ((int64_t)half * a.T);  // b * Hq + h
      const int b = (int)(bh / a.Hq);
      const int d0 = a.interleaved ? 2 * j : j;
      const int d1 = a.interleaved ? 2 * j + 1 : j + half;
      raw *qp = reinterpret_cast<raw *>(a.q) + (bh * a.T + t) * a.D;
      const raw *from = a.q_from ? reinterpret_cast<const raw *>(a.q_from) + (bh * a.T + t) * a.D : qp;
      float o0, o1;
      rope_pair(E::ld(from[d0]), E::ld(from[d1]), (float)((a.pos ? a.pos[b] : a.pos_all) + t), j, a.D, a.log2_base, &o0, &o1);
      qp[d0] = E::st(o0);
      qp[d1] = E::st(o1);
      continue;
    }
    const int d = (int)(idx % a.D);
    const int t = (int)((idx / a.D) % a.T);
    const int h = (int)((idx / ((int64_t)a.D * a.T)) % a.Hkv);
    const int b = (int)(idx / ((int64_t)a.D * a.T * a.Hkv));
    const int row = (a.pos ? a.pos[b] : a.pos_all) + t;
    if (row < 0 || row >= a.Lmax) continue;  // a full cache drops the row instead of writing out of bounds
    const raw *kn = reinterpret_cast<const raw *>(a.k_new) + ((((int64_t)b * a.Hkv + h) * a.T + t) * a.D);
    const raw *vn = reinterpret_cast<const raw *>(a.v_new) + ((((int64_t)b * a.Hkv + h) * a.T + t) * a.D);
    raw *kc = reinterpret_cast<raw *>(a.k_cache) + b * a.ks[0] + h * a.ks[1] + (int64_t)row * a.ks[2];
    raw *vc = reinterpret_cast<raw *>(a.v_cache) + b * a.vs[0] + h * a.vs[1] + (int64_t)row * a.vs[2];
    vc[d] = vn[d];
    if (!a.rope_k) {
      kc[d] = kn[d];
    } else {
      const bool first = a.interleaved ? (d % 2 == 0) : (d < half);
      const int j = a.interleaved ? d / 2 : (d < half ? d : d - half);
      const int dp = a.interleaved ? (first ? d + 1 : d - 1) : (first ? d + half : d - half);
      const float x0 = E::ld(first ? kn[d] : kn[dp]);
      const float x1 = E::ld(first ? kn[dp] : kn[d]);
      float o0, o1;
      rope_pair(x0, x1, (float)row, j, a.D, a.log2_base, &o0, &o1);
      kc[d] = E::st(first ? o0 : o1);
    }
  }
}
template <typename E>
__global__ __launch_bounds__(256) void kv_append_kernel(KvAppendArgs a) {
  request_args(a);
  append_elements<E>(a, gridDim.x);
}
// ... of rows that lie in the caller's arrays: the workgroups from n_blocks on copy those into the graph's buffers.
template <typename E>
__global__ __launch_bounds__(256) void kv_append_fed_kernel(KvAppendArgs a, CopyManyArgs fed, int n_blocks) {
  request_args(a);
  if ((int)blockIdx.x >= n_blocks) return copy_block<256>(fed, blockIdx.x - n_blocks);
  append_elements<E>(a, n_blocks);
}

// 16 bytes of a row, as raw elements
template <typename E>
union Chunk {
  uint4 u;
  typename E::raw e[E::kVec];
};

// x0[i], x1[i] -> rotated in place by (sn[i], cs[i]); same expressions as rope_pair
template <typename E>
__device__ inline void rotate_chunks(Chunk<E> &c0, Chunk<E> &c1, const float *sn, const float *cs) {
#pragma unroll
  for (int i = 0; i < E::kVec; i++) {
    float o0, o1;
    rope_rotate(E::ld(c0.e[i]), E::ld(c1.e[i]), sn[i], cs[i], &o0, &o1);
    c0.e[i] = E::st(o0);
    c1.e[i] = E::st(o1);
  }
}
template <typename E>
__device__ inline void rotate_interleaved(Chunk<E> &c, const float *sn, const float *cs) {
#pragma unroll
  for (int i = 0; i < E::kVec / 2; i++) {
    float o0, o1;
    rope_rotate(E::ld(c.e[2 * i]), E::ld(c.e[2 * i + 1]), sn[i], cs[i], &o0, &o1);
    c.e[2 * i] = E::st(o0);
    c.e[2 * i + 1] = E::st(o1);
  }
}
template <typename E>
__device__ inline void sincos_pairs(float pos, int j0, int n, int D, float log2_base, float *sn, float *cs) {
#pragma unroll
  for (int i = 0; i < E::kVec; i++) {
    if (i >= n) break;
    sincos_angle(pos * rope_inv_freq(j0 + i, D, log2_base), &sn[i], &cs[i]);
  }
}

// Rotary embedding, 16-byte chunks. grid.x covers (b, s, chunk), grid.y blocks of heads.
// IL = false: thread owns pairs j = c V .. c V + V - 1, i.e. chunk c of each half of the row.
// IL = true : thread owns pairs j = c V/2 .. , i.e. chunk c of the row.
template <typename E, bool IL>
__global__ __launch_bounds__(256) void rope_vec_kernel(RopeArgs a, int heads_per_block) {
  request_args(a);
  request_arg(heads_per_block);
  using raw = typename E::raw;
  constexpr int V = E::kVec;
  const int half = a.D / 2;
  const int cpr = IL ? a.D / V : half / V;  // chunks (threads) per row
  const int64_t total = (int64_t)a.B * a.S * cpr;
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= total) return;
  const int c = (int)(idx % cpr);
  const int s = (int)((idx / cpr) % a.S);
  const int b = (int)(idx / ((int64_t)cpr * a.S));
  const float pos = (float)((a.pos0 ? a.pos0[b] : a.prev_seq) + s);
  float sn[V], cs[V];
  sincos_pairs<E>(pos, IL ? c * (V / 2) : c * V, IL ? V / 2 : V, a.D, a.log2_base, sn, cs);
  // Heads in batches of kHeadBatch: all of a batch's loads are issued before the first is used, so a thread has up
  // to 2 * kHeadBatch 16-byte loads in flight (the ~1000 workgroups of a launch alone do not keep HBM busy).
  constexpr int kHeadBatch = 4;
  const int h0 = blockIdx.y * heads_per_block, h1 = min(a.H, h0 + heads_per_block);
  const raw *xrow = reinterpret_cast<const raw *>(a.x) + b * a.xs[0] + (int64_t)s * a.xs[2];
  raw *orow = reinterpret_cast<raw *>(a.out) + b * a.os[0] + (int64_t)s * a.os[2];
  for (int hb = h0; hb < h1; hb += kHeadBatch) {
    Chunk<E> c0[kHeadBatch], c1[kHeadBatch];
#pragma unroll
    for (int i = 0; i < kHeadBatch; i++) {
      if (hb + i >= h1) break;
      const raw *xp = xrow + (hb + i) * a.xs[1];
      c0[i].u = *reinterpret_cast<const uint4 *>(xp + c * V);
      if (!IL) c1[i].u = *reinterpret_cast<const uint4 *>(xp + half + c * V);
    }
#pragma unroll
    for (int i = 0; i < kHeadBatch; i++) {
      if (hb + i >= h1) break;
      raw *op = orow + (hb + i) * a.os[1];
      if (IL) {
        rotate_interleaved<E>(c0[i], sn, cs);
        *reinterpret_cast<uint4 *>(op + c * V) = c0[i].u;
      } else {
        rotate_chunks<E>(c0[i], c1[i], sn, cs);
        *reinterpret_cast<uint4 *>(op + c * V) = c0[i].u;
        *reinterpret_cast<uint4 *>(op + half + c * V) = c1[i].u;
      }
    }
  }
}

// Cache append, 16-byte chunks: a thread owns chunk c of each half of the new rows at (b, t) and walks the KV
// heads of its block (D is a multiple of 2 V), rotating K on the way when asked to. The angle depends on the row
// position and the pair, not on the head, so the sin / cos are evaluated once per thread (they were 17 % of a
// whole-prompt append when every (b, head, t) thread evaluated its own). grid.x covers (b, t, chunk), grid.y
// blocks of heads. The first head's rows are requested before the sin / cos are evaluated, each further head's before the one in
// front of it is stored, and the row's place comes from 32-bit multiplications instead of four 64-bit divisions: a launch that also
// stores 2 x 6.4 MB of k_new and v_new as they are (B=4 H=8 T=777 D=128 fp16) 10.9 -> 9.2 us.
template <typename E>
__device__ __forceinline__ void append_chunks(const KvAppendArgs &a, int heads_per_block, FastDiv by_chunk, FastDiv by_row) {
  using raw = typename E::raw;
  constexpr int V = E::kVec;
  const int half = a.D / 2;
  const int cpr = half / V;
  const uint32_t idx = blockIdx.x * 256 + threadIdx.x;  // below 2^31, as the divisors take it
  if (idx >= (uint32_t)a.B * a.T * cpr) return;
  const uint32_t bt = idx / by_chunk, bq = bt / by_row;
  const int c = (int)(idx - bt * cpr), t = (int)(bt - bq * a.T), b = (int)bq;
  const int row = (a.pos ? a.pos[b] : a.pos_all) + t;
  const bool fits = row >= 0 && row < a.Lmax;  // a full cache drops the row instead of writing out of bounds
  if (!fits && !a.k_copy && !a.v_copy) return;
  const int d0 = c * V, d1 = half + c * V;
  const int h0 = blockIdx.y * heads_per_block, h1 = min(a.Hkv, h0 + heads_per_block);
  Chunk<E> k0, k1;
  uint4 v0, v1;
  auto load = [&](int h) {
    const int64_t src = (((int64_t)b * a.Hkv + h) * a.T + t) * a.D;
    const raw *kn = reinterpret_cast<const raw *>(a.k_new) + src;
    const raw *vn = reinterpret_cast<const raw *>(a.v_new) + src;
    k0.u = load_stream_128(kn + d0);
    k1.u = load_stream_128(kn + d1);
    v0 = load_stream_128(vn + d0);
    v1 = load_stream_128(vn + d1);
  };
  load(h0);  // on its way while the sines are evaluated
  float sn0[V], cs0[V], sn1[V / 2], cs1[V / 2];
  if (a.rope_k) {
    if (a.interleaved) {
      sincos_pairs<E>((float)row, d0 / 2, V / 2, a.D, a.log2_base, sn0, cs0);
      sincos_pairs<E>((float)row, d1 / 2, V / 2, a.D, a.log2_base, sn1, cs1);
    } else {
      sincos_pairs<E>((float)row, d0, V, a.D, a.log2_base, sn0, cs0);
    }
  }
  for (int h = h0; h < h1; h++) {
    Chunk<E> x0 = k0, x1 = k1;
    const uint4 y0 = v0, y1 = v1;
    if (h + 1 < h1) load(h + 1);
    const int64_t src = (((int64_t)b * a.Hkv + h) * a.T + t) * a.D;
    if (a.k_copy) {
      raw *to = reinterpret_cast<raw *>(a.k_copy) + src;
      *reinterpret_cast<uint4 *>(to + d0) = x0.u;
      *reinterpret_cast<uint4 *>(to + d1) = x1.u;
    }
    if (a.v_copy) {
      raw *to = reinterpret_cast<raw *>(a.v_copy) + src;
      *reinterpret_cast<uint4 *>(to + d0) = y0;
      *reinterpret_cast<uint4 *>(to + d1) = y1;
    }
    if (!fits) continue;
    if (a.rope_k) {
      if (a.interleaved) {
        rotate_interleaved<E>(x0, sn0, cs0);
        rotate_interleaved<E>(x1, sn1, cs1);
      } else {
        rotate_chunks<E>(x0, x1, sn0, cs0);
      }
    }
    raw *kc = reinterpret_cast<raw *>(a.k_cache) + b * a.ks[0] + h * a.ks[1] + (int64_t)row * a.ks[2];
    raw *vc = reinterpret_cast<raw *>(a.v_cache) + b * a.vs[0] + h * a.vs[1] + (int64_t)row * a.vs[2];
    *reinterpret_cast<uint4 *>(kc + d0) = x0.u;
    *reinterpret_cast<uint4 *>(kc + d1) = x1.u;
    *reinterpret_cast<uint4 *>(vc + d0) = y0;
    *reinterpret_cast<uint4 *>(vc + d1) = y1;
  }
}

template <typename E>
__global__ __launch_bounds__(256) void kv_append_vec_kernel(KvAppendArgs a, int heads_per_block, FastDiv by_chunk, FastDiv by_row) {
  request_args(a);
  request_arg(heads_per_block);
  append_chunks<E>(a, heads_per_block, by_chunk, by_row);
}
// Copies are the grid's columns from blocks_x on.
template <typename E>
__global__ __launch_bounds__(256) void kv_append_vec_fed_kernel(KvAppendArgs a, int heads_per_block, FastDiv by_chunk, FastDiv by_row, CopyManyArgs fed, int blocks_x, int n_blocks) {
  request_args(a);
  request_arg(heads_per_block);
  if ((int)blockIdx.x >= blocks_x) {
    const int block = (blockIdx.x - blocks_x) * gridDim.y + blockIdx.y;
    if (block < n_blocks) copy_block<256>(fed, block);
    return;
  }
  append_chunks<E>(a, heads_per_block, by_chunk, by_row);
}

bool chunks_ok(const void *p0, const void *p1, const int64_t *s0, const int64_t *s1, int vec) {
  if ((reinterpret_cast<uintptr_t>(p0) | reinterpret_cast<uintptr_t>(p1)) & 15u) return false;
  for (int i = 0; i < 3; i++)
    if (s0[i] % vec != 0 || s1[i] % vec != 0) return false;
  return true;
}

template <typename E>
void launch_rope_vec(const RopeArgs &a, hipStream_t stream) {
  const int cpr = a.interleaved ? a.D / E::kVec : a.D / 2 / E::kVec;
  const int64_t blocks_x = ((int64_t)a.B * a.S * cpr + 255) / 256;
  // about 1024 workgroups fill the chip; beyond that, more heads per thread amortise the sin / cos
  // (C2's Q, 25 MB: 16.9 us with one head per thread, 11.0 us at 3; large tensors lose ~5 % to the longer threads)
#ifndef LMH_ROPE_WGS
#define LMH_ROPE_WGS 1024
#endif
  int blocks_y = (int)((LMH_ROPE_WGS + blocks_x - 1) / blocks_x);
  blocks_y = blocks_y < 1 ? 1 : (blocks_y > a.H ? a.H : blocks_y);
  const int heads_per_block = (a.H + blocks_y - 1) / blocks_y;
  blocks_y = (a.H + heads_per_block - 1) / heads_per_block;
  dim3 grid((unsigned)blocks_x, (unsigned)blocks_y), block(256);
  if (a.interleaved)
    hipLaunchKernelGGL((rope_vec_kernel<E, true>), grid, block, 0, stream, a, heads_per_block);
  else
    hipLaunchKernelGGL((rope_vec_kernel<E, false>), grid, block, 0, stream, a, heads_per_block);
}

int grid_for(int64_t total) {
  int64_t blocks = (total + 255) / 256;
  return (int)(blocks < 1 ? 1 : (blocks > 65536 ? 65536 : blocks));
}

}  // namespace

int launch_rope(const RopeArgs &a, int dtype, hipStream_t stream) {
  const int vec = dtype == LMH_F32 ? 4 : 8;
  const int64_t vec_threads = (int64_t)a.B * a.S * (a.D / vec);
  if (a.D % (a.interleaved ? vec : 2 * vec) == 0 && chunks_ok(a.x, a.out, a.xs, a.os, vec) &&
      a.H <= 65535 && vec_threads / 256 < (int64_t(1) << 31)) {
    switch (dtype) {
      case LMH_F32: launch_rope_vec<F32>(a, stream); break;
      case LMH_F16: launch_rope_vec<F16>(a, stream); break;
      case LMH_BF16: launch_rope_vec<BF16>(a, stream); break;
      default: return fail(LMH_E_UNSUPPORTED, "rope: unknown dtype %d", dtype);
    }
    LMH_HIP_TRY(hipGetLastError());
    return LMH_OK;
  }
  const int64_t total = (int64_t)a.B * a.H * a.S * (a.D / 2);
  dim3 grid(grid_for(total)), block(256);
  switch (dtype) {
    case LMH_F32: hipLaunchKernelGGL(rope_kernel<F32>, grid, block, 0, stream, a); break;
    case LMH_F16: hipLaunchKernelGGL(rope_kernel<F16>, grid, block, 0, stream, a); break;
    case LMH_BF16: hipLaunchKernelGGL(rope_kernel<BF16>, grid, block, 0, stream, a); break;
    default: return fail(LMH_E_UNSUPPORTED, "rope: unknown dtype %d", dtype);
  }
  LMH_HIP_TRY(hipGetLastError());
  return LMH_OK;
}

template <typename E>
static void launch_append_chunks(const KvAppendArgs &a, dim3 grid, int heads_per_block, const CopyManyArgs *fed, int n_copies, hipStream_t stream) {
  const FastDiv by_chunk = fast_div(a.D / (2 * E::kVec)), by_row = fast_div(a.T);
  if (n_copies == 0) {
    hipLaunchKernelGGL(kv_append_vec_kernel<E>, grid, dim3(256), 0, stream, a, heads_per_block, by_chunk, by_row);
    return;
  }
  const int blocks_x = (int)grid.x;
  grid.x += (n_copies + grid.y - 1) / grid.y;
  hipLaunchKernelGGL(kv_append_vec_fed_kernel<E>, grid, dim3(256), 0, stream, a, heads_per_block, by_chunk, by_row, *fed, blocks_x, n_copies);
}

template <typename E>
static void launch_append_elements(const KvAppendArgs &a, int n_blocks, const CopyManyArgs *fed, int n_copies, hipStream_t stream) {
  if (n_copies == 0)
    hipLaunchKernelGGL(kv_append_kernel<E>, dim3(n_blocks), dim3(256), 0, stream, a);
  else
    hipLaunchKernelGGL(kv_append_fed_kernel<E>, dim3(n_blocks + n_copies), dim3(256), 0, stream, a, *fed, n_blocks);
}

int launch_kv_append(KvAppendArgs a, int dtype, hipStream_t stream, CopyManyArgs *fed, int n_fed) {
  const int vec = dtype == LMH_F32 ? 4 : 8;
  const int64_t vec_chunks = (int64_t)a.B * a.Hkv * a.T * (a.D / (2 * vec));  // 16-byte chunk pairs to move
  const int64_t blocks_x = ((int64_t)a.B * a.T * (a.D / (2 * vec)) + 255) / 256;
  if (a.D % (2 * vec) == 0 && chunks_ok(a.k_cache, a.v_cache, a.ks, a.vs, vec) &&
      ((reinterpret_cast<uintptr_t>(a.k_new) | reinterpret_cast<uintptr_t>(a.v_new)) & 15u) == 0 &&
      vec_chunks >= 64 * 256 && blocks_x < (int64_t(1) << 23) && a.Hkv <= 65535) {  // a decode step's few rows: one element per thread is quicker
    // about 2048 workgroups keep enough loads in flight; beyond that a thread walks more heads with one set of sin / cos
    int blocks_y = (int)((2048 + blocks_x - 1) / blocks_x);
    blocks_y = blocks_y < 1 ? 1 : (blocks_y > a.Hkv ? a.Hkv : blocks_y);
    const int heads_per_block = (a.Hkv + blocks_y - 1) / blocks_y;
    blocks_y = (a.Hkv + heads_per_block - 1) / heads_per_block;
    dim3 grid((unsigned)blocks_x, (unsigned)blocks_y);
    // copies of the new rows are stores of what a thread has in its registers
    const int64_t bytes = (int64_t)a.B * a.Hkv * a.T * a.D * (16 / vec);
    auto take = [&](const void *x) -> void * {
      for (int j = 0; j < n_fed; j++)
        if (fed->src[j] == x && fed->bytes[j] == bytes && (reinterpret_cast<uintptr_t>(fed->dst[j]) & 15u) == 0) {
          void *dst = fed->dst[j];
          n_fed--;
          fed->dst[j] = fed->dst[n_fed]; fed->src[j] = fed->src[n_fed]; fed->bytes[j] = fed->bytes[n_fed];
          return dst;
        }
      return nullptr;
    };
    a.k_copy = take(a.k_new);
    a.v_copy = take(a.v_new);
    const int n_copies = n_fed ? (int)number_copy_blocks(*fed, n_fed) : 0;
    switch (dtype) {
      case LMH_F32: launch_append_chunks<F32>(a, grid, heads_per_block, fed, n_copies, stream); break;
      case LMH_F16: launch_append_chunks<F16>(a, grid, heads_per_block, fed, n_copies, stream); break;
      case LMH_BF16: launch_append_chunks<BF16>(a, grid, heads_per_block, fed, n_copies, stream); break;
      default: return fail(LMH_E_UNSUPPORTED, "kv append: unknown dtype %d", dtype);
    }
    LMH_HIP_TRY(hipGetLastError());
    if (!a.q) return LMH_OK;
    // prompt-sized: the queries take the rotary kernel of their own
    RopeArgs r;
    r.out = a.q; r.x = a.q_from ? a.q_from : a.q; r.pos0 = a.pos; r.prev_seq = a.pos_all;
    r.B = a.B; r.H = a.Hq; r.S = a.T; r.D = a.D;
    r.xs[0] = r.os[0] = (int64_t)a.Hq * a.T * a.D; r.xs[1] = r.os[1] = (int64_t)a.T * a.D; r.xs[2] = r.os[2] = a.D;
    r.log2_base = a.log2_base; r.interleaved = a.interleaved;
    return launch_rope(r, dtype, stream);
  }
  const int64_t total = (int64_t)a.B * a.Hkv * a.T * a.D + (a.q ? (int64_t)a.B * a.Hq * a.T * (a.D / 2) : 0);
  const int n_blocks = grid_for(total), n_copies = n_fed ? (int)number_copy_blocks(*fed, n_fed) : 0;
  switch (dtype) {
    case LMH_F32: launch_append_elements<F32>(a, n_blocks, fed, n_copies, stream); break;
    case LMH_F16: launch_append_elements<F16>(a, n_blocks, fed, n_copies, stream); break;
    case LMH_BF16: launch_append_elements<BF16>(a, n_blocks, fed, n_copies, stream); break;
    default: return fail(LMH_E_UNSUPPORTED, "kv append: unknown dtype %d", dtype);
  }
  LMH_HIP_TRY(hipGetLastError());
  return LMH_OK;
}

}  // namespace lmh
