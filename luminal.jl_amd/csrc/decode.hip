// Single-token decode attention over a KV cache, flash-decoding style.
//
// Semantics: the cached attention of reference src/Whisper.jl:584-620 (attend over rows
// 0 .. step_pos of a (B, H, max_seq, D) cache, plain softmax) with the GQA head sharing of
// reference src/NN.jl:305-317, per-sequence lengths and no cache rewrite.
//
// The op is HBM-bound: every K and V element has to cross the memory bus once and is used for
// 2*G flops. The design follows from that:
//   * one workgroup per (sequence, KV head, KV split): the G query heads that share a KV head are
//     processed together from registers, so K/V are read once per KV head, not once per query
//     head;
//   * a key row is covered by LPK adjacent lanes, each issuing one 128-bit load, so a wave's load
//     instruction touches 64/LPK complete, contiguous rows;
//   * U independent K loads and U V loads are in flight per lane before the first use;
//   * ragged lengths: grid.x spans ceil(Lmax/chunk) splits, a workgroup whose split starts past
//     kv_len[b] exits at once, and the merge kernel reads only the splits that exist;
//   * split partials (running max, sum, un-normalised output) go to a caller-owned workspace and
//     a second small kernel merges them with the log-sum-exp identity.
#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "copy.hpp"
#include "dtypes.hpp"
#include "rope.hpp"

namespace lmh {
namespace {

constexpr int kWaves = 4;
constexpr int kUnroll = 4;  // key steps per wave per iteration
constexpr float kLog2e = 1.4426950408889634f;

// All-reduce (sum) over the LPK adjacent lanes that share a key. Up to 16 lanes this is pure DPP
// (no LDS round trip): after the two quad steps every lane of a quad holds the quad sum, so the
// mirror patterns, which pair quad 0 with 1 (and 2 with 3), then half row 0 with 1, finish it.
template <int LPK>
__device__ inline float sum_within_key(float x) {
  if (LPK >= 2) x += dpp<kDppXor1>(x);
  if (LPK >= 4) x += dpp<kDppXor2>(x);
  if (LPK >= 8) x += dpp<kDppHalfMirror>(x);
  if (LPK >= 16) x += dpp<kDppMirror>(x);
  if (LPK >= 32) x += __shfl_xor(x, 16);
  if (LPK >= 64) x += __shfl_xor(x, 32);
  return x;
}
// Reductions over the key slots of a wave (lane bits at and above LPK); used once, after the loop.
template <int LPK>
__device__ inline float sum_across_slots(float x) {
#pragma unroll
  for (int off = LPK; off < 64; off <<= 1) x += __shfl_xor(x, off);
  return x;
}
template <int LPK>
__device__ inline float max_across_slots(float x) {
#pragma unroll
  for (int off = LPK; off < 64; off <<= 1) x = fmaxf(x, __shfl_xor(x, off));
  return x;
}

// q in the form the dot product wants: fp32 for fp32 tensors, the original packed 16-bit pairs for
// fp16 / bf16 (v_dot2_f32_f16 / v_dot2_f32_bf16: two exact products + fp32 accumulate per op).
template <typename E>
struct QFrag;
template <>
struct QFrag<F32> {
  float q[4];
  __device__ void load(const float *p, bool ok) {
#pragma unroll
    for (int e = 0; e < 4; e++) q[e] = ok ? p[e] : 0.f;
  }
  __device__ float dot(const Vec128<F32> &k) const { return q[0] * k.r.x + q[1] * k.r.y + q[2] * k.r.z + q[3] * k.r.w; }
};
template <>
struct QFrag<F16> {
  uint32_t q[4];
  __device__ void load(const _Float16 *p, bool ok) {
    const uint16_t *u = reinterpret_cast<const uint16_t *>(p);
#pragma unroll
    for (int e = 0; e < 4; e++) q[e] = ok ? ((uint32_t)u[2 * e] | ((uint32_t)u[2 * e + 1] << 16)) : 0u;
  }
  __device__ float dot(const Vec128<F16> &k) const {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    const uint32_t w[4] = {k.r.x, k.r.y, k.r.z, k.r.w};
    float acc = 0.f;
#pragma unroll
    for (int e = 0; e < 4; e++)
      acc = __builtin_amdgcn_fdot2(__builtin_bit_cast(h2, q[e]), __builtin_bit_cast(h2, w[e]), acc, false);
    return acc;
  }
};
template <>
struct QFrag<BF16> {
  uint32_t q[4];
  __device__ void load(const uint16_t *u, bool ok) {
#pragma unroll
    for (int e = 0; e < 4; e++) q[e] = ok ? ((uint32_t)u[2 * e] | ((uint32_t)u[2 * e + 1] << 16)) : 0u;
  }
  __device__ float dot(const Vec128<BF16> &k) const {
    typedef __bf16 b2 __attribute__((ext_vector_type(2)));
    const uint32_t w[4] = {k.r.x, k.r.y, k.r.z, k.r.w};
    float acc = 0.f;
#pragma unroll
    for (int e = 0; e < 4; e++)
      acc = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(b2, q[e]), __builtin_bit_cast(b2, w[e]), acc, false);
    return acc;
  }
};

// E: element type; LPK: lanes per key row (power of two, LPK * E::kVec >= D); G: query heads
// handled per workgroup (the GQA group, or a slice of it).
//
// Every key slot (a group of LPK lanes) runs its own online softmax over the keys it sees: the
// running max, sum and output slice are slot-local, so the loop has no traffic between slots and,
// for LPK <= 16, none through LDS at all. Slots, then waves, are merged once after the loop.
// W waves: four, several workgroups on a CU, or eight or sixteen for launches of few workgroups (one_split, few_units below). (With the next
// rows asked for ahead, the same short walks took longer: fp16 B=16 Hkv=16 L=258 D=80 6.6 us, 7.6 so.)
template <typename E, int LPK, int G, int W>
__global__ __launch_bounds__(W * 64) void decode_split_kernel(DecodeArgs a, int g_chunks) {
  request_args(a);
  request_arg(g_chunks);
  using raw = typename E::raw;
  constexpr int VEC = E::kVec;
  constexpr int KPW = 64 / LPK;                          // keys per wave per load step
  constexpr int KEYS_PER_ITER = W * kUnroll * KPW;  // keys per workgroup iteration

  const int split = blockIdx.x;
  const int kvh = blockIdx.y / g_chunks;
  const int g0 = (blockIdx.y % g_chunks) * G;  // first group member handled here
  const int b = blockIdx.z;
  const int group = a.Hq / a.Hkv;

  int L = a.kv_len ? a.kv_len[b] : a.Lmax;
  L = min(max(L, 0), a.Lmax);
  const int start = split * a.chunk;
  const int tid = threadIdx.x;
  if (start >= L) {  // ragged tail: this split does not exist for sequence b
    // ... and with a single split nobody else writes the rows of a sequence without keys: zeros, like every
    // other kernel of the library
    if (a.num_splits == 1) {
      for (int idx = tid; idx < G * a.D; idx += W * 64) {
        const int gi = g0 + idx / a.D;
        if (gi >= group) continue;
        const int64_t off = b * a.os[0] + q_head_of(kvh, gi, a.Hq, a.Hkv, a.head_map) * a.os[1] + idx % a.D;
        if (a.out_f32) reinterpret_cast<float *>(a.out)[off] = 0.f;
        else reinterpret_cast<raw *>(a.out)[off] = E::st(0.f);
      }
    }
    return;
  }
  const int end = min(L, start + a.chunk);

  const int lane = tid & 63, wave = tid >> 6;
  const int slot = lane / LPK;
  const int c = lane % LPK;
  const int d0 = c * VEC;
  const bool lane_active = d0 < a.D;  // D is a multiple of VEC (checked on the host)

  QFrag<E> qf[G];
#pragma unroll
  for (int g = 0; g < G; g++) {
    const int gi = g0 + g;
    const bool head_ok = gi < group;
    const int hq = q_head_of(kvh, head_ok ? gi : 0, a.Hq, a.Hkv, a.head_map);
    const raw *qp = reinterpret_cast<const raw *>(a.q) + b * a.qs[0] + hq * a.qs[1];
    qf[g].load(qp + (lane_active ? d0 : 0), lane_active && head_ok);
  }
  const float qmul = a.scale * kLog2e;  // scores in log2 units: softmax runs on exp2

  const raw *kbase = reinterpret_cast<const raw *>(a.k) + b * a.ks[0] + kvh * a.ks[1] + d0;
  const raw *vbase = reinterpret_cast<const raw *>(a.v) + b * a.vs[0] + kvh * a.vs[1] + d0;

  float m[G], l[G], acc[G][VEC];
#pragma unroll
  for (int g = 0; g < G; g++) {
    m[g] = -INFINITY;
    l[g] = 0.f;
#pragma unroll
    for (int e = 0; e < VEC; e++) acc[g][e] = 0.f;
  }

  // (A row and its use in functions of their own: written in one stretch the compiler moves the conversion of a V row into the branch around its load and
  // waits there, four times an iteration: fp16 B=92 Hkv=12 L=131 D=80 in one launch 12.7 us, 10.4 so. The two conditions of a load as one: a
  // branch for each of the first rows put steps of fp32 20 heads L=357 D=256 at 20.2 us, 19.7 so, as with the loop in one stretch.)
  struct Rows {
    Vec128<E> k[kUnroll], v[kUnroll];
    bool valid[kUnroll];
  };
  auto load = [&](Rows &r, int it0) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < kUnroll; u++) {
      const int key = it0 + (wave * kUnroll + u) * KPW + slot;
      r.valid[u] = key < end;
      if (r.valid[u] & lane_active) {
        r.k[u].load_stream(kbase + (int64_t)key * a.ks[2]);
      } else {
        r.k[u].zero();
      }
    }
#pragma unroll
    for (int u = 0; u < kUnroll; u++) {
      const int key = it0 + (wave * kUnroll + u) * KPW + slot;
      if (r.valid[u] & lane_active) {
        r.v[u].load_stream(vbase + (int64_t)key * a.vs[2]);
      } else {
        r.v[u].zero();
      }
    }
  };
  auto attend = [&](const Rows &r) __attribute__((always_inline)) {
    float s[kUnroll][G];  // not yet in log2 units
    float blk_max[G];
#pragma unroll
    for (int g = 0; g < G; g++) blk_max[g] = -INFINITY;
#pragma unroll
    for (int u = 0; u < kUnroll; u++) {
#pragma unroll
      for (int g = 0; g < G; g++) {
        s[u][g] = sum_within_key<LPK>(qf[g].dot(r.k[u]));
        blk_max[g] = fmaxf(blk_max[g], r.valid[u] ? s[u][g] * qmul : -INFINITY);
      }
    }
#pragma unroll
    for (int g = 0; g < G; g++) {
      const float m_new = fmaxf(m[g], blk_max[g]);
      // m_new is -inf only while this slot has seen no valid key; then everything stays 0.
      const float alpha = (m[g] == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f(m[g] - m_new);
      m[g] = m_new;
      l[g] *= alpha;
#pragma unroll
      for (int e = 0; e < VEC; e++) acc[g][e] *= alpha;
    }
#pragma unroll
    for (int u = 0; u < kUnroll; u++) {
      float vf[VEC];
      r.v[u].unpack(vf);
#pragma unroll
      for (int g = 0; g < G; g++) {
        const float p = r.valid[u] ? __builtin_amdgcn_exp2f(fmaf(s[u][g], qmul, -m[g])) : 0.f;
        l[g] += p;
#pragma unroll
        for (int e = 0; e < VEC; e++) acc[g][e] += p * vf[e];
      }
    }
  };
  for (int it0 = start; it0 < end; it0 += KEYS_PER_ITER) {
    Rows rows;
    load(rows, it0);
    attend(rows);
  }

  // Merge the key slots of each wave (bring them to the wave's max first), then the waves.
  __shared__ float sm_m[W][G];
  __shared__ float sm_l[W][G];
  __shared__ float sm_acc[W][G][LPK * VEC];
#pragma unroll
  for (int g = 0; g < G; g++) {
    const float m_wave = max_across_slots<LPK>(m[g]);
    const float f = (m[g] == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f(m[g] - m_wave);
    l[g] = sum_across_slots<LPK>(l[g] * f);
#pragma unroll
    for (int e = 0; e < VEC; e++) acc[g][e] = sum_across_slots<LPK>(acc[g][e] * f);
    if (slot == 0) {
#pragma unroll
      for (int e = 0; e < VEC; e++) sm_acc[wave][g][d0 + e] = acc[g][e];
      if (c == 0) {
        sm_m[wave][g] = m_wave;
        sm_l[wave][g] = l[g];
      }
    }
  }
  __syncthreads();

  for (int idx = tid; idx < G * a.D; idx += W * 64) {
    const int g = idx / a.D, d = idx % a.D;
    const int gi = g0 + g;
    if (gi >= group) continue;
    float M = -INFINITY;
#pragma unroll
    for (int w = 0; w < W; w++) M = fmaxf(M, sm_m[w][g]);
    float lsum = 0.f, o = 0.f;
#pragma unroll
    for (int w = 0; w < W; w++) {
      const float f = (sm_m[w][g] == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f(sm_m[w][g] - M);
      lsum += sm_l[w][g] * f;
      o += sm_acc[w][g][d] * f;
    }
    const int hq = q_head_of(kvh, gi, a.Hq, a.Hkv, a.head_map);
    if (a.num_splits == 1) {
      const int64_t off = b * a.os[0] + hq * a.os[1] + d;
      if (a.out_f32) reinterpret_cast<float *>(a.out)[off] = o / lsum;
      else reinterpret_cast<raw *>(a.out)[off] = E::st(o / lsum);
    } else {
      const int64_t row = ((int64_t)b * a.Hq + hq) * a.num_splits + split;
      a.ws_o[row * a.D + d] = o;
      if (d == 0) {
        a.ws_ml[row * 2 + 0] = M;
        a.ws_ml[row * 2 + 1] = lsum;
      }
    }
  }
}

// out[b,hq,:] = sum_s o_s 2^(m_s - M) / sum_s l_s 2^(m_s - M) over the splits that exist.
// One workgroup per (b, hq). The slot statistics are fetched in parallel (one slot per thread), reduced
// across the workgroup, and the per-slot weights go through LDS, so the loop over slots that follows
// issues independent loads of the partial outputs instead of a chain of dependent ones.
constexpr int kMergeThreads = 128;
constexpr int kMergeMaxSlots = 1024;  // weights kept in LDS; more slots than this take the strided path below
constexpr int kMergePrefetch = 16;     // partial rows fetched before the slot statistics are known
// STEP (lmh_decode_step): the row this step appends, kv_len[b], never went through the split kernel. It joins here as
// one more partial — score q . k_new (both rotated at position kv_len[b] when a.q_rope, and rounded to the element
// type as the stored rows are), sum 1, output v_new — and the workgroup of the first query head of every KV head
// writes the row into the caches (the reference rebuilds them with _kv_scatter, src/Whisper.jl:552-570).
template <typename E, bool STEP>
__device__ __forceinline__ void merge_row(const DecodeArgs &a, int hq, int b) {
  using raw = typename E::raw;
  __shared__ float w_s[kMergeMaxSlots];
  __shared__ uint16_t full_s[kMergeMaxSlots];  // slots behind the prefetched ones that hold something
  __shared__ float red_m[kMergeThreads / 64], red_l[kMergeThreads / 64], red_s[kMergeThreads / 64];
  const int tid = threadIdx.x;
  const int64_t off = b * a.os[0] + hq * a.os[1];
  const int64_t row0 = ((int64_t)b * a.Hq + hq) * a.num_splits;
  const float2 *ml = reinterpret_cast<const float2 *>(a.ws_ml) + row0;
  const float *po = a.ws_o + row0 * a.D;

  // The kernel is a chain of round trips to memory the split kernel has just written (kv_len, the slot statistics,
  // the partial rows), each about as long as the arithmetic of the whole kernel. The rows of the first slots do
  // not depend on the others: they are requested first, and travel while the statistics are reduced. Rows of
  // slots that turn out not to exist or to be empty are unset memory and are discarded unread below.
  // So is the new row, whose place in memory does not depend on the length either (asked for where each part is used, its value behind
  // everything else, steps of bf16 B=1 L=8192 D=128 took 14.2 us instead of 13.9, B=16 L=4096 46.4 instead of 45.9).
  const int kvh = STEP ? kv_head_of(hq, a.Hq, a.Hkv, a.head_map) : 0;
  const int64_t new_row = ((int64_t)b * a.Hkv + kvh) * a.D;
  const raw *v_new_row = reinterpret_cast<const raw *>(a.v_new) + new_row;
  // element d of the query and of the new key, with the partner that the rotation pairs it with, and of the new value
  struct Fresh { raw q, q_pair, k, k_pair, v; };
  auto partner = [&](int d) { return !a.q_rope ? d : a.rope_interleaved ? d ^ 1 : d < a.D / 2 ? d + a.D / 2 : d - a.D / 2; };
  auto fetch_new = [&](int d) {
    const raw *q_row = reinterpret_cast<const raw *>(a.q) + b * a.qs[0] + hq * a.qs[1];
    const raw *k_row = reinterpret_cast<const raw *>(a.k_new) + new_row;
    return Fresh{q_row[d], q_row[partner(d)], k_row[d], k_row[partner(d)], v_new_row[d]};
  };
  const int first_d = min(tid, a.D - 1);
  Fresh fresh = {};
  if (STEP) fresh = fetch_new(first_d);
  float pre[kMergePrefetch];
  const int n_pre = min(a.num_splits, kMergePrefetch);
#pragma unroll
  for (int u = 0; u < kMergePrefetch; u++) pre[u] = po[(int64_t)min(u, n_pre - 1) * a.D + first_d];

  int L = a.kv_len ? a.kv_len[b] : a.Lmax;
  L = min(max(L, 0), a.Lmax);
  const int n = (L + a.chunk - 1) / a.chunk;

  // (this thread's first slot statistics are requested before the new row's arithmetic, not after its barrier)
  const float2 ml_first = tid < n ? ml[tid] : make_float2(-INFINITY, 0.f);
  // the new row: its score in log2 units, and (first query head of the KV head only) its place in the caches
  float m_new = -INFINITY;
  const bool appends = STEP && L < a.Lmax;
  if (appends) {
    const bool writer = q_head_of(kvh, 0, a.Hq, a.Hkv, a.head_map) == hq;
    raw *k_dst = const_cast<raw *>(reinterpret_cast<const raw *>(a.k)) + b * a.ks[0] + kvh * a.ks[1] + (int64_t)L * a.ks[2];
    raw *v_dst = const_cast<raw *>(reinterpret_cast<const raw *>(a.v)) + b * a.vs[0] + kvh * a.vs[1] + (int64_t)L * a.vs[2];
    float dot = 0.f;
    for (int d = tid; d < a.D; d += kMergeThreads) {
      const Fresh x = d == tid ? fresh : fetch_new(d);
      raw qr = x.q, kr = x.k;
      if (a.q_rope) {  // (rope_element of both, with one sine)
        const bool first = a.rope_interleaved ? d % 2 == 0 : d < a.D / 2;
        const int j = a.rope_interleaved ? d / 2 : first ? d : d - a.D / 2;
        float sn, cs, o0, o1;
        sincos_angle((float)L * rope_inv_freq(j, a.D, a.rope_log2_base), &sn, &cs);
        rope_rotate(E::ld(first ? x.q : x.q_pair), E::ld(first ? x.q_pair : x.q), sn, cs, &o0, &o1);
        qr = E::st(first ? o0 : o1);
        rope_rotate(E::ld(first ? x.k : x.k_pair), E::ld(first ? x.k_pair : x.k), sn, cs, &o0, &o1);
        kr = E::st(first ? o0 : o1);
      }
      dot += E::ld(qr) * E::ld(kr);
      if (writer) {
        k_dst[d] = kr;
        v_dst[d] = x.v;
      }
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) dot += __shfl_xor(dot, o);
    if ((tid & 63) == 0) red_s[tid >> 6] = dot;
    __syncthreads();
    dot = 0.f;
#pragma unroll
    for (int w = 0; w < kMergeThreads / 64; w++) dot += red_s[w];
    m_new = dot * a.scale * kLog2e;
  }

  // running max over the slots
  float M = fmaxf(m_new, ml_first.x);
  for (int s = tid + kMergeThreads; s < n; s += kMergeThreads) M = fmaxf(M, ml[s].x);
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) M = fmaxf(M, __shfl_xor(M, o));
  if ((tid & 63) == 0) red_m[tid >> 6] = M;
  __syncthreads();
  M = red_m[0];
#pragma unroll
  for (int w = 1; w < kMergeThreads / 64; w++) M = fmaxf(M, red_m[w]);

  // weights 2^(m_s - M) (0 for a slot marked (-inf, 0): it was folded into an earlier slot of the same
  // run and its output row is unset) and the normaliser
  float lsum = 0.f;
  for (int s = tid; s < n; s += kMergeThreads) {
    const float2 v = s == tid ? ml_first : ml[s];
    const float w = v.x == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(v.x - M);
    if (s < kMergeMaxSlots) w_s[s] = w;
    lsum += v.y * w;
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) lsum += __shfl_xor(lsum, o);
  if ((tid & 63) == 0) red_l[tid >> 6] = lsum;
  __syncthreads();
  lsum = 0.f;
#pragma unroll
  for (int w = 0; w < kMergeThreads / 64; w++) lsum += red_l[w];
  // Most slots behind the prefetched ones are empty where a workgroup walks several chunks of a sequence (a slot per chunk, one
  // row per run of them): their rows are not read (B=64 H=32/8 up to 32768 keys D=128, 64 slots: the whole call 849.7 -> 842.2 us). Up to
  // twice as many slots as are prefetched, and where more than half hold something, all of them are fetched as they come, whose
  // addresses wait for nothing (B=1 L=32768, 32 slots, none empty: 29.0, skipping 30.4; B=2 H=32/4 L=26420 D=80, 207 of them: 37.5 and 44.7).
  const int n_lds = min(n, kMergeMaxSlots), n_p = min(n_lds, n_pre) & ~3;
  const bool counted = n_lds > 2 * kMergePrefetch;
  int n_full = 0;
  for (int base = n_p; counted && base < n_lds; base += 64) {  // (every wave finds the same ones)
    const int s = base + (tid & 63);
    const uint64_t full = __builtin_amdgcn_ballot_w64(s < n_lds && w_s[s] != 0.f);
    if (full >> (tid & 63) & 1) full_s[n_full + __builtin_popcountll(full & ((uint64_t(1) << (tid & 63)) - 1))] = (uint16_t)s;
    n_full += __builtin_popcountll(full);
  }
  const bool skip = counted && 2 * n_full <= n_lds - n_p;
  if (!skip) n_full = 0;
  const float w_new = appends ? __builtin_amdgcn_exp2f(m_new - M) : 0.f;  // the new row's sum is 1
  lsum += w_new;
  const float inv = lsum > 0.f ? 1.f / lsum : 0.f;

  for (int d = tid; d < a.D; d += kMergeThreads) {
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    int s = 0;
    if (d == tid) {  // the prefetched rows (same summation order as below: slot s adds to acc[s % 4])
#pragma unroll
      for (int u = 0; u < kMergePrefetch; u++) {
        if (u < n_p) {
          const float w = w_s[u];
          // the row of a zero-weight slot is unset memory: select, do not multiply
          acc[u & 3] += w != 0.f ? pre[u] * w : 0.f;
        }
      }
      s = n_p;
    }
    for (const int end = skip ? n_p : n_lds; s + 4 <= end; s += 4) {
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const float w = w_s[s + u];
        const float x = po[(int64_t)(s + u) * a.D + d];
        acc[u] += w != 0.f ? x * w : 0.f;
      }
    }
    for (int f = 0; f < n_full; f += 8) {
      float x[8];
#pragma unroll
      for (int u = 0; u < 8; u++) x[u] = f + u < n_full ? po[(int64_t)full_s[f + u] * a.D + d] : 0.f;
#pragma unroll
      for (int u = 0; u < 8; u++) {
        if (f + u >= n_full) break;
        const int slot = full_s[f + u];
        const float y = x[u] * w_s[slot];
#pragma unroll
        for (int q = 0; q < 4; q++) acc[q] += (slot & 3) == q ? y : 0.f;
      }
    }
    for (s = skip ? n_lds : s; s < n; s++) {
      const float w = s < kMergeMaxSlots ? w_s[s] : (ml[s].x == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(ml[s].x - M));
      const float x = po[(int64_t)s * a.D + d];
      acc[0] += w != 0.f ? x * w : 0.f;
    }
    float o = (acc[0] + acc[1]) + (acc[2] + acc[3]);
    if (appends) o += w_new * E::ld(d == tid ? fresh.v : v_new_row[d]);
    if (a.out_f32) reinterpret_cast<float *>(a.out)[off + d] = o * inv;
    else reinterpret_cast<raw *>(a.out)[off + d] = E::st(o * inv);
  }
}

template <typename E, bool STEP>
__global__ __launch_bounds__(kMergeThreads) void decode_merge_kernel(DecodeArgs a) {
  request_args(a);
  merge_row<E, STEP>(a, blockIdx.x, blockIdx.y);
}
// ... of a step whose operands lie in the caller's arrays: further workgroups copy those into the graph's buffers, which nothing
// else in the step waits for (bf16 steps of B=16 H=32/8 L=4096 D=128: 53.5 us with the copy in front, 50.3 here).
template <typename E>
__global__ __launch_bounds__(kMergeThreads) void decode_merge_fed_kernel(DecodeArgs a, CopyManyArgs fed, int n_copies) {
  request_args(a);
  if ((int)blockIdx.y >= a.B) {
    const int block = (blockIdx.y - a.B) * a.Hq + blockIdx.x;
    if (block < n_copies) copy_block<kMergeThreads>(fed, block);
    return;
  }
  merge_row<E, true>(a, blockIdx.x, blockIdx.y);
}

template <typename E>
int launch_merge(const DecodeArgs &a, hipStream_t stream, const CopyManyArgs *fed, int n_copies) {
  if (a.step && n_copies > 0) {
    hipLaunchKernelGGL((decode_merge_fed_kernel<E>), dim3(a.Hq, a.B + (n_copies + a.Hq - 1) / a.Hq), dim3(kMergeThreads), 0, stream, a, *fed, n_copies);
    LMH_HIP_TRY(hipGetLastError());
  } else if (a.step) {  // (with partials: a step of one split is one launch)
    hipLaunchKernelGGL((decode_merge_kernel<E, true>), dim3(a.Hq, a.B), dim3(kMergeThreads), 0, stream, a);
    LMH_HIP_TRY(hipGetLastError());
  } else if (a.num_splits > 1) {
    hipLaunchKernelGGL((decode_merge_kernel<E, false>), dim3(a.Hq, a.B), dim3(kMergeThreads), 0, stream, a);
    LMH_HIP_TRY(hipGetLastError());
  }
  return LMH_OK;
}

// What a launch of decode_split_kernel is made of.
struct SplitForm {
  int lanes, heads;   // lanes per key row, query heads per workgroup
  int64_t units;      // (sequence, KV head, slice of its query heads)
  int keys, wide_keys;  // that four waves, and the wide workgroup's, take an iteration
};
// (Four heads in 16 bits: on sixteen waves 72 decodes of head dims 72 to 192 and up to 16 units took 4 % more in the mean, B=2 4/1 heads L=20000 D=72 bf16 19.8 us
// and 24.5, 24.6 with partials of four waves.)
constexpr int wide_waves(int heads, int vec) { return heads * vec >= 32 ? 8 : 16; }
SplitForm split_form(const DecodeArgs &a, int vec) {
  SplitForm f;
  const int group = a.Hq / a.Hkv, chunks = (a.D + vec - 1) / vec;
  f.lanes = chunks <= 4 ? 4 : chunks <= 8 ? 8 : chunks <= 16 ? 16 : chunks <= 32 ? 32 : 64;
  f.heads = group == 1 ? 1 : group == 2 ? 2 : group <= 4 ? 4 : 8;
  f.units = (int64_t)a.B * a.Hkv * ((group + f.heads - 1) / f.heads);
  f.keys = kWaves * kUnroll * (64 / f.lanes);
  f.wide_keys = f.keys / kWaves * wide_waves(f.heads, vec);
  return f;
}
// Walks so short that one workgroup takes all of a unit's keys in less time than the merge launch adds: us with the partials and without, every sequence Lmax
// long, fp32 B=2 Hkv=16 L=182 D=128 10.9 and 6.7, B=4 Hkv=12 L=242 10.5 and 7.3, L=460 D=64 32 heads of 2 9.0 and 7.1, fp16 B=20 Hkv=4 L=174 D=80 10.4 and 6.0,
// bf16 B=5 Hkv=20 L=529 9.7 and 8.7. A CU fetches 65 bytes a ns, so it ends where the wide workgroup has two and a half iterations of 64 or 128 KB to walk,
// three and a half from half the CUs on (fp32 L=858 D=64 176 units 16.0 and 13.7); with two heads in 16 bits, short rows and up to a fifth of the CUs after two
// (fp16 B=2 12/6 heads L=575 D=72 9.2 and 10.1, B=17 2/1 L=520 9.8 and 10.9; B=50 2/1 L=258 D=192 13.5 and 10.8), with four and more the arithmetic counts as
// well (fp32 B=12 32/8 heads L=535 D=128 17.4 and 23.6, B=4 64/8 L=256 D=96 19.2 and 19.5). More units than CUs go round in four waves: fp32 B=54 Hkv=8 L=152
// D=64 13.1 and 7.1, fp16 B=21 64/32 heads L=183 D=80 16.9 and 10.4, fp32 B=11 Hkv=32 L=446 D=64 16.6 and 13.7. So do walks of up to three and a half
// iterations of four waves (bf16 B=3 24/12 heads L=83 D=80 5.3, on sixteen waves 6.4; fp32 B=9 48/12 heads L=117 D=128 10.2 and 8.5).
bool one_split(const SplitForm &f, int Lmax, int vec, int64_t cus) {
  if (f.units > cus) return Lmax <= (f.heads <= 2 ? 448 : 256);
  if (f.heads * vec >= 32) return Lmax * 5 <= f.wide_keys * 6;
  if (f.heads == 2 && vec == 8 && f.lanes <= 16 && 5 * f.units <= cus) return Lmax <= f.wide_keys * 2;
  return f.heads > 2 || 2 * f.units < cus ? Lmax * 5 <= f.wide_keys * 12 : Lmax * 5 <= f.wide_keys * 17;
}
// Few units and long walks: a wide workgroup a CU, and with it fewer partials (bf16 B=2 Hkv=1 L=29834 D=80 25.4 -> 16.4 us, fp16 B=3 Hkv=2 L=18681 24.3 ->
// 13.5, B=3 Hkv=4 L=24282 30.3 -> 19.8, fp32 B=2 8/4 heads L=11136 D=128 24.7 -> 20.8; 24 to 32 units come out even). 94 drawn ones of full length are
// 1.34 times as fast in the mean, 90 with lengths from Lmax / 4 up 1.23 times; of these, one or two sequences a third of Lmax long leave CUs idle, the worst loses
// 30 % (fp32 B=1 64/16 heads Lmax=12573 D=80 25.0 and 32.5). Where a CU gets less than an iteration of it the waves that stay idle cost more (bf16 Hkv=6
// L=1691 D=80 8.7 and 9.8, fp32 32/16 heads L=4792 D=64 12.0 and 12.8).
bool few_units(const SplitForm &f, int Lmax, int64_t cus) {
  return f.units * 16 <= cus && f.heads <= 4 && f.units * Lmax * 8 >= cus * f.wide_keys * (f.units <= 8 ? 7 : 12);
}

template <typename E, int LPK>
int launch_for_lpk(const DecodeArgs &a, hipStream_t stream) {
  const SplitForm f = split_form(a, E::kVec);
  const int64_t cus = device_cu_count();
  const bool wide = a.num_splits == 1 ? f.units <= cus && 2 * a.Lmax > 7 * f.keys && f.heads * E::kVec < 32 && one_split(f, a.Lmax, E::kVec, cus)
                                      : few_units(f, a.Lmax, cus) && f.units * a.num_splits <= cus;
  if (plan_only("decode_split_kernel<%s, lanes a key=%d, heads=%d, waves=%d> splits=%d", E::kName, LPK, f.heads, wide && f.heads <= 4 ? wide_waves(f.heads, E::kVec) : kWaves,
                a.num_splits))
    return LMH_OK;
  auto launch = [&](auto heads) {
    constexpr int G = decltype(heads)::value, W = wide_waves(G, E::kVec);
    const int g_chunks = (a.Hq / a.Hkv + G - 1) / G;
    const dim3 grid(a.num_splits, a.Hkv * g_chunks, a.B);
    if constexpr (G <= 4)
      if (wide) {
        hipLaunchKernelGGL((decode_split_kernel<E, LPK, G, W>), grid, dim3(W * 64), 0, stream, a, g_chunks);
        return;
      }
    hipLaunchKernelGGL((decode_split_kernel<E, LPK, G, kWaves>), grid, dim3(kWaves * 64), 0, stream, a, g_chunks);
  };
  if (f.heads == 1) launch(std::integral_constant<int, 1>{});
  else if (f.heads == 2) launch(std::integral_constant<int, 2>{});
  else if (f.heads == 4) launch(std::integral_constant<int, 4>{});
  else launch(std::integral_constant<int, 8>{});
  LMH_HIP_TRY(hipGetLastError());
  return launch_merge<E>(a, stream, nullptr, 0);
}

template <typename E>
int launch_for_dtype(const DecodeArgs &a, hipStream_t stream) {
  const int chunks = (a.D + E::kVec - 1) / E::kVec;
  if (chunks <= 4) return launch_for_lpk<E, 4>(a, stream);
  if (chunks <= 8) return launch_for_lpk<E, 8>(a, stream);
  if (chunks <= 16) return launch_for_lpk<E, 16>(a, stream);
  if (chunks <= 32) return launch_for_lpk<E, 32>(a, stream);
  if constexpr (256 / E::kVec > 32)  // (head dims up to 256)
    if (chunks <= 64) return launch_for_lpk<E, 64>(a, stream);
  return fail(LMH_E_UNSUPPORTED, "decode attention: head dim %d too large", a.D);
}

}  // namespace

int decode_chunk_for(int Lmax, int num_splits) {
  if (num_splits < 1) num_splits = 1;
  int chunk = (Lmax + num_splits - 1) / num_splits;
  chunk = (chunk + 63) / 64 * 64;
  return chunk < 64 ? 64 : chunk;
}

// Splits of decode_split_kernel where the caller leaves the count to the library, at most `most`.
int32_t decode_valu_splits(const DecodeArgs &a, int dtype, int32_t most) {
  const int vec = dtype == LMH_F32 ? F32::kVec : F16::kVec;
  const SplitForm f = split_form(a, vec);
  const int64_t cus = device_cu_count();
  if (one_split(f, a.Lmax, vec, cus)) return 1;
  return few_units(f, a.Lmax, cus) ? (int32_t)std::min<int64_t>(most, cus / f.units) : most;
}

int launch_decode(const DecodeArgs &a, int dtype, hipStream_t stream, CopyManyArgs *fed, int n_fed) {
  // (the matrix-core kernel deals its (b, kv head slice, chunk) units in 32-bit arithmetic)
  const int64_t mfma_units = (int64_t)a.B * a.Hkv * ((a.Hq / a.Hkv + 15) / 16) * a.num_splits;
  if (decode_mfma_takes(a, dtype) && mfma_units < (int64_t(1) << 31)) {
    if (plan_only("decode_%s_kernel<%s, D=%d> splits=%d", a.num_splits == 1 && (a.step || decode_by_pairs(a)) ? "pair" : "mfma", dtype == LMH_F16 ? F16::kName : BF16::kName, a.D,
                  a.num_splits))
      return LMH_OK;
    const int n_copies = n_fed ? (int)number_copy_blocks(*fed, n_fed) : 0;
    const int rc = launch_decode_mfma_split(a, dtype, stream, fed, n_copies);
    if (rc != LMH_OK || a.num_splits == 1) return rc;
    return dtype == LMH_F16 ? launch_merge<F16>(a, stream, fed, n_copies) : launch_merge<BF16>(a, stream, fed, n_copies);
  }
  if (a.step) return fail(LMH_E_UNSUPPORTED, "decode step: only the matrix-core decode kernel rotates q as it loads it");
  switch (dtype) {
    case LMH_F32: return launch_for_dtype<F32>(a, stream);
    case LMH_F16: return launch_for_dtype<F16>(a, stream);
    case LMH_BF16: return launch_for_dtype<BF16>(a, stream);
  }
  return fail(LMH_E_UNSUPPORTED, "decode attention: unknown dtype %d", dtype);
}

}  // namespace lmh
