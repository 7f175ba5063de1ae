// Copies of several ranges by the workgroups of one launch (map_ops.hip), or by extra workgroups of a launch that runs anyway
// (the append and merge kernels of a compiled graph's first step).
#pragma once

#include "common.hpp"

namespace lmh {

constexpr int kCopyChunk = 16384;  // bytes per workgroup

// Workgroup `block` of those that number_copy_blocks has numbered.
template <int THREADS>
__device__ inline void copy_block(const CopyManyArgs &a, int block) {
  int j = 0;
#pragma unroll
  for (int i = 1; i < kCopyMany; i++)
    if (block >= a.first_block[i]) j = i;
  const int64_t begin = (int64_t)(block - a.first_block[j]) * kCopyChunk;
  const int64_t end = min(begin + kCopyChunk, a.bytes[j]);
  char *dst = reinterpret_cast<char *>(a.dst[j]);
  const char *src = reinterpret_cast<const char *>(a.src[j]);
  if (((reinterpret_cast<uintptr_t>(dst) | reinterpret_cast<uintptr_t>(src)) & 15) == 0) {
    const int64_t whole = end & ~(int64_t)15;
    constexpr int N = kCopyChunk / (THREADS * 16);
    uint4 v[N];  // all loads before the first store: the two ranges do not meet, which the compiler cannot know
#pragma unroll
    for (int r = 0; r < N; r++) {
      const int64_t i = begin + (r * THREADS + threadIdx.x) * 16;
      v[r] = i < whole ? *reinterpret_cast<const uint4 *>(src + i) : make_uint4(0, 0, 0, 0);  // (left unset, v goes to LDS)
    }
#pragma unroll
    for (int r = 0; r < N; r++) {
      const int64_t i = begin + (r * THREADS + threadIdx.x) * 16;
      if (i < whole) *reinterpret_cast<uint4 *>(dst + i) = v[r];
    }
    const int64_t i = max(whole, begin) + threadIdx.x;
    if (i < end) dst[i] = src[i];
  } else {
    for (int64_t i = begin + threadIdx.x; i < end; i += THREADS) dst[i] = src[i];
  }
}

// `bytes`, a multiple of 16 and N 16-byte accesses of THREADS threads at most, at 16-byte aligned addresses. `wave` is uniform; the
// lane is asked for here, so that no register holds the thread's number until then.
template <int THREADS, int N>
__device__ inline void copy_span(void *dst, const void *src, int bytes, int wave) {
  const int tid = wave * 64 + __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0));
  uint4 v[N];
#pragma unroll
  for (int r = 0; r < N; r++) {
    const int i = (r * THREADS + tid) * 16;
    v[r] = i < bytes ? *reinterpret_cast<const uint4 *>(reinterpret_cast<const char *>(src) + i) : make_uint4(0, 0, 0, 0);
  }
#pragma unroll
  for (int r = 0; r < N; r++) {
    const int i = (r * THREADS + tid) * 16;
    if (i < bytes) *reinterpret_cast<uint4 *>(reinterpret_cast<char *>(dst) + i) = v[r];
  }
}

// Numbers the workgroups of the first n ranges: how many there are, or -1 where they are too many.
inline int64_t number_copy_blocks(CopyManyArgs &a, int n) {
  int64_t blocks = 0;
  for (int i = 0; i < kCopyMany; i++) {
    a.first_block[i] = (int32_t)blocks;
    if (i < n) blocks += (a.bytes[i] + kCopyChunk - 1) / kCopyChunk;
    if (blocks >= (int64_t(1) << 31)) return -1;
  }
  return blocks;
}

}  // namespace lmh
