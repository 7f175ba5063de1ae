// fp32 values as three bf16 pieces, for products on the bf16 matrix pipe (matmul.hip, prefill_f32_split.hip).
//
// x = x1 + x2 + x3, each the rest rounded to nearest: 8 bits and a sign a piece hold all 24 bits of x. What they do not hold:
//   * an infinity, a NaN, or a value that rounds up to an infinity: the later pieces are NaN, and so is every sum they enter;
//   * values below 2^-110: pieces below 2^-126 lose bits. Rows whose largest value is at least 2^-95 do not notice (2^-39 of it),
//     others are told by the bits of their first pieces.
#pragma once

#include "dtypes.hpp"

namespace lmh {

struct Pieces {
  bf16x8_t p[3];
};

__device__ inline void split_bf16x2(float a, float b, uint32_t *p1, uint32_t *p2, uint32_t *p3) {
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  auto round2 = [](float x, float y) { return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){x, y}, bf16x2)); };
  const uint32_t h1 = round2(a, b);
  const float ra = a - __uint_as_float(h1 << 16), rb = b - __uint_as_float(h1 & 0xffff0000u);
  const uint32_t h2 = round2(ra, rb);
  *p1 = h1;
  *p2 = h2;
  *p3 = round2(ra - __uint_as_float(h2 << 16), rb - __uint_as_float(h2 & 0xffff0000u));
}

// Eight values; their first pieces are or-ed into `bits`.
__device__ inline Pieces split_8(const floatx4_t &lo, const floatx4_t &hi, uint32_t *bits) {
  uint32_t w[3][4];
#pragma unroll
  for (int e = 0; e < 4; e++)
    split_bf16x2(e < 2 ? lo[2 * e] : hi[2 * e - 4], e < 2 ? lo[2 * e + 1] : hi[2 * e - 3], &w[0][e], &w[1][e], &w[2][e]);
  *bits |= w[0][0] | w[0][1];
  *bits |= w[0][2] | w[0][3];
  Pieces f;
#pragma unroll
  for (int i = 0; i < 3; i++) f.p[i] = __builtin_bit_cast(bf16x8_t, make_uint4(w[i][0], w[i][1], w[i][2], w[i][3]));
  return f;
}

// One of the or-ed values is at least 2^-95 (an exponent of 32 or more), or all are zero.
__device__ inline bool pieces_hold(uint32_t bits) { return (bits & 0x70007000u) != 0 || (bits & 0x7fff7fffu) == 0; }

}  // namespace lmh
