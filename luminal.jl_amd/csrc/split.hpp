// fp32 values as three bf16 pieces, for products on the bf16 matrix pipe (matmul.hip, prefill_f32_split.hip): the decomposition
// and the choice of six products of Henry, Tang and Heinecke, "Leveraging the bfloat16 Artificial Intelligence Datatype For
// Higher-Precision Computations" (ARITH 2019).
//
// x = x1 + x2 + x3, each the rest rounded to nearest: 8 bits and a sign a piece hold all 24 bits of x. What they do not hold:
//   * an infinity, a NaN, or a value that rounds up to an infinity: the later pieces are NaN, and so is every sum they enter;
//   * bits below 2^-126, the smallest normal piece. An fp32 value is a multiple of 2^-149: scaled by kPieceScale (which is exact,
//     or overflows into the case above) every one is held, whatever stands beside it. No test by magnitude of the values that
//     arrive can take the place of it: the largest of a row says nothing about a product that the others leave to a small one.
#pragma once

#include "dtypes.hpp"

namespace lmh {

constexpr float kPieceScale = 16777216.f;  // 2^24
constexpr float kPieceUnscale = 1.f / kPieceScale;

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

__device__ inline Pieces split_8(const floatx4_t &lo, const floatx4_t &hi) {
  uint32_t w[3][4];
#pragma unroll
  for (int e = 0; e < 4; e++)
    split_bf16x2(e < 2 ? lo[2 * e] : hi[2 * e - 4], e < 2 ? lo[2 * e + 1] : hi[2 * e - 3], &w[0][e], &w[1][e], &w[2][e]);
  Pieces f;
#pragma unroll
  for (int i = 0; i < 3; i++) f.p[i] = __builtin_bit_cast(bf16x8_t, make_uint4(w[i][0], w[i][1], w[i][2], w[i][3]));
  return f;
}

// x as two fp16 pieces, hi = x and lo = 2^11 (x - hi), each rounded to nearest: x = hi + lo / 2^11 to 2^-23 of itself, or to 2^-36 where
// that is more; |x| < 2^16 (above it hi is an infinity).
struct HalfPieces {
  half8_t hi, lo;
};
constexpr float kHalfGap = 2048.f;
// Values whose largest is `top`, in [2^14, 2^15) at its exponent: times half_up, and what comes of them times half_down. What is all below 2^-30 is
// left smaller. Infinities stay infinite.
constexpr int kHalfLeast = 97;  // biased exponent of 2^-30
__device__ inline int half_exponent(float top) { return max((int)(__float_as_uint(top) >> 23), kHalfLeast); }
__device__ inline float half_up(int exponent) { return __uint_as_float((uint32_t)(268 - exponent) << 23); }
__device__ inline float half_down(int exponent) { return __uint_as_float((uint32_t)(exponent - 14) << 23); }

__device__ inline uint32_t round_half2(float a, float b) {
  typedef _Float16 h2 __attribute__((ext_vector_type(2)));
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){a, b}, h2));
}

// `hi` and `lo` of a value, given what is rounded to hi and, from that, 2^11 times the rest.
template <class High, class Low>
__device__ inline HalfPieces split_half_8(const floatx4_t &x0, const floatx4_t &x1, const High &high, const Low &low) {
  typedef _Float16 h2 __attribute__((ext_vector_type(2)));
  uint32_t hi[4], lo[4];
#pragma unroll
  for (int e = 0; e < 4; e++) {
    const float a = e < 2 ? x0[2 * e] : x1[2 * e - 4], b = e < 2 ? x0[2 * e + 1] : x1[2 * e - 3];
    hi[e] = round_half2(high(a), high(b));
    const h2 h = __builtin_bit_cast(h2, hi[e]);
    lo[e] = round_half2(low(a, (float)h[0]), low(b, (float)h[1]));
  }
  return {__builtin_bit_cast(half8_t, make_uint4(hi[0], hi[1], hi[2], hi[3])), __builtin_bit_cast(half8_t, make_uint4(lo[0], lo[1], lo[2], lo[3]))};
}
// x times a power of two.
__device__ inline HalfPieces split_half_8(const floatx4_t &x0, const floatx4_t &x1, float up) {
  return split_half_8(x0, x1, [=](float x) { return x * up; }, [=](float x, float h) { return fmaf(h, -kHalfGap, x * (up * kHalfGap)); });
}
// The same of x (by + rest): hi is the rounded product, and what the rounding leaves of the exact one goes to lo.
__device__ inline HalfPieces split_half_8(const floatx4_t &x0, const floatx4_t &x1, float by, float rest) {
  return split_half_8(x0, x1, [=](float x) { return x * by; }, [=](float x, float h) { return fmaf(x, rest, fmaf(x, by, -h)) * kHalfGap; });
}

}  // namespace lmh
