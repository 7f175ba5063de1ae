// How a flash attention launch deals its work to workgroups: plain integer code for host and device.
#pragma once

#include <stdint.h>

namespace lmh {

// Quotients by launch constants as a multiplication, exact for every n < 2^31 and 0 < d < 2^31: with 2^(l-1) < d <= 2^l and
// m = floor(2^(31+l) / d) + 1 the product n m / 2^(31+l) exceeds n / d by less than 1 / d (Granlund and Montgomery, "Division
// by Invariant Integers using Multiplication"). (The device's own integer division is forty instructions through a
// floating-point reciprocal, and two of them stood in front of every workgroup's first load.)
struct FastDiv {
  uint32_t m, s;
};
inline FastDiv fast_div(uint32_t d) {
  const uint32_t l = d > 1 ? 32 - __builtin_clz(d - 1) : 0;
  return {(uint32_t)((uint64_t(1) << (31 + l)) / d + 1), l};
}
__host__ __device__ inline uint32_t operator/(uint32_t n, FastDiv f) { return (uint32_t)(((uint64_t)(2 * n) * f.m) >> 32) >> f.s; }

// How a flash attention launch deals its (b, hq) pairs ("heads") and their query tiles to workgroups.
struct Deal {
  int32_t heads, tiles;
  int32_t snake;                // CUs of an XCD, or 0
  FastDiv whole, all, hq, cus;  // divisors heads / 8 (1 if there are fewer), heads, Hq, `snake`
};

// Which (b, hq) and which of its tiles the i-th workgroup of XCD x takes (workgroup blockIdx.x goes to XCD blockIdx.x % 8).
// Whole heads go to one XCD each, eight at a time, so that a head's K and V stay in one L2; the tiles of the heads % 8 heads
// that are left go round the XCDs one by one. (As heads of their own they would leave most of the chip idle: one head of
// B = 1 Hq = 1 would run on 32 of 256 CUs.) Tiles come in the order of their rank, all heads' rank r before any head's rank
// r + 1; causal launches make the heaviest tile rank 0. Where all workgroups of such a launch are resident at once, nothing
// balances them afterwards: a CU keeps the ones it was dealt, the same place of every round of the XCD's CUs. Those launches
// deal every other round in the opposite order (`snake`), so that the heaviest shares its CU with the lightest.
// False: there is no such workgroup.
__host__ __device__ inline bool deal_tile(const Deal &t, int x, int i, int n_per_xcd, int *head, int *rank) {
  if (t.snake) {
    const int round = (int)((uint32_t)i / t.cus);
    if (round & 1) {
      const int first = round * t.snake, end = first + t.snake < n_per_xcd ? first + t.snake : n_per_xcd;
      i = first + end - 1 - i;
    }
  }
  const int whole = t.heads >> 3, left = t.heads & 7;
  if (left == 0) {
    const int r = (int)((uint32_t)i / t.whole);
    *rank = r;
    *head = (i - r * whole) * 8 + x;
    return r < t.tiles;
  }
  // before rank r, XCD x takes r tiles of each of its whole heads and those e < r * left with e % 8 == x of the others
  auto before = [&](int r) { return whole * r + ((left * r - x + 7) >> 3); };
  int r = (int)((8u * (uint32_t)i) / t.all);
  while (before(r) > i) r--;
  while (before(r + 1) <= i) r++;
  const int k = i - before(r);
  *rank = r;
  const int e0 = r * left;
  *head = k < whole ? k * 8 + x : whole * 8 + ((x - e0) & 7) + 8 * (k - whole);
  return r < t.tiles;
}
// The same head by head, for launches of one round whose order does not matter. n_whole = heads / 8 * tiles.
__host__ __device__ inline bool deal_tile_by_head(int heads, int tiles, int n_whole, int x, int i, int *head, int *rank) {
  if (i < n_whole) {
    const int h = i / tiles;
    *rank = i - h * tiles;
    *head = h * 8 + x;
    return true;
  }
  const int e = (i - n_whole) * 8 + x, h = e / tiles;
  *rank = e - h * tiles;
  *head = (heads & ~7) + h;
  return *head < heads;
}
// Workgroups of such a launch. The kernels count them, and eight times a workgroup's place on its XCD, in 31 bits: the
// launchers refuse more (check_grid).
inline int64_t deal_grid(int64_t heads, int64_t tiles) { return 8 * ((heads >> 3) * tiles + ((heads & 7) * tiles + 7) / 8); }

// resident: workgroups that fit a CU (0: no reason to deal backwards). deal_grid(B Hq, tiles) < 2^31.
inline Deal make_deal(int B, int Hq, int tiles, int resident, int n_cus) {
  Deal t;
  t.heads = B * Hq;
  t.tiles = tiles;
  const int64_t grid = deal_grid(t.heads, tiles);
  t.snake = grid > n_cus && grid <= (int64_t)resident * n_cus ? n_cus / 8 : 0;
  t.whole = fast_div(t.heads >= 8 ? t.heads / 8 : 1);
  t.all = fast_div(t.heads);
  t.hq = fast_div(Hq);
  t.cus = fast_div(t.snake ? t.snake : 1);
  return t;
}

}  // namespace lmh
