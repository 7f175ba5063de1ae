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

// How a flash attention launch deals its (b, hq) pairs ("heads") and their query tiles to workgroups. The kernels take it in front
// of their other arguments: a workgroup reads its argument block as one batch of scalar loads in the order of the block, and
// waits for all of it. Behind PrefillArgs the same block took launches of less than 10 us 0.1 to 0.2 us longer when the host
// enqueued them one by one (B=1 H=8 S=128 D=64 causal fp16 5.87 us, in front 5.67; B=1 H=32 S=512 8.08 and 7.89; the number of
// words makes no difference, nor does either in a recorded graph).
struct Deal {
  int32_t heads, tiles;
  int32_t n_per_xcd;     // workgroups of an XCD
  int32_t snake;         // CUs of an XCD; more than n_per_xcd where the order of all rounds is the same
  FastDiv all, hq, cus;  // divisors heads, Hq, snake
};

// Which (b, hq) and which of its tiles the i-th workgroup of XCD x takes (workgroup blockIdx.x goes to XCD blockIdx.x % 8).
// Whole heads go to one XCD each, eight at a time, so that a head's K and V stay in one L2; the tiles of the heads % 8 heads
// that are left go round the XCDs one by one. (As heads of their own they would leave most of the chip idle: one head of
// B = 1 Hq = 1 would run on 32 of 256 CUs.) Tiles come in the order of their rank, all heads' rank r before any head's rank
// r + 1; causal launches make the heaviest tile rank 0. Where all workgroups of such a launch are resident at once, nothing
// balances them afterwards: a CU keeps the ones it was dealt, the same place of every round of the XCD's CUs. Those launches
// deal every other round in the opposite order (`snake`), so that the heaviest shares its CU with the lightest.
// All launches take the same few scalar instructions: a workgroup that jumps over the instructions of other cases waits for
// the next ones from memory (1024 workgroups of B=8 H=32 S=256 D=64 causal fp16: 10.2 us with branches, 10.1 without; B=8
// H=32/8 S=512 D=128 causal bf16 40.2 -> 39.8; B=3 H=6 Sq=166 Sk=1333 D=64 fp16 14.1 -> 14.0).
// False: there is no such workgroup.
__host__ __device__ inline bool deal_tile(const Deal &t, int x, int i, int *head, int *rank) {
  const int round = (int)((uint32_t)i / t.cus), first = round * t.snake;
  const int end = first + t.snake < t.n_per_xcd ? first + t.snake : t.n_per_xcd;
  i = (round & 1) ? first + end - 1 - i : i;
  // Before rank r, XCD x takes r tiles of each of its heads / 8 whole heads and those e < r * left of the others with
  // e % 8 == x: (r heads + 7 - x) / 8 tiles in all. That is at most i as long as r heads <= 8 i + x.
  const int whole = t.heads >> 3, left = t.heads & 7;
  const int r = (int)((uint32_t)(8 * i + x) / t.all);
  const int k = i - ((r * t.heads + 7 - x) >> 3);
  *rank = r;
  *head = 8 * k + (k < whole ? x : (x - r * left) & 7);
  return r < t.tiles;
}
// Rows by which the row tiles of a causal launch begin before row 0. Where they do not fill the rows, the rows that a tile lacks
// are those of the first one, whose keys are few, and not of the last one, which walks all of them whether it has one row or
// all: S=777 in tiles of 128 rows is 49 key tiles of 64 a head in place of 55, S=1337 121 in place of 131. The shift is a multiple
// of the key tile (a power of two), so that every tile's diagonal lies where it would without one; rows before row 0 see no key. Where a
// row tile is no higher than a key tile the shift is zero; left out there, the fp16 and bf16 kernels of two key groups took longer: fp16 B=1 H=6 S=2143
// D=128 31.6 -> 32.6 us, H=12 S=1524 24.5 -> 25.1, bf16 H=8 S=1584 28.8 -> 29.1 (B=7 H=8/4 S=1994 D=64 52.4 -> 52.1).
__host__ __device__ inline int causal_shift(int tiles, int rows, int Sq, int key_tile) {
  return (int)(((uint32_t)tiles * (uint32_t)rows - (uint32_t)Sq) & ~(uint32_t)(key_tile - 1));
}
// deal_tile head by head, for launches of one round whose order does not matter. n_whole = heads / 8 * tiles.
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
// Workgroups of such a launch. The kernels count them in 31 bits: the launchers refuse more (check_grid).
inline int64_t deal_grid(int64_t heads, int64_t tiles) { return 8 * ((heads >> 3) * tiles + ((heads & 7) * tiles + 7) / 8); }

// resident: workgroups that fit a CU (0: no reason to deal backwards). deal_grid(B Hq, tiles) < 2^31.
inline Deal make_deal(int B, int Hq, int tiles, int resident, int n_cus) {
  Deal t;
  t.heads = B * Hq;
  t.tiles = tiles;
  const int64_t grid = deal_grid(t.heads, tiles);
  t.n_per_xcd = (int32_t)(grid >> 3);
  t.snake = n_cus >= 8 && grid > n_cus && grid <= (int64_t)resident * n_cus ? n_cus / 8 : t.n_per_xcd + 1;
  t.all = fast_div(t.heads);
  t.hq = fast_div(Hq);
  t.cus = fast_div(t.snake);
  return t;
}

}  // namespace lmh
