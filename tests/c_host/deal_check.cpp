// Host build of the kernels' work distribution (csrc/deal.hpp): every (head, tile) exactly once, whatever their number.
// Input lines: "B Hq tiles resident cus" deals a launch; "divide d" compares quotients by d. One "ok" or "wrong ..." a line.
#define __host__
#define __device__
#include "../../luminal.jl_amd/csrc/deal.hpp"

#include <stdio.h>
#include <string.h>

#include <vector>

using namespace lmh;

static void launch(int B, int Hq, int tiles, int resident, int cus) {
  const Deal t = make_deal(B, Hq, tiles, resident, cus);
  const int64_t heads = (int64_t)B * Hq, grid = deal_grid(heads, tiles);
  std::vector<uint8_t> seen(heads * tiles, 0), by_head(heads * tiles, 0);
  int64_t out = 0, twice = 0, split = 0, moved = 0, missing = 0;
  for (int64_t bid = 0; bid < grid; bid++) {
    int head = -1, rank = -1;
    if (deal_tile(t, (int)(bid & 7), (int)(bid >> 3), &head, &rank)) {
      if (head < 0 || head >= heads || rank < 0 || rank >= tiles) out++;
      else if (seen[(int64_t)head * tiles + rank]++) twice++;
      else if ((int)((uint32_t)head / t.hq) != head / Hq) split++;
      else if (head < (heads & ~7) && (head & 7) != (bid & 7)) moved++;
    }
    if (deal_tile_by_head((int)heads, tiles, (int)(heads / 8 * tiles), (int)(bid & 7), (int)(bid >> 3), &head, &rank)) {
      if (head < 0 || head >= heads || rank < 0 || rank >= tiles) out++;
      else if (by_head[(int64_t)head * tiles + rank]++) twice++;
    }
  }
  for (auto *v : {&seen, &by_head})
    for (uint8_t x : *v) missing += x == 0;
  if (out || twice || split || moved || missing)
    printf("wrong B=%d Hq=%d tiles=%d: %lld out of range, %lld twice, %lld missing, %lld of the wrong sequence, %lld on the wrong XCD\n", B, Hq, tiles,
           (long long)out, (long long)twice, (long long)missing, (long long)split, (long long)moved);
  else printf("ok\n");
}

static void divide(uint32_t d) {
  const FastDiv f = fast_div(d);
  const uint32_t top = 0x7fffffffu;
  auto right = [&](uint32_t n) { return n / f == n / d; };
  bool ok = right(0) && right(top) && right(top - 1);
  for (uint32_t i = 0; i < 200000 && ok; i++) {
    const uint32_t q = (uint32_t)((uint64_t)i * (top / d) / 199999);  // multiples of d over the whole range, and their neighbours
    const uint32_t n = q * d;
    ok = right(n) && (n == 0 || right(n - 1)) && (n == top || right(n + 1));
  }
  printf(ok ? "ok\n" : "wrong quotients by %u\n", d);
}

int main() {
  char line[256];
  while (fgets(line, sizeof line, stdin)) {
    int v[5];
    unsigned d;
    if (sscanf(line, "divide %u", &d) == 1) divide(d);
    else if (sscanf(line, "%d %d %d %d %d", v, v + 1, v + 2, v + 3, v + 4) == 5) launch(v[0], v[1], v[2], v[3], v[4]);
  }
  return 0;
}
