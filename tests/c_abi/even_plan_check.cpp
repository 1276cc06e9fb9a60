// Brute force over the integer arithmetic of csrc/attn_even_plan.h: every tile of every item belongs to exactly one
// workgroup, first_workgroup / last_workgroup name exactly those that hold one, and no workgroup has two partial
// results for one place.  Prints what is wrong and returns 1, or the number of plans looked at.
#include <stdio.h>
#include <stdlib.h>

#include <vector>

#include "attn_even_plan.h"

using namespace sdv2::attn;

struct Item {
  ItemKind kind;
  int tiles;
};

static int check(const std::vector<Item>& of_pair, int pairs, int workgroups) {
  EvenPlan e{};
  for (const Item& it : of_pair) e.total += pairs * it.kind.units(it.tiles);
  e.share = (e.total + workgroups - 1) / workgroups;
  if (e.share < kWholeTile.units(4)) e.share = kWholeTile.units(4);
  e.div_share = FastDiv::by((uint32_t)e.share);
  std::vector<std::vector<int>> owner;
  for (int p = 0, off = 0; p < pairs; ++p)
    for (const Item& it : of_pair) {
      const int t = it.tiles;
      std::vector<int> of(t, -1);
      for (int w = 0; w < workgroups; ++w) {
        const int begin = w * e.share;
        if (begin >= e.total) break;
        const int end = begin + e.share < e.total ? begin + e.share : e.total;
        for (int i = it.kind.tile_at(begin - off, t); i < it.kind.tile_at(end - off, t); ++i) {
          if (of[i] != -1) return printf("tile %d of item at %d twice\n", i, off), 1;
          of[i] = w;
        }
      }
      for (int i = 0; i < t; ++i)
        if (of[i] < 0 || (i > 0 && of[i] != of[i - 1] && of[i] != of[i - 1] + 1)) return printf("tile %d of item at %d: %d\n", i, off, of[i]), 1;
      const int first = first_workgroup(e.div_share, it.kind, off), last = last_workgroup(e.div_share, it.kind, off, t);
      if (of[0] != first || of[t - 1] != last)
        return printf("item at %d: workgroups %d..%d, said to be %d..%d (share %d, tiles %d)\n", off, of[0], of[t - 1], first, last, e.share, t), 1;
      owner.push_back(of);
      off += it.kind.units(t);
    }
  // a workgroup's places: [0] the rest or the middle of an item, [1] the start of one that others go on with
  std::vector<int> used(2 * workgroups, 0);
  for (const auto& of : owner)
    for (size_t i = 0; i < of.size(); ++i)
      if ((i == 0 || of[i] != of[i - 1]) && of.front() != of.back() && ++used[2 * of[i] + (of[i] == of.front())] > 1)
        return printf("workgroup %d: two results in one place\n", of[i]), 1;
  return 0;
}

int main() {
  srand(1);
  int plans = 0;
  for (int i = 0; i < 3000; ++i) {
    const int whole = rand() % 9, blocks = whole ? rand() % 5 : 1 + rand() % 4, pairs = 1 + rand() % 20, workgroups = 8 * (1 + rand() % 32);
    const int most = 1 + (i % 3 ? rand() % 60 : rand() % 400);
    std::vector<Item> items;
    for (int k = 0; k < whole + (blocks > 0); ++k)     // the mask shortens items
      items.push_back({k < whole ? kWholeTile : rest_kind(blocks), i % 2 ? 1 + rand() % (i % 5 ? most : 3) : most});
    if (check(items, pairs, workgroups)) return 1;
    ++plans;
  }
  for (uint32_t d : {1u, 2u, 3u, 7u, 36u, 37u, 608u, 65535u, 1000003u, 0x3fffffffu})
    for (int64_t n = 0; n < (1ll << 31); n = n * 3 + 1 + rand() % 5)
      for (int64_t m : {n, n / d * d, n / d * d + d - 1})
        if (m < (1ll << 31) && FastDiv::by(d)((int)m) != (int)(m / d)) return printf("%lld / %u\n", (long long)m, d), 1;
  printf("%d plans\n", plans);
  return 0;
}
