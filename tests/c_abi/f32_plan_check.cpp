// Brute force over the shares of the fp32 attention (EvenPlanF32 in csrc/attn_f32_plan.h): every tile of every item
// belongs to exactly one workgroup, first_workgroup / last_workgroup name exactly those that hold one, and no workgroup
// has two partial results for one place.  Prints what is wrong and returns 1, or the number of plans looked at.
#include <stdio.h>
#include <stdlib.h>

#include <vector>

#include "attn_f32_plan.h"

using namespace sdv2::attn;

static int check(int pairs, int whole_tiles, int rest_blocks, int tiles, int start, int share) {
  const ItemKind whole{start, kWholeTileF32.per_tile};
  const int per_pair = whole_tiles + (rest_blocks > 0);
  const int total = pairs * (whole_tiles * whole.units(tiles) + (rest_blocks ? rest_kind_f32(rest_blocks).units(tiles) : 0));
  const int workgroups = (total + share - 1) / share;
  const FastDiv div_share = FastDiv::by((uint32_t)share);
  std::vector<int> used(2 * workgroups, 0);
  for (int i = 0, off = 0; i < pairs * per_pair; ++i) {
    const ItemKind kind = i % per_pair < whole_tiles ? whole : rest_kind_f32(rest_blocks);
    std::vector<int> of(tiles, -1);
    for (int w = 0; w < workgroups; ++w) {
      const int begin = w * share, end = begin + share < total ? begin + share : total;
      for (int t = kind.tile_at(begin - off, tiles); t < kind.tile_at(end - off, tiles); ++t) {
        if (of[t] != -1) return printf("tile %d of item %d twice\n", t, i), 1;
        of[t] = w;
      }
    }
    for (int t = 0; t < tiles; ++t)
      if (of[t] < 0 || (t > 0 && of[t] != of[t - 1] && of[t] != of[t - 1] + 1)) return printf("tile %d of item %d: %d\n", t, i, of[t]), 1;
    const int first = first_workgroup(div_share, kind, off), last = last_workgroup(div_share, kind, off, tiles);
    if (of[0] != first || of[tiles - 1] != last)
      return printf("item %d: workgroups %d..%d, said to be %d..%d\n", i, of[0], of[tiles - 1], first, last), 1;
    if (first != last)
      for (int w = first; w <= last; ++w)
        if (++used[2 * w + (w == first)] > 1) return printf("workgroup %d: two results in one place\n", w), 1;
    off += kind.units(tiles);
  }
  return 0;
}

int main() {
  srand(1);
  int plans = 0;
  for (int i = 0; i < 2000; ++i, ++plans) {
    const int rest = rand() % 3, whole = rest ? rand() % 9 : 1 + rand() % 9, pairs = 1 + rand() % 20, tiles = 1 + rand() % (i % 3 ? 60 : 400);
    const int units = kWholeTileF32.units(tiles), least = kWholeTileF32.units(4) > units / 16 ? kWholeTileF32.units(4) : units / 16;
    const int share = least + rand() % (3 * units);
    if (check(pairs, whole, rest, tiles, kWholeTileF32.start, share)) return printf("pairs %d whole %d rest %d tiles %d share %d\n", pairs, whole, rest, tiles, share), 1;
    for (int pieces = 2; rest == 0 && pieces <= 16 && tiles / pieces >= 4; ++pieces) {
      const int equal = (16 * tiles + pieces - 1) / pieces;
      if (check(pairs, whole, 0, tiles, equal * pieces - 16 * tiles, equal)) return printf("pairs %d whole %d tiles %d pieces %d\n", pairs, whole, tiles, pieces), 1;
    }
  }
  printf("%d plans\n", plans);
  return 0;
}
