// Which tile a product takes (csrc/linear_tiles.h): rows, columns, contraction and sums or not as arguments, four by four; prints
// the tile of each, its rows and columns.
#include <stdio.h>
#include <stdlib.h>

#include "linear_tiles.h"

int main(int argc, char** argv) {
  for (int i = 1; i + 3 < argc; i += 4) {
    const int t = sdv2::linear::best_tile(atoll(argv[i]), atoll(argv[i + 1]), atoll(argv[i + 2]), atoi(argv[i + 3]) != 0);
    printf("%d %d\n", t < 0 ? 0 : sdv2::linear::kTiles[t].m, t < 0 ? 0 : sdv2::linear::kTiles[t].n);
  }
  return 0;
}
