// The tiles of sdv2_linear and which of them a product takes, in plain C++.
#ifndef SDV2KV_LINEAR_TILES_H
#define SDV2KV_LINEAR_TILES_H

#include <stdint.h>

namespace sdv2 {
namespace linear {

constexpr int kDepth = 64;                   // of a stage, along the contraction

// The tiles there are.  us: what a stage of 64 takes by itself, beside what it brings (tile_us).
struct Tile {
  int m, n;
  float us;
};
constexpr Tile kTiles[] = {{64, 64, 0.073f},   {96, 64, 0.073f},   {160, 64, 0.091f},  {96, 128, 0.102f},  {128, 128, 0.121f},
                           {160, 128, 0.138f}, {192, 128, 0.150f}, {224, 128, 0.163f}, {256, 128, 0.187f}, {224, 160, 0.225f}};
constexpr int kTileCount = sizeof(kTiles) / sizeof(kTiles[0]);
constexpr int kCus = 256;

inline int64_t tiles_of(const Tile& t, int64_t m, int64_t n) { return (m + t.m - 1) / t.m * (n / t.n); }

// What a stage brings counts, 14 ns a kilobyte, and only rows there are do (those past the last repeat it): the mean of the
// row tiles.  A row tile with few of them goes ahead of the others and brings the weights to L2 for them, up to 11 ns for
// every kilobyte that the fullest has more than the mean, where the contraction is long.  Of 1447 products in every tile that
// is one round, weights cold, in graphs, 97 to 7020 rows of 4 to 64 heads, the one this picks takes 1.009 of the best one's
// time, 38 more than 1.1, 1.27 at worst.  Without the last two (a stage's time by its tile and the number of tiles) it was
// 1.022, 126 and 1.42: 352 x 4352 x 4352 37.3 -> 27.3 us, 359 x 5120 x 5120 46.7 -> 33.0, 508 x 6144 x 6144 62.5 -> 53.1.
inline double tile_us(const Tile& t, int64_t m, int64_t n, int64_t k) {
  const int64_t row_tiles = (m + t.m - 1) / t.m, rounds = (tiles_of(t, m, n) + kCus - 1) / kCus;
  const double stages = (double)k / kDepth, kilobyte = 2 * kDepth / 1000.0, rows = (double)m / (double)row_tiles;
  const double longer = stages < 24 ? 0 : stages < 80 ? (stages - 24) / 56 : 1, more = (m < t.m ? m : t.m) - rows;
  return (double)rounds * (0.5 + stages * (t.us + kilobyte * (0.0139 * (rows + t.n) - 0.0106 * longer * more)));
}

// The tile that takes least, or -1 where none divides n.
inline int best_tile(int64_t m, int64_t n, int64_t k, bool squares) {
  int best = -1;
  double best_us = 0;
  for (int i = 0; i < kTileCount; ++i) {
    if (n % kTiles[i].n != 0 || (squares && kTiles[i].n == 160)) continue;        // (80 columns of a wave are no groups of 32)
    const double us = tile_us(kTiles[i], m, n, k);
    if (best < 0 || us < best_us) {
      best = i;
      best_us = us;
    }
  }
  return best;
}

}  // namespace linear
}  // namespace sdv2

#endif  // SDV2KV_LINEAR_TILES_H
