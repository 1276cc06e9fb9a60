// Equal shares of a call's key tiles for a fixed number of workgroups: the integer
// arithmetic of swa_attn_fwd_even.hip, on the host and on the device (and in a plain
// C++ test of it).
#ifndef SDV2KV_ATTN_EVEN_PLAN_H
#define SDV2KV_ATTN_EVEN_PLAN_H

#include <stdint.h>

#include "attn_tiles.h"

namespace sdv2 {
namespace attn {

// The work is a row of items: the whole 256-row query tiles of all (row, head) pairs, pairs slowest, and behind them the
// rows past the last whole tile, one item for each pair.  First every workgroup takes an equal number of items whole
// (`rounds`, neighbours side by side: they stream the same keys at the same time).  What is left is cut into equal
// shares.  An item is as long as its key tiles take, in sixteenths of what a whole query tile's take, plus a start and
// end in front: a workgroup that begins with the rest of an item has paid one such start, as all have, and pays
// another for each item that begins in its share.  Workgroup w takes units [w * share, (w + 1) * share) of what is left.
struct ItemKind {
  int32_t start, per_tile;
  SDV2_BOTH int units(int tiles) const { return start + per_tile * tiles; }
  // first tile of an item that lies at or past `units` from the item's start
  SDV2_BOTH int tile_at(int units, int tiles) const {
    const int past = units - start + per_tile / 2;
    const int t = past < 0 ? 0 : (int)((uint32_t)past / (uint32_t)per_tile);
    return t < tiles ? t : tiles;
  }
};
constexpr ItemKind kWholeTile{80, 16};
// The rows past the last whole tile, in blocks of 32 (one per wave).  One block is work of its own kind (the waves share
// its queries); up to four are a query tile with one wave at work on a SIMD, and take four fifths of the time; a tile
// with more counts as whole.
constexpr ItemKind kOneBlock{64, 8}, kFewBlocks{80, 13};
constexpr int kMostRestBlocks = 4;
SDV2_BOTH ItemKind rest_kind(int blocks) { return blocks == 1 ? kOneBlock : kFewBlocks; }

struct EvenPlan {
  int32_t workgroups, rounds;            // a multiple of 8; items that each takes whole
  int32_t pairs, whole_tiles, rest_blocks;       // (row, head) pairs; query tiles and further 32-row blocks of each
  int32_t tiles;                         // key tiles of an item ...
  int32_t shortened;                     // ... unless the mask inside the chunk shortens them, in all rows alike (no rounds then)
  int32_t whole_units, rest_units;       // units of all whole tiles past the rounds; of one pair's rest
  int32_t pair_units;                    // shortened: units of a pair's whole tiles
  int32_t total, share;                  // units of all that is cut; of a share
  FastDiv div_share, div_whole, div_rest, div_tiles;     // by share; by the units of a whole tile (shortened: of a pair's);
                                                         // by rest_units; by whole_tiles
};
// The workgroups with a tile of the item that starts at `off`: a border between two shares is half a tile off at most,
// so a share holds a tile when it reaches half of one past the item's start, and begins half of one before its end.
SDV2_BOTH int first_workgroup(FastDiv div_share, ItemKind kind, int off) {
  return div_share(off + kind.start + kind.per_tile - kind.per_tile / 2 - 1);
}
SDV2_BOTH int last_workgroup(FastDiv div_share, ItemKind kind, int off, int tiles) {
  return div_share(off + kind.units(tiles) - kind.per_tile / 2 - 1);
}

// Key tiles of a pair's item: of 64 keys, as many as its last query sees.
SDV2_BOTH int item_tiles(int seq, int item, bool one_block, int q_tokens, int chunk_start, int block, FastDiv div_block) {
  const int past = item * 256 + 256, q_last = (past < q_tokens ? past : q_tokens) - 1;
  // (the waves of a block go by 32 keys)
  const int tile = one_block ? 32 : 64, count = visible_tiles(tile, seq, q_last, q_tokens, chunk_start, block, div_block).count;
  return one_block ? (count + 1) / 2 : count;
}

}  // namespace attn
}  // namespace sdv2

#endif  // SDV2KV_ATTN_EVEN_PLAN_H
