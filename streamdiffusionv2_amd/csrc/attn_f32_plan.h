// Shares of a call's key tiles in the fp32 attention (swa_attn_fwd_f32.hip): integer arithmetic on the host and on the
// device (and in a plain C++ test of it).
#ifndef SDV2KV_ATTN_F32_PLAN_H
#define SDV2KV_ATTN_F32_PLAN_H

#include <stdint.h>

#include "attn_even_plan.h"

namespace sdv2 {
namespace attn {

// Items are 128 rows by tiles of 32 keys, and one or two blocks past the last whole 128 rows, whose keys the four waves
// deal out among themselves, at more than their share of a tile's time: they read memory as they go.  The items of a
// (row, head) lie side by side, the rest behind the whole ones, so that the rests are spread over the XCDs (all of them
// at the end: 2 x 821 x 40 queries against 13331 keys 3867 us instead of 3720).  Measured: one block as 5 / 6 / 8
// sixteenths of a tile 508 / 503 / 518 us (780 x 40 against 4000 keys), two as 9 / 11 / 14 772 / 683 / 697 (3 x 960 x 12
// against 5000).
constexpr ItemKind kWholeTileF32{16, 16}, kOneBlockF32{32, 6}, kTwoBlocksF32{32, 11};
constexpr int kMostRestBlocksF32 = 2;
SDV2_BOTH ItemKind rest_kind_f32(int blocks) { return blocks == 1 ? kOneBlockF32 : kTwoBlocksF32; }

struct EvenPlanF32 {
  int32_t workgroups;                            // a multiple of 8
  int32_t pairs, whole_tiles, rest_blocks, tiles;        // whole query tiles and further blocks of a pair; key tiles
  int32_t whole_start;                           // of a whole query tile: kWholeTileF32's or a little more
  int32_t whole_units, rest_units, pair_units, total, share;     // share = 0: one item for each workgroup
  FastDiv div_share, div_whole, div_pair;
};

}  // namespace attn
}  // namespace sdv2

#endif  // SDV2KV_ATTN_F32_PLAN_H
