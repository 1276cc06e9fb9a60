// Integer arithmetic of the attention kernels' work lists, on the host and on the device (and in plain C++).
#ifndef SDV2KV_ATTN_TILES_H
#define SDV2KV_ATTN_TILES_H

#include <stdint.h>

#ifdef __HIPCC__
#define SDV2_BOTH __host__ __device__ __forceinline__
#else
#define SDV2_BOTH inline
#endif

namespace sdv2 {
namespace attn {

// Division of a number below 2^31 by a launch constant without a division: the
// work list is decoded by every workgroup before it can ask for its first tile,
// and six integer divisions are a microsecond on the way there.
struct FastDiv {
  uint32_t mul, shift;
  static FastDiv by(uint32_t d) {
    FastDiv f{1, 0};
    while ((1ull << f.shift) < d) ++f.shift;
    f.mul = (uint32_t)(((1ull << 32) * ((1ull << f.shift) - d)) / d + 1);
    return f;
  }
  SDV2_BOTH int operator()(int n) const {
    const uint32_t high = (uint32_t)(((uint64_t)(uint32_t)n * mul) >> 32);
    return (int)((high + (uint32_t)n) >> shift);
  }
};

// Tiles of `tile` keys that the queries up to q_last have to see of `seq` keys, where the chunk's own keys start at
// chunk_start and are hidden block by block (block = 0: not at all).  Entries [hole, hole + skipped) of all tiles
// hold nothing but keys that are hidden from q_last, and so from every query before it.
struct TileSpan {
  int count, hole, skipped;
};
SDV2_BOTH TileSpan visible_tiles(int tile, int seq, int q_last, int q_tokens, int chunk_start, int block, FastDiv div_block) {
  TileSpan t{(seq + tile - 1) / tile, 0x7fffffff, 0};
  if (block > 0) {
    const int lo = chunk_start + (div_block(q_last) + 1) * block, hi = chunk_start + q_tokens;
    const int h0 = (lo + tile - 1) / tile, h1 = hi >= seq ? t.count : hi / tile;
    if (h1 > h0) {
      t.hole = h0;
      t.skipped = h1 - h0;
      t.count -= t.skipped;
    }
  }
  return t;
}

}  // namespace attn
}  // namespace sdv2

#endif  // SDV2KV_ATTN_TILES_H
