// out = x W^T + bias in bf16 for gfx950 (MI355X): the projections around the
// attention (models/wan/causal_model.py:212-218, :389; wan_base/modules/model.py:181,
// :195) at the sizes of a chunk, where the vendor library's kernels leave the chip
// idle.  fp32 accumulation in the order of the contraction, 32 products at a time, one
// rounding after the bias; at every size tried the bits of the vendor library's.
//
// What bounds it: a chunk's projection is one round of workgroups, 24 steps of 64
// along a contraction of 1536.  A workgroup is four waves that multiply, one per
// SIMD, and four that fetch.  A wave's products need its LDS reads and LDS takes
// what the transfers bring, so the split of a tile over the waves decides: 2 x 2 waves
// of 80 x 64 read 9 fragments for 20 products (LDS busy 432 of 320 matrix cycles,
// the transfers' writes included).  Fetching is the work of waves of its own because a
// wave that waits for room in the memory pipe issues no products: with the transfers
// dealt out between the products of four waves 160 x 128 tiles took 15 us for what
// the products alone take 8.8 and the transfers alone 7.6; with waves for each, 10.
//
// In a stream the weights come from memory, a trip longer than the stages in
// flight: as many as LDS holds (seven of 96 x 64 instead of four: 512 x 1536 15.0 ->
// 13.1 us).  Bringing lines to L2 ahead of that, by the waves that multiply, costs
// more than it gives: 64 rows are 64 lines to ask for (736 x 5120 x 5120 51 -> 65 us).
//
// With x and the weights in L2 a workgroup alone runs its matrix pipe 76 to 87 % full (a stage of 128 x 128
// 0.28 us, of 224 x 128 0.43); on all CUs the same stages take 0.4 and 0.65, 1.2 and 1.4 PFLOP/s, what a
// large product reaches on the board's power.  (What a stage takes with weights that come from memory:
// linear_tiles.h.)  So what counts is one round of workgroups,
// whatever the tile that takes, and the larger the tile the less energy: 224 x 128 and
// 224 x 160 where 160 x 128 would be two rounds (linear_wide.hip), 1560 x 4608 x 1536 31.6
// -> 24.3 us, 3648 x 1536 x 1536 25.6 -> 20.8, 1560 x 5120 x 5120 117 -> 73.
//
// The vendor's and this one, weights cold: 3120 x 1536 x 1536 24.5 -> 18.6 us, 1560 x 1536 x 1536
// 17.6 -> 13.4, 1560 x 4608 x 1536 28.3 -> 24.3, 528 x 3712 x 3712 32.6 -> 23.4, 256 x 5120 x 5120
// 49.7 -> 30.5.
//
// Stages of 64 along the contraction lie in LDS as rows of 128 bytes (x's rows, then
// W's), 16-byte chunk c of row r at c ^ r % 8: 16 rows of one chunk are read without
// a bank conflict.  kStages of them are in use at a time.  Output: W's rows are the A operand, so a
// lane ends up with four neighbouring columns of a row; each wave turns its part
// through LDS and writes whole lines.
#include "linear_kernel.h"
#include "linear_tiles.h"

extern "C" int sdv2_linear_one_round(int64_t m, int32_t n, int32_t k, int32_t row_squares) {
  if (m <= 0 || n <= 0 || k <= 0 || n % 64 != 0 || k % kDepth != 0) return 0;
  // One round of tiles, of which each CU has one.  1441 such products of 97 to 7020 rows, 4 to 64 heads (q, k and v in one among
  // them), weights cold, in graphs: contractions of up to 2048 take 0.77 of the vendor's time on the geometric mean, 2 of 549
  // are slower by more than 2 %; longer ones 0.88 (1560 x 5120 x 5120 72.8 and 88.7 us, 352 x 4352 x 4352 27.3 and 34.1), 58 of
  // 892 are slower by more than 2 %, 6 of those by more than 10.  These lie at 97 to 960 rows in 64-column or 96-row tiles whose
  // row tiles are full, so that none goes ahead (464 x 3840 x 3840 34.6 and 29.2 us, 496 rows 26.1 and 30.9): with whatever
  // tile is best 37 would stay, and a line that leaves them out loses as much on their neighbours (of contractions past 3000 in
  // tiles of 160 x 64 and 96 x 128, 96 % full, 14 of 28 are the slower ones, 1.016 together).  A second round costs a launch's
  // start and end again and leaves CUs idle: 480 tiles 1.1 to 1.23 of the vendor's time.
  // Of few rows and a long contraction the vendor's cuts the contraction (16 x 5120 x 5120 14.9 against 22.1 us, 64 x 5120 x
  // 5120 21.3 and 29.6, 64 x 7680 x 2560 15.6 and 17.6; the other way round 100 x 5120 x 5120, 27.5 and 25.7, and 100 x 3712 x
  // 3712, 18.8 and 17.4).
  if (m <= 96 && k > 2048) return 0;
  const int i = best_tile(m, n, k, row_squares != 0);
  return i >= 0 && tiles_of(kTiles[i], m, n) <= kCus;
}

extern "C" int sdv2_linear_preferred(int64_t m, int32_t n, int32_t k) {
  // The narrower answer that callers of the first tiles were given: widths up to 16 heads, tiles of up to 160 x 128.
  constexpr int kMostK = 2048, kMostRows = 160, kMostColumns = 128;
  if (k > kMostK || !sdv2_linear_one_round(m, n, k, 0)) return 0;
  for (const Tile& t : kTiles)
    if (t.m <= kMostRows && t.n <= kMostColumns && n % t.n == 0 && tiles_of(t, m, n) <= kCus) return 1;
  return 0;
}

extern "C" int sdv2_linear(const sdv2_linear_params* p) {
  if (!p) return SDV2_ERR_INVALID_ARG;
  if (p->dtype != SDV2_BF16 || p->n <= 0 || p->k <= 0 || p->n % 64 != 0 || p->k % kDepth != 0) return SDV2_ERR_UNSUPPORTED;
  if (p->m < 0) return SDV2_ERR_INVALID_ARG;
  if (p->m == 0) return SDV2_OK;
  if (!p->x || !p->weight || !p->out) return SDV2_ERR_INVALID_ARG;
  if ((reinterpret_cast<uintptr_t>(p->x) | reinterpret_cast<uintptr_t>(p->weight) | reinterpret_cast<uintptr_t>(p->out)) & 15)
    return SDV2_ERR_INVALID_ARG;
  if ((reinterpret_cast<uintptr_t>(p->bias) & 7) || (reinterpret_cast<uintptr_t>(p->row_squares) & 3)) return SDV2_ERR_INVALID_ARG;
  // rows of 16-byte vectors that do not overlap; offsets within a tile's rows are 32-bit
  constexpr int64_t kMostStride = 1 << 22;
  for (int64_t st : {p->x_row_stride, p->weight_row_stride})
    if (st < p->k || st % 8 != 0 || st > kMostStride) return SDV2_ERR_INVALID_ARG;
  if (p->out_row_stride < p->n || p->out_row_stride % 8 != 0) return SDV2_ERR_INVALID_ARG;
  const int i = best_tile(p->m, p->n, p->k, p->row_squares != nullptr);
  if (p->m > 0x7fffffff - 256 || tiles_of(kTiles[i], p->m, p->n) > (1 << 22)) return SDV2_ERR_UNSUPPORTED;
  LinearArgs a;
  a.x = static_cast<const uint16_t*>(p->x);
  a.w = static_cast<const uint16_t*>(p->weight);
  a.bias = static_cast<const uint16_t*>(p->bias);
  a.out = static_cast<uint16_t*>(p->out);
  a.x_st = p->x_row_stride;
  a.w_st = p->weight_row_stride;
  a.out_st = p->out_row_stride;
  a.m = (int32_t)p->m;
  a.squares = p->row_squares;
  a.square_groups = p->n / 32;
  a.stages = p->k / kDepth;
  a.row_tiles = (int32_t)((p->m + kTiles[i].m - 1) / kTiles[i].m);
  a.col_tiles = p->n / kTiles[i].n;
  hipStream_t stream = static_cast<hipStream_t>(p->stream);
  switch (i) {
    case 0: return launch<2, 2, 9>(a, stream);
    case 1: return launch<3, 2, 7>(a, stream);
    case 2: return launch<5, 2, 5>(a, stream);
    case 3: return launch<3, 4, 5>(a, stream);
    case 4: return launch<4, 4, 5>(a, stream);
    case 5: return launch<5, 4, 4>(a, stream);
    case 6: return launch_192x128(a, stream);
    case 7: return launch_224x128(a, stream);
    case 8: return launch_256x128(a, stream);
    default: return launch_224x160(a, stream);
  }
}
