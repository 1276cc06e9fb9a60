// What the two sources of sdv2_linear share: the launch arguments (linear_kernel.h has the kernel, linear.hip the entry).
#ifndef SDV2KV_LINEAR_ARGS_H
#define SDV2KV_LINEAR_ARGS_H

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "linear_tiles.h"

namespace sdv2 {
namespace linear {

struct LinearArgs {
  const uint16_t* x;
  const uint16_t* w;
  const uint16_t* bias;
  uint16_t* out;
  float* squares;                            // [row][n / 32], or null
  int64_t x_st, w_st, out_st;                // elements between rows
  int32_t m, stages;                         // rows; stages of the contraction
  int32_t row_tiles, col_tiles, square_groups;       // square_groups = n / 32
};

// the tiles of 192 and more rows (linear_wide.hip)
int launch_192x128(const LinearArgs& a, hipStream_t stream);
int launch_224x128(const LinearArgs& a, hipStream_t stream);
int launch_256x128(const LinearArgs& a, hipStream_t stream);
int launch_224x160(const LinearArgs& a, hipStream_t stream);       // (no sums of squares)

}  // namespace linear
}  // namespace sdv2

#endif  // SDV2KV_LINEAR_ARGS_H
