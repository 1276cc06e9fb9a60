// The kernel of swa_attn_fwd_m16.hip for query tiles of five and of six blocks of 32 rows, whose waves 4 to 7 share the fifth,
// or the fifth and the sixth, by key (SharedBlock in attn_m16_device.h).  Of five blocks they also move the key tiles, having
// a quarter of a block's work each (waves 0 to 3: 158.1 -> 165.4 us for 3200 x 12 heads against 9344 keys); of six waves 0 to 3
// do (waves 4 to 7: 188.9 -> 196.0 us for 3840 x 12).
#include "attn_m16_kernel.h"

int sdv2::attn::launch_m16_shared(const AttnKernelArgs& a, uint32_t workgroups, hipStream_t stream) {
  return a.q_tile_rows > 5 * kQBlock ? launch_one<false, 0, 2>(a, workgroups, stream)
                                     : launch_one<false, kIssuers, 4>(a, workgroups, stream);
}
