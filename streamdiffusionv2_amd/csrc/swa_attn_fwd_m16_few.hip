// The kernel of swa_attn_fwd_m16.hip for query tiles of at most four blocks of 32 rows: waves 4 to 7, which have no rows, move
// the key tiles (first_issuer).  Compiled apart, with the number of the first of them known: as an argument it changed nothing
// that one can see in the loop of the wide tiles (the same instructions on the same vector registers), and cost it 0.7 %
// (2 x 10800 x 12 heads against 75600 keys 7483 -> 7537 us, medians of 60 in turn, quartiles 7473 to 7493 and 7511 to 7555).
#include "attn_m16_kernel.h"

int sdv2::attn::launch_m16_few(const AttnKernelArgs& a, uint32_t workgroups, hipStream_t stream) {
  return launch<kIssuers>(a, workgroups, stream);
}
