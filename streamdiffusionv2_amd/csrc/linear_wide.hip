// The kernel of linear.hip (which see) with the tiles of 192 and more rows.
#include "linear_kernel.h"

int sdv2::linear::launch_192x128(const LinearArgs& a, hipStream_t stream) { return launch<6, 4, 4>(a, stream); }
int sdv2::linear::launch_224x128(const LinearArgs& a, hipStream_t stream) { return launch<7, 4, 3>(a, stream); }
int sdv2::linear::launch_256x128(const LinearArgs& a, hipStream_t stream) { return launch<8, 4, 3>(a, stream); }
int sdv2::linear::launch_224x160(const LinearArgs& a, hipStream_t stream) { return launch<7, 5, 3>(a, stream); }
