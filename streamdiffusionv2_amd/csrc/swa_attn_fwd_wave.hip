// Sliding-window (sink + window) flash attention for small calls, for gfx950 (MI355X).
//
// Same operator and arguments as the kernel in swa_attn_fwd.hip (which see for the
// reference lines it stands in for, and for the rules that pick one of the four).
//
// What bounds a small call is not the matrix pipe but how long one workgroup takes
// and how few there are: 256 queries x 12 heads are 12 query tiles of the other
// kernels, 48 workgroups with the keys cut four ways, and the ranges meet through
// memory.  Here a workgroup is 8 waves on ONE 32-query block (96 workgroups for
// that call), the waves take the keys 32 at a time in turn, each by itself, and
// meet once, in LDS, at the end: no barrier while the keys stream, no partial results
// in memory, no ticket.  The price is that no wave shares a key it has fetched with
// another: every workgroup streams all keys from L2, and those trips bound its
// loop, 1.22 us per 256 keys (128 KB) whether 8 workgroups run or 240; the products
// alone would take 0.8.  256 x 12 heads against 1536 keys: 21.6 us with the tile
// kernels' best plan, 13.7 with this one; 512 keys 17.0 and 9.0.
// A block's way through a workgroup: attn_wave_device.h.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>

#include "sdv2kv.h"
#include "sdv2kv_profile.h"
#include "sdv2kv_internal.h"
#include "attn_wave_device.h"

namespace {

using namespace sdv2::attn;
using namespace sdv2::attn::wave;

template <bool kMask, bool kRope>
__global__ __launch_bounds__(kThreads, 1)
void swa_attn_fwd_wave_kernel(const AttnKernelArgs a) {
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  sdv2::fetch_arguments<AttnKernelArgs>();
  WorkItem w;
  if (!w.decode(a, blockIdx.x)) return;
  f32x4 sum[2];
  stream_block<kMask, kRope, true>(a, (lds_char*)smem, w.head, w.row, w.qtile * kQBlock, 0, 0x7fffffff, sum);
  write_row(a, w.head, w.row, w.qtile * kQBlock, sum);
}

}  // namespace

int sdv2::attn::launch_wave(const AttnKernelArgs& a, uint32_t workgroups, hipStream_t stream) {
  // the V blocks exceed the static limit: ask for the dynamic size once per device
  static std::atomic<bool> lds_ready[kMaxDevices];
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= kMaxDevices) return SDV2_ERR_LAUNCH;
  auto launch = [&](auto kernel) { sdv2::launch_timed(SDV2_KERNEL_ATTENTION, kernel, dim3(workgroups), dim3(kThreads), kLdsBytes, stream, a); };
  if (!lds_ready[device].load(std::memory_order_acquire)) {
    for (const void* kernel : {reinterpret_cast<const void*>(swa_attn_fwd_wave_kernel<false, false>),
                               reinterpret_cast<const void*>(swa_attn_fwd_wave_kernel<false, true>),
                               reinterpret_cast<const void*>(swa_attn_fwd_wave_kernel<true, false>),
                               reinterpret_cast<const void*>(swa_attn_fwd_wave_kernel<true, true>)})
      if (hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, kLdsBytes) != hipSuccess) return SDV2_ERR_LAUNCH;
    lds_ready[device].store(true, std::memory_order_release);
  }
  if (a.mask_block_tokens > 0) {
    if (a.freqs) launch(swa_attn_fwd_wave_kernel<true, true>);
    else launch(swa_attn_fwd_wave_kernel<true, false>);
  } else {
    if (a.freqs) launch(swa_attn_fwd_wave_kernel<false, true>);
    else launch(swa_attn_fwd_wave_kernel<false, false>);
  }
  return hipGetLastError() == hipSuccess ? SDV2_OK : SDV2_ERR_LAUNCH;
}
