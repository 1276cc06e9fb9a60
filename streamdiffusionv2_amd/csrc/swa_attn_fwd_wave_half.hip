// The kernel of swa_attn_fwd_wave.hip (which see) with two workgroups for a 32-query block, each with half of V's columns.
//
// A workgroup's loop is bound by what its CU brings in, 110 bytes a ns: 128 KB of 256 keys take 1.22 us, and with half of V
// 96 KB.  Where the query blocks are at most half as many as the CUs the other half of those would stand idle.
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

template <bool kMask>
__global__ __launch_bounds__(kThreads, 1)
void swa_attn_fwd_wave_half_kernel(const AttnKernelArgs a) {
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  sdv2::fetch_arguments<AttnKernelArgs>();
  WorkItem w;
  if (!w.decode(a, blockIdx.x)) return;        // (two of the list's query tiles to a block: neighbours, on one XCD)
  f32x4 sum[1];
  const int q0 = (w.qtile >> 1) * kQBlock, part = w.qtile & 1;
  stream_block<kMask, false, true, 2>(a, (lds_char*)smem, w.head, w.row, q0, 0, 0x7fffffff, sum, part);
  write_half_row(a, w.head, w.row, q0, part, sum[0]);
}

}  // namespace

int sdv2::attn::launch_wave_half(const AttnKernelArgs& a, uint32_t workgroups, hipStream_t stream) {
  // the blocks exceed the static limit: ask for the dynamic size once per device
  static std::atomic<bool> lds_ready[kMaxDevices];
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= kMaxDevices) return SDV2_ERR_LAUNCH;
  if (!lds_ready[device].load(std::memory_order_acquire)) {
    for (const void* kernel : {reinterpret_cast<const void*>(swa_attn_fwd_wave_half_kernel<false>),
                               reinterpret_cast<const void*>(swa_attn_fwd_wave_half_kernel<true>)})
      if (hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, kLdsBytes) != hipSuccess) return SDV2_ERR_LAUNCH;
    lds_ready[device].store(true, std::memory_order_release);
  }
  auto launch = [&](auto kernel) { sdv2::launch_timed(SDV2_KERNEL_ATTENTION, kernel, dim3(workgroups), dim3(kThreads), kLdsBytes, stream, a); };
  if (a.mask_block_tokens > 0) launch(swa_attn_fwd_wave_half_kernel<true>);
  else launch(swa_attn_fwd_wave_half_kernel<false>);
  return hipGetLastError() == hipSuccess ? SDV2_OK : SDV2_ERR_LAUNCH;
}
