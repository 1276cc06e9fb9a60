// Device helpers shared by the sdv2kv kernels (gfx950 only).
#ifndef SDV2KV_INTERNAL_H
#define SDV2KV_INTERNAL_H

#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>
#include <stddef.h>
#include <stdint.h>

#include "sdv2kv.h"

namespace sdv2 {

// sdv2_swa_attn_fwd for fp32 tensors (swa_attn_fwd_f32.hip): fp32 arithmetic throughout; unsplit when the
// workspace is missing or too small
int attn_fwd_f32(const sdv2_attn_params* p, void* workspace, size_t workspace_bytes);

// Measurement hooks (sdv2kv_profile.h), kept per calling thread in
// sdv2kv_api.hip: the event pair armed for the next launch of a kernel (taken
// = disarmed).
struct TimingPair {
  void* start;
  void* stop;
};
TimingPair take_timing(int kernel);

// Launch kernel `which` (an sdv2_profile_kernel); when the calling thread has
// armed timing events for it they are attached to the kernel's own dispatch.
template <typename Kernel, typename Args>
inline void launch_timed(int which, Kernel kernel, dim3 grid, dim3 block, uint32_t lds_bytes, hipStream_t stream,
                         const Args& args) {
  const TimingPair t = take_timing(which);
  if (t.start && t.stop)
    hipExtLaunchKernelGGL(kernel, grid, block, lds_bytes, stream, static_cast<hipEvent_t>(t.start),
                          static_cast<hipEvent_t>(t.stop), 0, args);
  else
    hipLaunchKernelGGL(kernel, grid, block, lds_bytes, stream, args);
}

// One word of every 64-byte line of the kernel's arguments, asked for together.  A fresh launch finds its arguments in
// memory, and the compiler loads them where they are used: four or five trips one after another at the start of
// every workgroup.  Behind this the rest come from the scalar cache.  Eight layers of 256
// tokens x 12 heads against 1536 keys 178 -> 167 us; in the 16x16x32 attention 0.7 to 1 us of a launch (2560 x 12 heads
// against 1024 keys 22.3 -> 21.7, 1560 x 12 in three ranges of 9360 84.8 -> 83.8, in equal shares 97.6 -> 96.9), 0.4 to 1 in the sink decision.  (In
// sdv2_linear it makes no difference; in the
// 32x32x16 kernel it costs 0.5 to 1 %: that one is short of scalar registers at its start.)
template <typename Args>
__device__ __forceinline__ void fetch_arguments() {
  const auto* words = (const __attribute__((address_space(4))) uint32_t*)__builtin_amdgcn_kernarg_segment_ptr();
  constexpr int kLines = (sizeof(Args) + 63) / 64;
  uint32_t x[kLines];
#pragma unroll
  for (int i = 0; i < kLines; ++i) x[i] = words[16 * i];
#pragma unroll
  for (int i = 0; i < kLines; ++i) asm volatile("" ::"s"(x[i]));
}

// Cache positions of the chunk's own first key, one per row: the caller's device array, or host values that travel in
// the launch's arguments.
struct ChunkStarts {
  const int32_t* device;               // null: `value`
  int32_t value[SDV2_MAX_ROWS];
};
// Row `row` (wave-uniform) of the ChunkStarts at byte kOffset of the kernel's arguments, one scalar load either way.
// (Read where the arguments lie: indexing the by-value block with a run-time row would move the whole block out of
// scalar registers.)
template <int kOffset>
__device__ __forceinline__ int row_chunk_start(const int32_t* device, int row) {
  typedef const __attribute__((address_space(4))) char* arg_bytes;
  typedef const __attribute__((address_space(4))) int32_t* arg_words;
  const arg_words carried = (arg_words)((arg_bytes)__builtin_amdgcn_kernarg_segment_ptr() + kOffset + offsetof(ChunkStarts, value));
  return device ? device[row] : carried[row];
}
// host: fill `starts` from a call's parameters; the mask is on
inline int set_chunk_starts(const sdv2_attn_params& p, ChunkStarts* starts) {
  if ((p.chunk_key_start != nullptr) == (p.chunk_key_start_host != nullptr)) return SDV2_ERR_INVALID_ARG;
  starts->device = p.chunk_key_start;
  if (starts->device) return SDV2_OK;
  if (p.rows > SDV2_MAX_ROWS) return SDV2_ERR_INVALID_ARG;
  for (int i = 0; i < p.rows; ++i) {
    const int64_t first = p.chunk_key_start_host[i];
    if (first < 0 || first > (int64_t)p.max_seq_len - p.q_tokens) return SDV2_ERR_OUT_OF_RANGE;
    starts->value[i] = (int32_t)first;
  }
  return SDV2_OK;
}

// float -> bfloat16 bit pattern, round-to-nearest-even, NaN -> 0x7FC0: the
// rounding PyTorch applies when a float (or a double already narrowed to
// float) is stored as bfloat16.
__device__ __forceinline__ uint32_t f32_to_bf16_rne(float f) {
  const uint32_t u = __float_as_uint(f);
  if (f != f) return 0x7fc0u;
  return (u + 0x7fffu + ((u >> 16) & 1u)) >> 16;
}

__device__ __forceinline__ float bf16_bits_to_f32(uint32_t b) { return __uint_as_float(b << 16); }

// Two floats -> packed bfloat16 pair (lo in the low half), nearest-even: the
// hardware conversion v_cvt_pk_bf16_f32.  Same bits as f32_to_bf16_rne for every
// number; a NaN stays a NaN but keeps its sign and payload bits (PyTorch itself
// encodes a NaN result differently on its scalar, vectorised and GPU paths:
// 0x7FC0, 0xFFFF, 0x7FFF).
__device__ __forceinline__ uint32_t pack_bf16_rne(float lo, float hi) {
  typedef __attribute__((ext_vector_type(2))) float f32x2_t;
  typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2_t;
  const f32x2_t x = {lo, hi};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(x, bf16x2_t));
}

}  // namespace sdv2

#endif  // SDV2KV_INTERNAL_H
