// Sliding-window (sink + window) flash attention of a chunk's queries against
// the ring KV cache on 16x16x32 matrix instructions, for gfx950 (MI355X).
//
// Same operator, arguments, key-range splits and workspace as the kernel in
// swa_attn_fwd.hip (which see for the reference lines it stands in for and for
// the rules that pick one of the four); what differs is the matrix instruction,
// with it every register layout, and the depth of the pipeline.
//
// What bounds it: on long launches the board's power, so what counts is the
// energy of a multiply.  v_mfma_f32_16x16x32_bf16 accumulates 32 products into
// each of 256 fp32 accumulators where v_mfma_f32_32x32x16_bf16 accumulates 16 into
// each of 1024: half the accumulator traffic per product.  On random bf16 operands
// in registers the chip sustains 2063 TFLOP/s of the former and 1811 of the latter
// (on zeros, where nothing toggles, 2434 and 2466).  4 x 4680 queries x 12 heads
// against 18720 keys, same box: 1970 us with the other kernel, 1810 with this one
// (1093 -> 1189 TFLOP/s, 1.91 GHz, matrix pipe 64 % busy).  Row sums are taken by the
// matrix pipe too (mfma_row_sum): v_dot2c_f32_bf16, which adds up two packed weights,
// waits some 20 cycles for it to run empty, a fifth of the whole loop.
//
// Work decomposition: workgroup = 8 waves = up to 256 query rows of one (row, head),
// one workgroup per CU, two waves per SIMD with 256 registers each; wave w owns
// the 32-row block 32w..32w+31.  Keys stream through LDS in tiles of 64, four
// buffers per matrix, filled three tiles ahead by global->LDS transfers that never
// touch registers.
// The loop itself, its matrix layout and its softmax: attn_m16_device.h.
#include "attn_m16_kernel.h"

int sdv2::attn::launch_m16(const AttnKernelArgs& a, uint32_t workgroups, hipStream_t stream) {
  return launch<0>(a, workgroups, stream);
}
