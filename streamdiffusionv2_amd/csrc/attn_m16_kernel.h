// The kernel of swa_attn_fwd_m16.hip (which see), for the sources that compile it: kFirstIssuer is the first of the
// waves that move the tiles, 0, or 4 in query tiles with rows for four waves (first_issuer) and in those whose waves 4 to 7
// share a block (kShare: SharedBlock).
#ifndef SDV2KV_ATTN_M16_KERNEL_H
#define SDV2KV_ATTN_M16_KERNEL_H

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>

#include "sdv2kv.h"
#include "sdv2kv_profile.h"
#include "sdv2kv_internal.h"
#include "attn_m16_device.h"

namespace {

using namespace sdv2::attn;
using namespace sdv2::attn::m16;

template <bool kMask, int kFirstIssuer, int kShare>
__global__ __launch_bounds__(kThreads, 1)
void swa_attn_fwd_m16_kernel(const AttnKernelArgs args) {
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  lds_char* lds = (lds_char*)smem;
  lds_int* flags = reinterpret_cast<lds_int*>(lds + kLdsFlags);

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int n16 = lane & 15, g = lane >> 4;

  sdv2::fetch_arguments<AttnKernelArgs>();
  WorkItem w;
  if (!w.decode(args, blockIdx.x)) return;
  late_args<AttnKernelArgs>& a = read_late<AttnKernelArgs>();
  const int qtile = w.qtile, head = w.head, row = w.row, split = w.split, nsplits = w.nsplits;

  const int seq = row_keys(a, row);
  const int q_first = qtile * a.q_tile_rows, q_end = tile_end_row(a, qtile, a.q_tile_rows);
  const TileSpan list = tile_list<kMask>(a, q_end, kMask ? row_chunk_start(a, row) : 0, seq);
  const int per_split = (list.count + nsplits - 1) / nsplits;
  const int tile_begin = split * per_split;
  int tile_end = tile_begin + per_split;
  tile_end = tile_end < list.count ? tile_end : list.count;

  LaneConst c;
  f32x4 oacc[8][2];
  float l_tot[2];
  auto key0_of = [=](int tile) { return (kMask && tile >= list.hole ? tile + list.skipped : tile) * kKTile; };
  stream_range<kMask, kFirstIssuer, kShare>(a, lds, q_first, q_end, head, row, seq, key0_of, tile_begin, tile_end, c, oacc, l_tot);
  late_args<AttnKernelArgs>& b = read_late<AttnKernelArgs>();
  const int q0 = qtile * b.q_tile_rows + wave_block<kShare>(wave) * kQBlock;           // of this wave
  const bool idle = __builtin_amdgcn_readfirstlane(q0 >= tile_end_row(b, qtile, b.q_tile_rows) || share_part<kShare>(wave) > 0);

  // ---- epilogue ---------------------------------------------------------------
  // (every wave is done with the K / V buffers: the barrier above, or the last one of the exact pass)
  const int block = q0 / kQBlock;                       // this wave's 32-row block within the (row, head)
  float inv[2];
#pragma unroll
  for (int qt = 0; qt < 2; ++qt) {
    inv[qt] = l_tot[qt] > 0.f ? 1.0f / l_tot[qt] : 0.f;
  }

  lds_char* stage = lds + wave * kStage16;

  if (nsplits > 1) {
    // Partial result of a key range: the normalised row divided by its largest
    // magnitude, as fp16 (values in [-1, 1]: 11 bits against the row's scale,
    // sixteen times finer than the bf16 of the final result), plus that scale
    // and the log-sum-exp.  Stored in register order - 16-byte piece db of a lane
    // holds its accumulators of dimension block db, both queries - so that every
    // store and, later, every load is one contiguous kilobyte per wave.
    const int64_t slab = (int64_t)b.rows * b.heads * b.q_blocks;
    const int64_t blk0 = ((int64_t)row * b.heads + head) * b.q_blocks + block;
    if (!idle) {
      float row_scale[2], to_unit[2], lse[2];
#pragma unroll
      for (int qt = 0; qt < 2; ++qt) {
        float amax = 0.f;
#pragma unroll
        for (int db = 0; db < 8; ++db)
#pragma unroll
          for (int i = 0; i < 4; ++i) amax = vmax(amax, __builtin_fabsf(oacc[db][qt][i]));
        amax = col_max(amax) * inv[qt];
        row_scale[qt] = amax > 0.f && amax < INFINITY ? amax : 1.0f;
        to_unit[qt] = inv[qt] / row_scale[qt];
        lse[qt] = l_tot[qt] > 0.f ? __builtin_amdgcn_logf(l_tot[qt]) - c.neg_ref[qt] : -INFINITY;
      }
      const int64_t blk = split * slab + blk0;
      char* dst = reinterpret_cast<char*>(b.part_o + blk * kPartBlockHalves + lane * 8);
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        u32x4 x[4];
#pragma unroll
        for (int jj = 0; jj < 4; ++jj)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int db = 4 * half + jj, qt = e >> 1, i = 2 * (e & 1);
            x[jj][e] = pack_f16x2(oacc[db][qt][i] * to_unit[qt], oacc[db][qt][i + 1] * to_unit[qt]);
          }
        store_coherent_x4(dst + half * 4096, x[0], x[1], x[2], x[3]);
      }
      if (g < 2) {        // lanes 0-15 the first query tile's rows, 16-31 the second's
        store_coherent(b.part_lse + blk * kQBlock + lane, g ? lse[1] : lse[0]);
        store_coherent(b.part_scale + blk * kQBlock + lane, g ? row_scale[1] : row_scale[0]);
      }
    }
    // Ticket.  Every wave has waited for its stores to be acknowledged before the
    // barrier; then one lane draws.  The workgroup that draws the last ticket of
    // its (row, head, query tile) finds every other range's results in memory,
    // and leaves the ticket at zero for the next call.
    __builtin_amdgcn_s_waitcnt(0x0F70);       // vmcnt(0)
    __syncthreads();
    if (tid == 0) {
      int32_t* ticket = b.tickets + ((int64_t)row * b.heads + head) * b.q_tiles + qtile;
      const int drawn = __hip_atomic_fetch_add(ticket, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const int last = drawn == nsplits - 1;
      if (last) __hip_atomic_store(ticket, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      flags[1] = last;
    }
    __syncthreads();
    if (flags[1] == 0 || idle) return;

    // combine: out = sum_s 2^(lse_s - LSE) O_s over the ranges in their fixed
    // order (every range, this workgroup's own included, as it lies in memory:
    // the sum does not depend on which workgroup happens to be last).  A trip to
    // memory costs the same microsecond and a half whatever it carries, so the
    // statistics of four ranges travel with half of their outputs, and the other
    // half follows (all of it at once does not fit the registers).
    constexpr int kBatch = 4;
    float lse_max[2] = {-INFINITY, -INFINITY};
    float lse[kBatch][2], ws[kBatch][2];
    auto fetch = [&](int s0) {
#pragma unroll
      for (int u = 0; u < kBatch; ++u) {
        const int sp = s0 + u < nsplits ? s0 + u : nsplits - 1;
        const int64_t at = (sp * slab + blk0) * kQBlock + n16;
#pragma unroll
        for (int qt = 0; qt < 2; ++qt) {
          lse[u][qt] = load_coherent(b.part_lse + at + 16 * qt);
          ws[u][qt] = load_coherent(b.part_scale + at + 16 * qt);
        }
      }
    };
    auto part_at = [&](int sp, int half) {
      return reinterpret_cast<const char*>(b.part_o + ((sp < nsplits ? sp : nsplits - 1) * slab + blk0) * kPartBlockHalves +
                                           lane * 8) + half * 4096;
    };
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      f32x4 acc[4][2];
#pragma unroll
      for (int db = 0; db < 4; ++db) acc[db][0] = acc[db][1] = f32x4{0.f, 0.f, 0.f, 0.f};
      float wsum[2] = {0.f, 0.f};
      for (int s0 = 0; s0 < nsplits; s0 += kBatch) {
        u32x4 x[kBatch][4];
        if (half == 0 || nsplits > kBatch) fetch(s0);
        load_coherent_4x4(part_at(s0, half), part_at(s0 + 1, half), part_at(s0 + 2, half), part_at(s0 + 3, half), x);
        if (half == 0 && s0 == 0)
#pragma unroll
          for (int qt = 0; qt < 2; ++qt) {
#pragma unroll
            for (int u = 0; u < kBatch; ++u) lse_max[qt] = fmaxf(lse_max[qt], lse[u][qt]);      // (entries past the last range repeat it)
            for (int sp = kBatch; sp < nsplits; ++sp)
              lse_max[qt] = fmaxf(lse_max[qt], load_coherent(b.part_lse + (sp * slab + blk0) * kQBlock + n16 + 16 * qt));
          }
#pragma unroll
        for (int u = 0; u < kBatch; ++u) {
          float w2[2];
#pragma unroll
          for (int qt = 0; qt < 2; ++qt) {
            const float e = (s0 + u >= nsplits || lse[u][qt] == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f(lse[u][qt] - lse_max[qt]);
            wsum[qt] += e;
            w2[qt] = e * ws[u][qt];             // weight times the row's fp16 scale
          }
          if (s0 + u < nsplits)
#pragma unroll
            for (int db = 0; db < 4; ++db) {
              const f16x8 h = __builtin_bit_cast(f16x8, x[u][db]);
#pragma unroll
              for (int e = 0; e < 8; ++e) acc[db][e >> 2][e & 3] += w2[e >> 2] * static_cast<float>(h[e]);
            }
        }
      }
#pragma unroll
      for (int qt = 0; qt < 2; ++qt) inv[qt] = wsum[qt] > 0.f ? 1.0f / wsum[qt] : 0.f;
#pragma unroll
      for (int db = 0; db < 4; ++db) stage_out(stage, lane, 4 * half + db, acc[db], inv);
    }
  } else if (idle) {
    return;
  } else {
#pragma unroll
    for (int db = 0; db < 8; ++db) stage_out(stage, lane, db, oacc[db], inv);
  }

  write_block(b, stage, q0, head, row, lane);
}

// the tile buffers exceed the static limit: ask for the dynamic size once per device
template <bool kMask, int kFirstIssuer, int kShare>
int launch_one(const AttnKernelArgs& a, uint32_t workgroups, hipStream_t stream) {
  constexpr int kLds = kShare > 0 ? kLdsSharedBytes : kLdsBytes;
  auto kernel = swa_attn_fwd_m16_kernel<kMask, kFirstIssuer, kShare>;
  static std::atomic<bool> lds_ready[kMaxDevices];
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= kMaxDevices) return SDV2_ERR_LAUNCH;
  if (!lds_ready[device].load(std::memory_order_acquire)) {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, kLds) != hipSuccess)
      return SDV2_ERR_LAUNCH;
    lds_ready[device].store(true, std::memory_order_release);
  }
  sdv2::launch_timed(SDV2_KERNEL_ATTENTION, kernel, dim3(workgroups), dim3(kThreads), kLds, stream, a);
  return hipGetLastError() == hipSuccess ? SDV2_OK : SDV2_ERR_LAUNCH;
}
template <int kFirstIssuer>
int launch(const AttnKernelArgs& a, uint32_t workgroups, hipStream_t stream) {
  return a.mask_block_tokens > 0 ? launch_one<true, kFirstIssuer, 0>(a, workgroups, stream)
                                 : launch_one<false, kFirstIssuer, 0>(a, workgroups, stream);
}

}  // namespace

#endif  // SDV2KV_ATTN_M16_KERNEL_H
