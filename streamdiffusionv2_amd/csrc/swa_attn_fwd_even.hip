// Sliding-window (sink + window) flash attention of a chunk's queries against the
// ring KV cache, for gfx950 (MI355X), with equal shares of the key tiles for all
// workgroups.
//
// Same operator and arguments as the kernel in swa_attn_fwd.hip (which see for the
// reference lines it stands in for, and for the rule that picks this one); the loop over
// the key tiles is that of swa_attn_fwd_m16.hip (attn_m16_device.h).
//
// What bounds the kernels that hand out one query tile and key range per workgroup, once
// the ranges are long, is how the pieces fall on the 256 CUs: 1560 x 40 heads are 280
// query tiles, 40 of them for 24 rows that take three quarters of a tile's time.  Here
// the launch is one workgroup per CU.  Each takes as many query tiles whole as all can
// (neighbours side by side, so that they stream the same keys at the same time), and
// then an equal share of what is left, laid end to end: a query tile's keys are cut
// wherever a share ends (attn_even_plan.h).  A single 32-row block past the last query
// tile goes the way of a small call (attn_wave_device.h), half a tile's time.
//
// An item whose pieces meet starts at the key that its neighbours' loops have reached
// when it starts (`turn`), and goes round: all workgroups that stream one head's keys stay
// together.  With every item starting at its first key the pieces of an XCD were spread
// over the whole range, every tile came from beyond the L2, and a tile took 1.86 us
// instead of 1.55.  (4 x 4680 x 12 heads against 18720 keys 1991 -> 1664 us.)
//
// Pieces meet through memory in fp32 (what a whole item keeps in registers loses nothing
// when it is cut).  The piece that ends an item's share of its workgroup looks first
// whether all the others have left theirs - the rest of an item is the first thing the
// next workgroup does - and then keeps its own in registers; otherwise it leaves its
// result too, and the last to draw a ticket combines, in the order of the keys.  Results
// and tickets go past the L2s as in swa_attn_fwd_m16.hip; nothing waits.
//
// Against the best plan of the other kernels, same box: 1560 x 40 heads against 9360
// keys 284 -> 250 us, 2 x 1560 x 12 172 -> 163, 4 x 4680 x 12 against 18720 1755 -> 1667,
// 3807 x 12 in mask blocks of 1269 against 11421 keys 237 -> 215.  It costs some ten
// microseconds of starts, ends and meetings more than a plan that happens to fit, and
// loses below about 100 us (1560 x 12 against 9360 keys 88 -> 96).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>

#include "sdv2kv.h"
#include "sdv2kv_profile.h"
#include "sdv2kv_internal.h"
#include "attn_m16_device.h"
#include "attn_wave_device.h"

namespace {

using namespace sdv2::attn;
using namespace sdv2::attn::m16;

constexpr int kLdsEvenFlags = kLdsBytes > wave::kLdsBytes ? kLdsBytes : wave::kLdsBytes;
constexpr int kLdsEven = kLdsEvenFlags + 64;

__device__ __forceinline__ bool one_block(late_args<EvenArgs>& b, int item) {
  return item >= b.plan.whole_tiles && b.plan.rest_blocks == 1;
}
__device__ __forceinline__ ItemKind item_kind(late_args<EvenArgs>& b, int item) {
  return item < b.plan.whole_tiles ? kWholeTile : rest_kind(b.plan.rest_blocks);
}
// key tiles of the pair's item `item`, as the shares were cut
template <bool kMask>
__device__ __forceinline__ int planned_tiles(late_args<EvenArgs>& b, int item) {
  if (!kMask || !b.plan.shortened) return b.plan.tiles;
  return item_tiles(b.call.max_seq_len, item, one_block(b, item), b.call.q_tokens, row_chunk_start(b.call, 0),
                    b.call.mask_block_tokens, read_div(b.call.div_mask_block));
}

// Has every other workgroup with a piece of the item left its result?
__device__ __forceinline__ bool others_arrived(int32_t* ticket, int parts, lds_int* flag) {
  if (threadIdx.x == 0) *flag = __hip_atomic_load(ticket, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == parts - 1;
  __syncthreads();
  return *flag;
}
// This workgroup's own result is in memory once its stores are acknowledged; is it the last?
__device__ __forceinline__ bool arrive(int32_t* ticket, int parts, lds_int* flag) {
  __builtin_amdgcn_s_waitcnt(0x0F70);       // vmcnt(0)
  __syncthreads();
  if (threadIdx.x == 0) *flag = __hip_atomic_fetch_add(ticket, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == parts - 1;
  __syncthreads();
  return *flag;
}

// weights of the sum so far and of the next result, log-sum-exps `top` (of the largest so far) and `lse`
struct Meet {
  float top = -INFINITY, sum = 0.f;
  __device__ __forceinline__ void next(float lse, float& old, float& weight) {
    const float m = fmaxf(top, lse);
    old = top == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(top - m);
    weight = lse == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(lse - m);
    top = m;
    sum = sum * old + weight;
  }
};

template <bool kMask>
__global__ __launch_bounds__(kThreads, 1)
void swa_attn_fwd_even_kernel(const EvenArgs args) {
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  lds_char* lds = (lds_char*)smem;
  lds_int* flags = reinterpret_cast<lds_int*>(lds + kLdsEvenFlags);

  // Workgroups are dealt to the XCDs round robin by id; each XCD takes runs of neighbouring items and shares.
  const int per_xcd = gridDim.x >> 3, xcd = blockIdx.x & 7, in_xcd = blockIdx.x >> 3;
  sdv2::fetch_arguments<EvenArgs>();
  int round = 0;
  int begin = 0, end = 0, off = 0, pair = 0, item = 0;
  for (bool again = false;; again = true) {
    late_args<EvenArgs>& a = read_late<EvenArgs>();
    const int whole_tiles = a.plan.whole_tiles, whole_units = a.plan.whole_units;
    if (round < a.plan.rounds) {
      const int index = (xcd * a.plan.rounds + round) * per_xcd + in_xcd;
      pair = read_div(a.plan.div_tiles)(index);
      item = index - pair * whole_tiles;
    } else if (round == a.plan.rounds) {
      // the first item of this workgroup's share
      begin = (xcd * per_xcd + in_xcd) * a.plan.share;
      if (begin >= a.plan.total) return;
      end = begin + a.plan.share < a.plan.total ? begin + a.plan.share : a.plan.total;
      if (begin >= whole_units) {
        pair = read_div(a.plan.div_rest)(begin - whole_units);
        item = whole_tiles;
        off = whole_units + pair * a.plan.rest_units;
      } else if (kMask && a.plan.shortened) {
        pair = read_div(a.plan.div_whole)(begin);
        item = 0;
        off = pair * a.plan.pair_units;
        // (tiles whose last query lies in the same block of the mask are equally long)
        for (;;) {
          const int units = kWholeTile.units(planned_tiles<kMask>(a, item));
          const int block = a.call.mask_block_tokens, q_last = item * kQTile + kQTile - 1;
          const int alike = ((read_div(a.call.div_mask_block)(q_last) + 1) * block - 1 - q_last) / kQTile + 1;
          const int left = (begin - off) / units, step = left < alike ? left : alike;
          off += step * units;
          item += step;
          if (left < alike || step == 0) break;
        }
      } else {
        const int at = read_div(a.plan.div_whole)(begin), index = at + a.plan.rounds * (int)gridDim.x;
        pair = read_div(a.plan.div_tiles)(index);
        item = index - pair * whole_tiles;
        off = at * kWholeTile.units(a.plan.tiles);
      }
    }
    const bool is_block = one_block(a, item);
    const ItemKind kind = item_kind(a, item);
    const int tiles = planned_tiles<kMask>(a, item);
    const int next_off = off + kind.units(tiles);
    const bool in_round = round < a.plan.rounds;
    int tile_begin = in_round ? 0 : kind.tile_at(begin - off, tiles), tile_end = in_round ? tiles : kind.tile_at(end - off, tiles);
    if (tile_end > tile_begin) {
      const bool whole = tile_begin == 0 && tile_end == tiles;
      const int row = read_div(a.call.div_heads)(pair), head = pair - row * a.call.heads;
      if (again) __syncthreads();            // every wave is done with the buffers of the piece before
      // who has a piece of a cut item, and where their results meet
      const FastDiv div_share = read_div(a.plan.div_share);
      const int first_wg = first_workgroup(div_share, kind, off);
      const int parts = whole ? 1 : last_workgroup(div_share, kind, off, tiles) - first_wg + 1;
      const int wg = xcd * per_xcd + in_xcd;
      int32_t* ticket = whole ? nullptr : a.call.tickets + pair * (whole_tiles + (a.plan.rest_blocks > 0)) + item;
      auto part = [&](int w) { return (int64_t)(2 * w + (w == first_wg)); };

      if (!is_block) {
        const int seq = row_keys(a.call, row);
        const TileSpan list = tile_list<kMask>(a.call, tile_end_row(a.call, item, kQTile), kMask ? row_chunk_start(a.call, row) : 0, seq);
        // (a row may hold fewer keys than the longest one)
        tile_begin = tile_begin < list.count ? tile_begin : list.count;
        tile_end = tile_end < list.count ? tile_end : list.count;
        // the item's first tile is the one its neighbours are at when it starts
        int turn = in_round ? 0 : (off - read_div(a.plan.div_share)(off) * a.plan.share) / kWholeTile.per_tile;
        if (list.count > 0) turn = (int)((uint32_t)turn % (uint32_t)list.count);
        turn = __builtin_amdgcn_readfirstlane(turn);
        auto key0_of = [=](int entry) {
          int tile = entry + turn;
          tile = tile >= list.count ? tile - list.count : tile;
          return (kMask && tile >= list.hole ? tile + list.skipped : tile) * kKTile;
        };
        LaneConst c;
        f32x4 oacc[8][2];
        float l_sum[2];
        // (a piece that ends the share finds the others of its item done, more often than not)
        const bool ends = !whole && next_off >= end && tile_end > tile_begin;
        stream_range<kMask>(a.call, lds, item * kQTile, tile_end_row(a.call, item, kQTile), head, row, seq, key0_of, tile_begin, tile_end, c, oacc, l_sum,
                            Peek{ends ? ticket : nullptr, parts - 1, flags});

        late_args<EvenArgs>& b = read_late<EvenArgs>();
        int tid = threadIdx.x;
        asm volatile("" : "+v"(tid));
        const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        const int n16 = lane & 15, g = lane >> 4;
        const bool idle = item * kQTile + wave * kQBlock >= b.call.q_tokens;
        float inv[2];
#pragma unroll
        for (int qt = 0; qt < 2; ++qt) inv[qt] = l_sum[qt] > 0.f ? 1.0f / l_sum[qt] : 0.f;
        lds_char* stage = lds + wave * kStage16;

        if (whole) {
          if (!idle) {
#pragma unroll
            for (int db = 0; db < 8; ++db) stage_out(stage, lane, db, oacc[db], inv);
            write_block(b.call, stage, item * kQTile + wave * kQBlock, head, row, lane);
          }
        } else {
          float lse[2];
#pragma unroll
          for (int qt = 0; qt < 2; ++qt) {
            lse[qt] = l_sum[qt] > 0.f ? __builtin_amdgcn_logf(l_sum[qt]) - c.neg_ref[qt] : -INFINITY;
#pragma unroll
            for (int db = 0; db < 8; ++db)
#pragma unroll
              for (int i = 0; i < 4; ++i) oacc[db][qt][i] *= inv[qt];
          }
          float* const part_o = b.part_o + wave * (kQBlock * kD) + lane * 4;
          float* const part_lse = b.part_lse + wave * kQBlock;
          bool last = ends && flags[0];
          if (!last) {
            if (!idle) {
              char* dst = reinterpret_cast<char*>(part_o + part(wg) * kEvenPartFloats);
#pragma unroll
              for (int db = 0; db < 8; db += 2)
                store_coherent_x4(dst + db * 2048, __builtin_bit_cast(u32x4, oacc[db][0]), __builtin_bit_cast(u32x4, oacc[db][1]),
                                  __builtin_bit_cast(u32x4, oacc[db + 1][0]), __builtin_bit_cast(u32x4, oacc[db + 1][1]));
              if (g < 2) store_coherent(part_lse + part(wg) * kEvenPartRows + lane, g ? lse[1] : lse[0]);
            }
            last = arrive(ticket, parts, flags + 1);
          }
          if (last) {
            if (tid == 0) __hip_atomic_store(ticket, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (!idle) {
              auto stats = [&](int w, int qt) { return load_coherent(part_lse + part(w) * kEvenPartRows + n16 + 16 * qt); };
              auto result = [&](int w) { return reinterpret_cast<const char*>(part_o + part(w) * kEvenPartFloats); };
              if (parts == 2) {
                // the other one's result in one trip; two terms, each rounded, have no order
#pragma clang fp contract(off)
                const int w = wg == first_wg ? wg + 1 : first_wg;
                const float lse2[2] = {stats(w, 0), stats(w, 1)};
                u32x4 x[4][4];
                const char* src = result(w);
                load_coherent_4x4(src, src + 4096, src + 8192, src + 12288, x);
                float mine[2], other[2];
#pragma unroll
                for (int qt = 0; qt < 2; ++qt) {
                  const float top = fmaxf(lse[qt], lse2[qt]);
                  mine[qt] = lse[qt] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(lse[qt] - top);
                  other[qt] = lse2[qt] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(lse2[qt] - top);
                  const float sum = mine[qt] + other[qt];
                  inv[qt] = sum > 0.f ? 1.0f / sum : 0.f;
                }
#pragma unroll
                for (int db = 0; db < 8; ++db) {
                  f32x4 o[2];
#pragma unroll
                  for (int qt = 0; qt < 2; ++qt) {
                    const f32x4 y = __builtin_bit_cast(f32x4, x[db >> 1][2 * (db & 1) + qt]);
#pragma unroll
                    for (int i = 0; i < 4; ++i) o[qt][i] = oacc[db][qt][i] * mine[qt] + y[i] * other[qt];
                  }
                  stage_out(stage, lane, db, o, inv);
                }
              } else {
                // in the order of the keys, half of the columns and two results at a time
                const int last_wg = first_wg + parts - 1;
#pragma unroll
                for (int half = 0; half < 2; ++half) {
                  f32x4 acc[4][2];
                  Meet meet[2];
#pragma unroll
                  for (int db = 0; db < 4; ++db) acc[db][0] = acc[db][1] = f32x4{0.f, 0.f, 0.f, 0.f};
                  for (int w0 = first_wg; w0 <= last_wg; w0 += 2) {
                    const int w1 = w0 < last_wg ? w0 + 1 : w0;
                    float part_lse2[2][2] = {{stats(w0, 0), stats(w0, 1)}, {stats(w1, 0), stats(w1, 1)}};
                    u32x4 x[4][4];
                    const char *src0 = result(w0) + half * 8192, *src1 = result(w1) + half * 8192;
                    load_coherent_4x4(src0, src0 + 4096, src1, src1 + 4096, x);
#pragma unroll
                    for (int u = 0; u < 2; ++u) {
                      if (u == 1 && w1 == w0) break;
                      const bool own = (u ? w1 : w0) == wg;
#pragma unroll
                      for (int qt = 0; qt < 2; ++qt) {
                        float old, weight;
                        meet[qt].next(own ? lse[qt] : part_lse2[u][qt], old, weight);
#pragma unroll
                        for (int db = 0; db < 4; ++db) {
                          const f32x4 y = __builtin_bit_cast(f32x4, x[2 * u + (db >> 1)][2 * (db & 1) + qt]);
#pragma unroll
                          for (int i = 0; i < 4; ++i)
                            acc[db][qt][i] = acc[db][qt][i] * old + weight * (own ? oacc[4 * half + db][qt][i] : y[i]);
                        }
                      }
                    }
                  }
#pragma unroll
                  for (int qt = 0; qt < 2; ++qt) inv[qt] = meet[qt].sum > 0.f ? 1.0f / meet[qt].sum : 0.f;
#pragma unroll
                  for (int db = 0; db < 4; ++db) stage_out(stage, lane, 4 * half + db, acc[db], inv);
                }
              }
              write_block(b.call, stage, item * kQTile + wave * kQBlock, head, row, lane);
            }
          }
        }
      } else {
        const int q0 = item * kQTile;
        f32x4 sum[2];
        wave::stream_block<kMask, false, false>(a.call, lds, head, row, q0, 2 * tile_begin, 2 * tile_end, sum);
        late_args<EvenArgs>& b = read_late<EvenArgs>();
        bool write = whole;
        if (!whole) {
          const float lse = wave::row_lse(lds, b.call.scale_log2);
          const int at = (threadIdx.x >> 4) * kD + (threadIdx.x & 15) * 8;
          write = next_off >= end && others_arrived(ticket, parts, flags);
          if (!write) {
            store_coherent_x2(b.part_o + part(wg) * kEvenPartFloats + at, sum[0], sum[1]);
            if ((threadIdx.x & 15) == 0) store_coherent(b.part_lse + part(wg) * kEvenPartRows + (threadIdx.x >> 4), lse);
            write = arrive(ticket, parts, flags + 1);
          }
          if (write) {
            if (threadIdx.x == 0) __hip_atomic_store(ticket, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            f32x4 acc[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
            Meet meet;
            for (int w = first_wg; w < first_wg + parts; ++w) {
              float part_lse = lse, old, weight;
              f32x4 x[2] = {sum[0], sum[1]};
              if (w != wg) {
                part_lse = load_coherent(b.part_lse + part(w) * kEvenPartRows + (threadIdx.x >> 4));
                load_coherent_x2(b.part_o + part(w) * kEvenPartFloats + at, x[0], x[1]);
              }
              meet.next(part_lse, old, weight);
#pragma unroll
              for (int k = 0; k < 2; ++k)
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[k][i] = acc[k][i] * old + weight * x[k][i];
            }
            const float inv = meet.sum > 0.f ? 1.0f / meet.sum : 0.f;
#pragma unroll
            for (int k = 0; k < 2; ++k)
#pragma unroll
              for (int i = 0; i < 4; ++i) sum[k][i] = acc[k][i] * inv;
          }
        }
        if (write) wave::write_row(b.call, head, row, q0, sum);
      }
    }
    if (in_round) {
      ++round;
      continue;
    }
    if (next_off >= end) return;
    round = 0x7fffffff;        // (the next item is this one's neighbour)
    off = next_off;
    if (item < whole_tiles && ++item == whole_tiles) {
      item = 0;
      ++pair;
    } else if (item == whole_tiles) {
      ++pair;
    }
    if (off == whole_units) {
      pair = 0;
      item = whole_tiles;
    }
  }
}

}  // namespace

int sdv2::attn::launch_even(const EvenArgs& a, hipStream_t stream) {
  // the tile buffers exceed the static limit: ask for the dynamic size once per device
  static std::atomic<bool> lds_ready[kMaxDevices];
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= kMaxDevices) return SDV2_ERR_LAUNCH;
  if (!lds_ready[device].load(std::memory_order_acquire)) {
    for (const void* kernel : {reinterpret_cast<const void*>(swa_attn_fwd_even_kernel<false>),
                               reinterpret_cast<const void*>(swa_attn_fwd_even_kernel<true>)})
      if (hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, kLdsEven) != hipSuccess) return SDV2_ERR_LAUNCH;
    lds_ready[device].store(true, std::memory_order_release);
  }
  auto launch = [&](auto kernel) { sdv2::launch_timed(SDV2_KERNEL_ATTENTION, kernel, dim3(a.plan.workgroups), dim3(kThreads), kLdsEven, stream, a); };
  if (a.call.mask_block_tokens > 0) launch(swa_attn_fwd_even_kernel<true>);
  else launch(swa_attn_fwd_even_kernel<false>);
  return hipGetLastError() == hipSuccess ? SDV2_OK : SDV2_ERR_LAUNCH;
}
