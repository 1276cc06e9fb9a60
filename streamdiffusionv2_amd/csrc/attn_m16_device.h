// The streaming loop of the bf16 attention on 16x16x32 matrix instructions (gfx950
// only): 8 waves = up to 256 query rows of one (row, head) against a range of its keys, for
// the kernels that give a workgroup one such range (swa_attn_fwd_m16.hip) or a
// share of several (swa_attn_fwd_even.hip).
//
// Keys stream through LDS in tiles of 64, four buffers per matrix, filled three tiles
// ahead by global->LDS transfers that never touch registers; wave w owns the 32 query
// rows 32w..32w+31.
//
// Matrix layout (D = A(16x32) * B(32x16) + C; lane l: n = l % 16, g = l / 16):
//   S^T = K Q^T   A = K: key n, head dimensions 8 g..8 g + 7 of a 32-wide step
//                 (ds_read_b128); B = Q: query n, the same dimensions, in
//                 registers for the whole kernel.  D: query n, keys 4 g..4 g + 3.
//   O^T = V^T P^T One instruction contracts a whole 32-key block.  B = P^T is the
//                 packed accumulators of the block's two 16-key score tiles as
//                 they stand, keys {4 g.., 16 + 4 g..}: no cross-lane movement.
//                 A = V^T of the same keys, two ds_read_b64_tr_b16 (LDS transpose
//                 loads) 16 keys apart.
//   A wave's 32 queries are two column tiles (qt), so every A fragment feeds two
//   matrix instructions and a lane owns TWO queries, n and 16 + n.
//
// Softmax: exp2 of the scaled scores against a fixed reference per query, the
// largest score among the first 32 keys of the workgroup's range; nothing is
// rescaled.  A wave that finds a row sum outside [2^-100, 2^100] after its last
// tile redoes its block with the running-maximum recurrence (exact_pass).
//
// LDS tile layout: row r (key) holds sixteen 16-byte chunks; chunk c is stored at
// position c ^ swz16(r) (attn_device.h).
#ifndef SDV2KV_ATTN_M16_DEVICE_H
#define SDV2KV_ATTN_M16_DEVICE_H

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "sdv2kv.h"
#include "sdv2kv_internal.h"
#include "rope_device.h"
#include "attn_device.h"

namespace sdv2 {
namespace attn {
namespace m16 {

constexpr int kWaves = 8;
constexpr int kThreads = kWaves * 64;
constexpr int kQTile = kWaves * kQBlock;
constexpr int kStages = 4;
constexpr int kHalf = 32 * 256;             // bytes of half a tile: one 32-key block
constexpr int kSub = 16 * 256;              // bytes of 16 keys
constexpr int kStage16 = 8192;              // epilogue staging per wave: 32 rows x 256 B
constexpr int kLdsFlags = 2 * kStages * kTileBytes;
constexpr int kLdsBytes = kLdsFlags + 256;
constexpr int kLdsSharedBytes = kLdsBytes + 4 * 512;       // with the row sums of waves that share a block
static_assert(kWaves * kStage16 <= kLdsFlags, "the epilogue stages in the tile buffers");

// LDS map: kStages K tile buffers, then kStages V tile buffers.  The DS
// instructions carry a 16-bit offset, so V fragment addresses are kept
// relative to the first V buffer with the base folded into the address register.
constexpr int kLdsBuf(int buf) { return buf * kTileBytes; }
constexpr int kLdsVBase = kStages * kTileBytes;

// The MFMAs of the fast pass are asm with the register class of every operand
// named: scores feed the vector ALU and stay in VGPRs, the output tile and the
// query fragments live in AGPRs (at 256 registers per wave at most 128 are
// VGPRs).  `kPending` is the s_waitcnt that makes the A fragment valid; -1 = it
// was already waited for.  The compiler's hazard tracking does not see inside:
// scores are read by the vector ALU at least two matrix instructions after the
// one that finished them, P is written a full slot before it is read, and O is
// only read behind a drain.
template <int kPending>
__device__ __forceinline__ void mfma_s_first(f32x4& d, const u32x4& a, const bf16x8& b) {
  if constexpr (kPending >= 0)
    asm volatile("s_waitcnt lgkmcnt(%3)\n\tv_mfma_f32_16x16x32_bf16 %0, %1, %2, 0"
                 : "=&v"(d) : "v"(a), "a"(b), "n"(kPending));
  else
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=&v"(d) : "v"(a), "a"(b));
}
template <int kPending>
__device__ __forceinline__ void mfma_s(f32x4& d, const u32x4& a, const bf16x8& b) {
  if constexpr (kPending >= 0)
    asm volatile("s_waitcnt lgkmcnt(%3)\n\tv_mfma_f32_16x16x32_bf16 %0, %1, %2, %0"
                 : "+v"(d) : "v"(a), "a"(b), "n"(kPending));
  else
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(d) : "v"(a), "a"(b));
}
template <int kPending>
__device__ __forceinline__ void mfma_o(f32x4& d, const u32x4& a, const u32x4& b) {
  if constexpr (kPending >= 0)
    asm volatile("s_waitcnt lgkmcnt(%3)\n\tv_mfma_f32_16x16x32_bf16 %0, %1, %2, %0"
                 : "+a"(d) : "v"(a), "v"(b), "n"(kPending));
  else
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(d) : "v"(a), "v"(b));
}

// row sums of the packed weights: every register of d is the sum of all 32 weights of the lane's query
__device__ __forceinline__ void mfma_row_sum(f32x4& d, const u32x4& ones, const u32x4& p) {
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(d) : "a"(ones), "v"(p));
}

// One 64-key tile of K or of V: instruction i (0..15, kPieces per issuing wave)
// fills rows 4i..4i+3; lane l lands on row 4i + l/16, physical chunk l%16, so it
// fetches logical chunk (l%16) ^ swz16(row).  The lane's part of that offset is worked out
// per instruction from two registers (a table of eight does not fit beside the loop's own):
// swz16(4 j + g) = g << 1 ^ piece_swizzle(j).  The last, partial tile redirects rows
// at or past the valid length to the last valid key (their scores are masked).
// (Dealing the transfers out between the matrix instructions of a slot, with four
// or with all eight waves issuing, was measured 2-5 % slower than this clump behind
// the barrier.)
constexpr int piece_swizzle(int j) { return ((j ^ j >> 1) & 1) << 3 | (j >> 1 & 1); }
struct LaneFetch {
  uint32_t chunk;         // 16 * (l % 16 ^ (l / 16) << 1)
  uint32_t k_row, v_row;  // bytes from the wave's first row to this lane's of a piece: (l / 16) * token stride
};
__device__ __forceinline__ void issue_tile(const char* base, uint32_t tok_bytes, uint32_t chunk, uint32_t row_off, int key0,
                                           int seq, uint32_t lds_dst, int issuer, int lane) {
  if ((unsigned)issuer >= kIssuers) return;
  const char* tile = base + (int64_t)key0 * tok_bytes;      // wave-uniform
  if (key0 + kKTile <= seq) {
#pragma unroll
    for (int j = 0; j < kPieces; ++j)
      dma16(tile + (uint64_t)((issuer * kPieces + j) * 4) * tok_bytes, (chunk ^ (uint32_t)(piece_swizzle(j) << 4)) + row_off,
            lds_dst + (issuer * kPieces + j) * 1024);
  } else {
    const int last_rel = seq - 1 - key0;
#pragma unroll
    for (int j = 0; j < kPieces; ++j) {
      const int r = 4 * (issuer * kPieces + j) + (lane >> 4);
      const int rr = r < last_rel ? r : last_rel;
      dma16(tile, (uint32_t)rr * tok_bytes + (chunk ^ (uint32_t)(piece_swizzle(j) << 4)), lds_dst + (issuer * kPieces + j) * 1024);
    }
  }
}
static_assert(kPieces == 4, "piece_swizzle");

// See mfma_drain in swa_attn_fwd.hip: nothing the compiler generates may touch S
// or O while an asm MFMA is in flight.  (The operands are tied in a second,
// empty statement: one statement does not take them all.)
template <int kTag>
__device__ __forceinline__ void mfma_drain(f32x4 (&o)[8][2], f32x4 (&s)[2][2][2]) {
  asm volatile("s_nop 15\n\ts_nop 15 ; matrix pipe drained, site %8"
               : "+v"(s[0][0][0]), "+v"(s[0][0][1]), "+v"(s[0][1][0]), "+v"(s[0][1][1]), "+v"(s[1][0][0]),
                 "+v"(s[1][0][1]), "+v"(s[1][1][0]), "+v"(s[1][1][1])
               : "n"(kTag));
#pragma unroll
  for (int db = 0; db < 8; db += 4)
    asm volatile("; site %8"
                 : "+a"(o[db][0]), "+a"(o[db][1]), "+a"(o[db + 1][0]), "+a"(o[db + 1][1]), "+a"(o[db + 2][0]),
                   "+a"(o[db + 2][1]), "+a"(o[db + 3][0]), "+a"(o[db + 3][1])
                 : "n"(kTag));
}

struct LaneConst {
  u32x4 ones;             // eight bf16 ones
  uint32_t k_addr[4];     // K fragment of d-step ks: key row lane%16 of a 16-key tile
  uint32_t v_addr[8];     // V^T fragment of d block db, keys 4 g.. of a 32-key block
  float c2;               // softmax scale * log2(e)
  float neg_ref[2];       // minus the query's exponent reference, in log2 units (0 until it is chosen)
  int g4;                 // 4 * (lane / 16)
  // Block-causal mask inside the chunk: the chunk's own keys are [m_first, m_hi), blocks of m_block; a query sees the
  // blocks up to its own.  m_lo: the first key hidden from the wave's first query (all wave-uniform; what a lane's own
  // two queries see is worked out again in the few blocks that need it: registers are short).
  int m_first, m_lo, m_hi, m_block, q_first;
  FastDiv m_div;
};

// s[kt][qt]: scores of keys key0 + 16 kt + 4 g + i; those at or past the end of the valid keys count for nothing, nor
// do those the mask inside the chunk hides.  (One compare and one select per score: with the two conditions in one
// expression the compiler branched for every score, a microsecond per block; a query tile across a border of the mask,
// 40 such blocks, ended 45 us after the others.  3807 queries x 12 heads in blocks of 1269 against 11421 keys, three
// layer calls: 767 -> 707 us.)
template <bool kMask>
__device__ __forceinline__ void mask_block(f32x4 (&s)[2][2], const LaneConst& c, int key0, int seq) {
  if (key0 + 32 > seq) {
    const int left = seq - key0 - c.g4;
#pragma unroll
    for (int qt = 0; qt < 2; ++qt)
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int i = 0; i < 4; ++i) s[kt][qt][i] = 16 * kt + i < left ? s[kt][qt][i] : -INFINITY;
  }
  if constexpr (kMask) {
    const int n16 = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0)) & 15;
#pragma unroll
    for (int qt = 0; qt < 2; ++qt) {
      const int m_lo = c.m_first + (c.m_div(c.q_first + 16 * qt + n16) + 1) * c.m_block;
      const uint32_t first = (uint32_t)(key0 + c.g4 - m_lo), hidden = m_lo < c.m_hi ? (uint32_t)(c.m_hi - m_lo) : 0u;
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int i = 0; i < 4; ++i) s[kt][qt][i] = first + (uint32_t)(16 * kt + i) < hidden ? -INFINITY : s[kt][qt][i];
    }
  }
}

// ---------------------------------------------------------------------------
// One pipeline slot.  Keys advance in blocks of 32; slot j runs
//   S(j+1) = K_{j+1} Q^T   16 MFMAs on 8 K fragments
//   SM(j)  = exp2(scale * S - reference), packed, row sums    16 scores per lane
//   PV(j-1): O^T += V^T P^T  16 MFMAs on 8 V fragments
// together: the matrix instructions of the two products alternate (a score
// accumulator is taken up again after seven others), and the softmax
// instructions of block j are dealt out between them.  S(j) lives in s[j&1], P(j)
// in p[j&1]; the slot parity is a template argument, so this is register naming.
// ---------------------------------------------------------------------------
// Groups whose fragments are requested ahead of their use, across the border between two slots too: an LDS read takes
// as long as a group's own matrix instructions (one ahead is 1 % slower; three do not fit the registers).
constexpr int kAhead = 2;

// fragments of the first groups of the coming slot, requested by the one before it
struct Ahead {
  u32x4 k[kAhead], v[kAhead];
};

template <int kVOff>
__device__ __forceinline__ u32x4 read_v(const LaneConst& c, int g) {
  const u32x2 lo = lds_read_tr16_b64<kVOff>(c.v_addr[g]), hi = lds_read_tr16_b64<kVOff + kSub>(c.v_addr[g]);
  return __builtin_shufflevector(lo, hi, 0, 1, 2, 3);
}
template <int kKOff>
__device__ __forceinline__ u32x4 read_k(const LaneConst& c, int g) {
  return (g & 1) ? lds_read_b128<kKOff + kSub>(c.k_addr[g >> 1]) : lds_read_b128<kKOff>(c.k_addr[g >> 1]);
}

// kKNext / kVNext: where the coming slot reads; kNext false: there is none
template <bool kMask, int kPar, int kKOff, int kVOff, int kKNext, int kVNext, bool kDoS, bool kDoPV, bool kDoSM, bool kNext>
__device__ __forceinline__ void slot(const LaneConst& c, const bf16x8 (&qf)[2][4], f32x4 (&s)[2][2][2], u32x4 (&p)[2][2],
                                     f32x4 (&oacc)[8][2], f32x4 (&lacc)[2], Ahead& ahead, int key0, int key_end) {
  f32x4 (&s_cur)[2][2] = s[kPar];
  f32x4 (&s_nxt)[2][2] = s[kPar ^ 1];
  u32x4 kfrag[8 + kAhead], vfrag[8 + kAhead];
  u32x2 vlo;
#pragma unroll
  for (int g = 0; g < kAhead; ++g) {
    kfrag[g] = ahead.k[g];
    vfrag[g] = ahead.v[g];
  }

  if constexpr (kDoSM) {
    // The last, partial tile, and blocks with hidden keys.  The test value goes through an empty asm so that the
    // compiler cannot fold this uniform, rarely taken branch into the per-lane compares and hoist those.
    int masked = key0 + 32 - key_end;
    if constexpr (kMask) {
      const int into_hidden = key0 + 32 - c.m_lo < c.m_hi - key0 ? key0 + 32 - c.m_lo : c.m_hi - key0;
      masked = masked > into_hidden ? masked : into_hidden;
    }
    asm volatile("" : "+s"(masked));
    if (masked > 0) mask_block<kMask>(s_cur, c, key0, key_end);
  }
  __builtin_amdgcn_sched_barrier(0);

  // Group g = fragment pair g of the two products: four matrix instructions, two scores, and the reads of group
  // g + kAhead (the next slot's from 8 on) dealt out between them.
  constexpr int kSteps = 16;
  float scaled[kSteps], weight[kSteps];
  auto scale = [&](auto tc) {
    constexpr int t = decltype(tc)::value;       // score t = (query tile t / 8, key tile t / 4 % 2, register t % 4)
    if constexpr (kDoSM) {
      scaled[t] = __builtin_fmaf(s_cur[t / 4 % 2][t / 8][t % 4], c.c2, c.neg_ref[t / 8]);
      pin(scaled[t]);
    }
  };
  auto exponent = [&](auto tc) {
    constexpr int t = decltype(tc)::value;
    if constexpr (kDoSM) {
      weight[t] = __builtin_amdgcn_exp2f(scaled[t]);
      pin(weight[t]);
    }
  };
  auto pack = [&](auto uc) {
    constexpr int u = decltype(uc)::value;       // scores 2 u, 2 u + 1
    if constexpr (kDoSM) {
      uint32_t packed = pack_bf16x2(weight[2 * u], weight[2 * u + 1]);
      pin(packed);
      p[kPar][u / 4][u % 4] = packed;
    }
  };

  static_for<8>([&](auto gc) {
    constexpr int g = decltype(gc)::value, a = g + kAhead;
    constexpr bool kSame = a < 8;                 // the reads of group a belong to this slot
    // LDS returns in order: a fragment is there once at most the reads issued after it are in flight.  A group's first
    // product waits for its K and V reads together, until only the groups between it and a are in flight; in a slot
    // without scores V waits by itself, and group a's K read may be in flight too.
    // (Groups below kAhead were requested by the slot before, which asks for both.)
    constexpr auto k_reads = [](int x) { return x >= 8 ? (kNext ? 1 : 0) : (x < kAhead || kDoS ? 1 : 0); };
    constexpr auto v_reads = [](int x) { return x >= 8 ? (kNext ? 2 : 0) : (x < kAhead || kDoPV ? 2 : 0); };
    constexpr int kBetween = [&] {
      int sum = 0;
      for (int x = g + 1; x < a; ++x) sum += k_reads(x) + v_reads(x);
      return sum;
    }();
    constexpr int kPendingV = kBetween + k_reads(a);
    using T0 = std::integral_constant<int, 2 * g>;
    using T1 = std::integral_constant<int, 2 * g + 1>;

    if constexpr (kDoS) {
      if constexpr (g < 2) mfma_s_first<kBetween>(s_nxt[g & 1][0], kfrag[g], qf[0][g >> 1]);
      else mfma_s<kBetween>(s_nxt[g & 1][0], kfrag[g], qf[0][g >> 1]);
    }
    if constexpr (k_reads(a) > 0) kfrag[a] = read_k<kSame ? kKOff : kKNext>(c, a & 7);
    scale(T0{});
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (kDoS) {
      if constexpr (g < 2) mfma_s_first<-1>(s_nxt[g & 1][1], kfrag[g], qf[1][g >> 1]);
      else mfma_s<-1>(s_nxt[g & 1][1], kfrag[g], qf[1][g >> 1]);
    }
    if constexpr (v_reads(a) > 0) vlo = lds_read_tr16_b64<kSame ? kVOff : kVNext>(c.v_addr[a & 7]);
    exponent(T0{});
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (kDoPV) mfma_o<kDoS ? -1 : kPendingV>(oacc[g][0], vfrag[g], p[kPar ^ 1][0]);
    scale(T1{});
    if constexpr (g > 0) pack(std::integral_constant<int, (g > 0 ? g - 1 : 0)>{});
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (kDoPV) mfma_o<-1>(oacc[g][1], vfrag[g], p[kPar ^ 1][1]);
    if constexpr (v_reads(a) > 0) {
      const u32x2 vhi = lds_read_tr16_b64<(kSame ? kVOff : kVNext) + kSub>(c.v_addr[a & 7]);
      vfrag[a] = __builtin_shufflevector(vlo, vhi, 0, 1, 2, 3);
    }
    exponent(T1{});
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (kDoPV && g >= 6) mfma_row_sum(lacc[g - 6], c.ones, p[kPar ^ 1][g - 6]);
  });
  pack(std::integral_constant<int, 7>{});
  if constexpr (kNext)
#pragma unroll
    for (int g = 0; g < kAhead; ++g) {
      ahead.k[g] = kfrag[8 + g];
      ahead.v[g] = vfrag[8 + g];
    }
}

// ---------------------------------------------------------------------------
// Query tiles of five or six blocks of 32 rows.  With a wave for each block one or two SIMDs have two of them, the others one
// and half of the work, and at every tile's barrier these wait.  Here waves 0 to 3 have a block each, and waves 4 to 7 share
// the others by key: kShare = 4 of them the fifth block, 16 keys of every tile each, or kShare = 2 of them the fifth and two
// the sixth, 32 keys each.  All that share a block find the same exponent reference, so what they have summed up is simply
// added at the end, through LDS.
// A tile of five blocks 1.135 -> 0.97 us, of six 1.20 -> 1.15: 3200 queries x 12 heads against 1024 keys 27.8 -> 25.7 us, 9344
// keys 184.6 -> 158.1; 3840 x 12 against 1024 29.2 -> 28.0, 9344 197.8 -> 188.9 (same errors against 64 bits, to five digits).
// ---------------------------------------------------------------------------
template <int kShare>
__device__ __forceinline__ int wave_block(int wave) {
  if constexpr (kShare > 0) return wave < 4 ? wave : 4 + (wave - 4) / kShare;
  return wave;
}
// which of those that share its block a wave is; the first one ends up with the block's result
template <int kShare>
__device__ __forceinline__ int share_part(int wave) {
  if constexpr (kShare > 0) return wave < 4 ? 0 : (wave - 4) % kShare;
  return 0;
}

// What a sharing wave does of every tile, in the compiler's order: it has a quarter or half of the work of the wave beside it,
// and asks for a tile's K one tile ahead.  (Two statements that each waited for their LDS reads: five blocks 3 % slower, six
// 5 %.  The scores of the next tile ahead of this one's values: spills, six blocks 2 % slower.)  The LDS reads are the
// compiler's own: it knows nothing of the transfers into LDS, which are waited for at the barriers.
template <int kShare>
struct SharedBlock {
  static constexpr int kSubs = 4 / kShare;           // groups of 16 keys of a tile that are this wave's
  const LaneConst& c;
  const bf16x8 (&qf)[2][4];
  f32x4 (&oacc)[8][2];
  f32x4 lacc[2];
  u32x4 p[2];

  static __device__ __forceinline__ bf16x8 read_k(uint32_t addr) {
    return *reinterpret_cast<const __attribute__((address_space(3))) bf16x8*>(addr);
  }
  static __device__ __forceinline__ u32x2 read_v(uint32_t addr) {
    typedef __attribute__((ext_vector_type(4))) short s16x4;
    return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)addr));
  }
  // K of the groups at `off`
  template <int kCount>
  __device__ __forceinline__ void fetch_k(uint32_t off, bf16x8 (&kf)[kCount][4]) const {
#pragma unroll
    for (int j = 0; j < kCount; ++j)
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) kf[j][ks] = read_k(c.k_addr[ks] + off + j * kSub);
  }
  template <int kCount>
  __device__ __forceinline__ void scores(const bf16x8 (&kf)[kCount][4], f32x4 (&s)[kCount][2]) const {
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
#pragma unroll
      for (int j = 0; j < kCount; ++j)
#pragma unroll
        for (int qt = 0; qt < 2; ++qt)
          s[j][qt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[j][ks], qf[qt][ks], ks ? s[j][qt] : f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
  }
  // packed weights of 16 keys, key0 the first of them, into registers 2 kAt and 2 kAt + 1 of p
  template <int kAt>
  __device__ __forceinline__ void weights(f32x4 (&s)[2], int key0, int seq) {
    if (key0 + 16 > seq) {
      const int left = seq - key0 - c.g4;
#pragma unroll
      for (int qt = 0; qt < 2; ++qt)
#pragma unroll
        for (int i = 0; i < 4; ++i) s[qt][i] = i < left ? s[qt][i] : -INFINITY;
    }
#pragma unroll
    for (int qt = 0; qt < 2; ++qt)
#pragma unroll
      for (int u = 0; u < 2; ++u)
        p[qt][2 * kAt + u] = pack_bf16x2(__builtin_amdgcn_exp2f(__builtin_fmaf(s[qt][2 * u], c.c2, c.neg_ref[qt])),
                                         __builtin_amdgcn_exp2f(__builtin_fmaf(s[qt][2 * u + 1], c.c2, c.neg_ref[qt])));
  }
  // V^T of 32 keys, 16 at off_lo and 16 at off_hi
  __device__ __forceinline__ void fetch_v(uint32_t off_lo, uint32_t off_hi, bf16x8 (&vf)[8]) const {
#pragma unroll
    for (int db = 0; db < 8; ++db) {
      const u32x2 lo = read_v(c.v_addr[db] + off_lo), hi = read_v(c.v_addr[db] + off_hi);
      vf[db] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3));
    }
  }
  // Behind the next barrier transfers fill the buffers that this tile's K and V were read from.  The compiler knows nothing of
  // that, and what takes the fragments up touches no memory: it could wait for them, and use them, behind the barrier.
  // So what K was read for is in registers ahead of it, and so are V's fragments.  (Text for the check of the assembly.)
  __device__ __forceinline__ void k_has_been_read() const {
    asm volatile("; shared block: K has been read" ::"v"(p[0]), "v"(p[1]));
  }
  __device__ __forceinline__ void v_has_been_read(const bf16x8 (&vf)[8]) const {
    asm volatile("; shared block: V has been read" ::"v"(vf[0]), "v"(vf[1]), "v"(vf[2]), "v"(vf[3]), "v"(vf[4]), "v"(vf[5]), "v"(vf[6]),
                 "v"(vf[7]));
  }
  __device__ __forceinline__ void values(const bf16x8 (&vf)[8]) {
    const bf16x8 pf[2] = {__builtin_bit_cast(bf16x8, p[0]), __builtin_bit_cast(bf16x8, p[1])};
#pragma unroll
    for (int db = 0; db < 8; ++db)
#pragma unroll
      for (int qt = 0; qt < 2; ++qt) oacc[db][qt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[db], pf[qt], oacc[db][qt], 0, 0, 0);
#pragma unroll
    for (int qt = 0; qt < 2; ++qt)
      lacc[qt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, c.ones), pf[qt], lacc[qt], 0, 0, 0);
  }
};

// Conventional online softmax with a running maximum over the workgroup's key
// range, tiles double-buffered.  Every wave keeps the tiles coming and meets the
// barriers; only the waves whose fast result was unsafe redo their block.
template <bool kMask, typename KeyOf>
__device__ __forceinline__ void exact_pass(LaneConst& c, const bf16x8 (&qf)[2][4], f32x4 (&oacc)[8][2], float (&l_sum)[2],
                                           bool compute, const char* kbase, const char* vbase,
                                           uint32_t k_tok_bytes, uint32_t v_tok_bytes, const LaneFetch& f, int tile_begin,
                                           int n, int seq,
                                           KeyOf key0_of, uint32_t lds_addr0, int issuer, int lane) {
  float m_run[2] = {-INFINITY, -INFINITY}, l_run[2] = {0.f, 0.f};
  if (compute) {
#pragma unroll
    for (int qt = 0; qt < 2; ++qt) {
#pragma unroll
      for (int db = 0; db < 8; ++db) oacc[db][qt] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
  }
  auto issue = [&](int T) {
    const int key0 = key0_of(tile_begin + T);
    issue_tile(kbase, k_tok_bytes, f.chunk, f.k_row, key0, seq, lds_addr0 + kLdsBuf(T & 1), issuer, lane);
    issue_tile(vbase, v_tok_bytes, f.chunk, f.v_row, key0, seq, lds_addr0 + kLdsVBase + kLdsBuf(T & 1), issuer, lane);
  };
  __syncthreads();       // everyone is done with the buffers of the fast pass
  issue(0);
  for (int T = 0; T < n; ++T) {
    const uint32_t buf = kLdsBuf(T & 1);
    if (T + 1 < n) {
      issue(T + 1);      // into the buffer tile T - 1 left at the barrier that ended the last trip
      __builtin_amdgcn_s_waitcnt(0x0F70 | (2 * kPieces));
    } else {
      __builtin_amdgcn_s_waitcnt(0x0F70);
    }
    __syncthreads();     // tile T has landed for every wave
    if (compute) {
      for (int kb = 0; kb < 2; ++kb) {             // 32 keys at a time
        const int key0 = key0_of(tile_begin + T) + 32 * kb;
        f32x4 s[2][2];
#pragma unroll
        for (int kt = 0; kt < 2; ++kt) {
          s[kt][0] = s[kt][1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int ks = 0; ks < 4; ++ks) {
            const bf16x8 kf = lds_read_b128_now(c.k_addr[ks] + buf + kb * kHalf + kt * kSub);
#pragma unroll
            for (int qt = 0; qt < 2; ++qt) s[kt][qt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[qt][ks], s[kt][qt], 0, 0, 0);
          }
        }
        if (key0 + 32 > seq || (kMask && key0 + 32 > c.m_lo && key0 < c.m_hi)) mask_block<kMask>(s, c, key0, seq);
        u32x4 pf[2];
#pragma unroll
        for (int qt = 0; qt < 2; ++qt) {
          float m_new = m_run[qt];
#pragma unroll
          for (int i = 0; i < 4; ++i) m_new = fmaxf(m_new, fmaxf(s[0][qt][i], s[1][qt][i]));
          m_new = fmaxf(m_run[qt], col_max(m_new));
          // -inf only while every key so far was masked for this query: then nothing has been summed yet
          const float alpha = m_new == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f((m_run[qt] - m_new) * c.c2);
          const float mc = m_new == -INFINITY ? 0.0f : m_new * c.c2;
          m_run[qt] = m_new;
          float sum = 0.f;
#pragma unroll
          for (int kt = 0; kt < 2; ++kt)
#pragma unroll
            for (int i = 0; i < 4; i += 2) {
              const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[kt][qt][i], c.c2, -mc));
              const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[kt][qt][i + 1], c.c2, -mc));
              sum += p0 + p1;
              pf[qt][2 * kt + i / 2] = pack_bf16x2(p0, p1);
            }
          l_run[qt] = l_run[qt] * alpha + sum;
#pragma unroll
          for (int db = 0; db < 8; ++db)
#pragma unroll
            for (int i = 0; i < 4; ++i) oacc[db][qt][i] *= alpha;
        }
#pragma unroll
        for (int db = 0; db < 8; ++db) {
          const uint32_t addr = c.v_addr[db] + buf + kb * kHalf;
          const bf16x8 vf = lds_read_tr16_b64x2_now(addr, addr + kSub);
#pragma unroll
          for (int qt = 0; qt < 2; ++qt)
            oacc[db][qt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, __builtin_bit_cast(bf16x8, pf[qt]), oacc[db][qt], 0, 0, 0);
        }
      }
    }
    __syncthreads();     // tile T's buffer is free for tile T + 2
  }
  if (compute)
#pragma unroll
    for (int qt = 0; qt < 2; ++qt) {
      l_sum[qt] = col_sum(l_run[qt]);
      c.neg_ref[qt] = -m_run[qt] * c.c2;
    }
}

// Tiles of 64 keys that a query tile's workgroup has to stream of `seq` keys: with the mask inside the chunk those that
// are hidden from every query of the workgroup (from the last one, that is) are left out, and key ranges are cut from
// what is left.
template <bool kMask>
__device__ __forceinline__ TileSpan tile_list(late_args<AttnKernelArgs>& a, int q_end, int chunk_start, int seq) {
  return visible_tiles(kKTile, seq, q_end - 1, a.q_tokens, chunk_start, kMask ? a.mask_block_tokens : 0,
                       read_div(a.div_mask_block));
}

__device__ __forceinline__ int row_keys(late_args<AttnKernelArgs>& a, int row) {
  int seq = a.seq_lens ? a.seq_lens[row] : a.max_seq_len;
  seq = seq < a.max_seq_len ? seq : a.max_seq_len;
  return seq < 0 ? 0 : seq;
}

// The row behind the last one of query tile `qtile`, of tiles of `rows` rows
__device__ __forceinline__ int tile_end_row(late_args<AttnKernelArgs>& a, int qtile, int rows) {
  const int end = (qtile + 1) * rows;
  return end < a.q_tokens ? end : a.q_tokens;
}

// A word of memory looked at by thread 0 before the range's last matrix instructions, for the time behind them.
struct Peek {
  const int32_t* word;       // null: nothing to look at
  int want;
  lds_int* found;            // was it that?  (for all threads, once stream_range is back)
  __device__ __forceinline__ int begin() const {
    return word && threadIdx.x == 0 ? __hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0;
  }
  __device__ __forceinline__ void end(int seen) const {
    if (word && threadIdx.x == 0) *found = seen == want;
  }
};
struct NoPeek {
  __device__ __forceinline__ int begin() const { return 0; }
  __device__ __forceinline__ void end(int) const {}
};

// The workgroup's query rows, q_first .. q_end - 1, 32 a wave, against entries [tile_begin, tile_end) of a tile list, the first
// key of entry t being key0_of(t): sums of the weighted values
// (oacc), the queries' row sums (l_sum) and the exponent references both are relative to (c.neg_ref).  Behind it every
// wave is done with the tile buffers.
template <bool kMask, int kFirstIssuer = 0, int kShare = 0, typename KeyOf, typename LookAt = NoPeek>
__device__ __forceinline__ void stream_range(late_args<AttnKernelArgs>& a, lds_char* lds, int q_first, int q_end, int head, int row, int seq,
                                             KeyOf key0_of, int tile_begin, int tile_end, LaneConst& c,
                                             f32x4 (&oacc)[8][2], float (&l_sum)[2], LookAt look = LookAt()) {
  lds_int* flags = reinterpret_cast<lds_int*>(lds + kLdsFlags);
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));      // (what is derived from it is worked out per range, not held across them)
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wave_u = __builtin_amdgcn_readfirstlane(wave);
  const int issuer = wave_u - kFirstIssuer;
  const int n16 = lane & 15, g = lane >> 4;
  const int n = tile_end - tile_begin;       // tiles this workgroup streams

  const uint32_t lds_addr0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)lds);
  const char* kbase = uniform_pointer(a.k + row * a.k_st.row + head * a.k_st.head);
  const char* vbase = uniform_pointer(a.v + row * a.v_st.row + head * a.v_st.head);
  const uint32_t k_tok_bytes = (uint32_t)(a.k_st.token * 2);
  const uint32_t v_tok_bytes = (uint32_t)(a.v_st.token * 2);

  LaneFetch f;
  f.chunk = (uint32_t)(n16 ^ g << 1) << 4;
  f.k_row = g * k_tok_bytes;
  f.v_row = g * v_tok_bytes;
  // T is the tile index inside this workgroup's range
  auto issue_k = [&](int T, int buf) {
    issue_tile(kbase, k_tok_bytes, f.chunk, f.k_row, key0_of(tile_begin + T), seq, lds_addr0 + kLdsBuf(buf), issuer, lane);
  };
  auto issue_v = [&](int T, int buf) {
    issue_tile(vbase, v_tok_bytes, f.chunk, f.v_row, key0_of(tile_begin + T), seq, lds_addr0 + kLdsVBase + kLdsBuf(buf), issuer, lane);
  };

  // ---- this lane's two query rows, and the first tiles ------------------------
  // Loads return in the order they were issued.  A query that arrives rotated is
  // asked for ahead of the first tiles, so that both come back in one trip to
  // memory; one that is to be rotated here needs several trips for the rotation
  // table and is fetched behind the tiles the first two slots need, the rest of
  // the look-ahead after it.
  const int q_row = q_first + wave_block<kShare>(wave) * kQBlock + n16;      // and q_row + 16
  bf16x8 qf[2][4];
  const uint16_t* q_ptr[2];
  int q_tok[2];
#pragma unroll
  for (int qt = 0; qt < 2; ++qt) {
    q_tok[qt] = q_row + 16 * qt < a.q_tokens ? q_row + 16 * qt : a.q_tokens - 1;
    q_ptr[qt] = a.q + row * a.q_st.row + (int64_t)q_tok[qt] * a.q_st.token + head * a.q_st.head + 8 * g;
  }
  if (a.freqs == nullptr) {
#pragma unroll
    for (int qt = 0; qt < 2; ++qt)
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) qf[qt][ks] = *reinterpret_cast<const bf16x8*>(q_ptr[qt] + 32 * ks);
  }
  if (n > 0) {
    issue_k(0, 0);
    issue_v(0, 0);
    issue_k(n > 1 ? 1 : n - 1, 1);
    // V buffer kStages - 1 stands in for "V tile -1" in the first slot, where it meets the
    // all-zero P(-1): any finite values do, so it is cleared (two 16-byte stores per lane)
    {
      const u32x4 zero = {0u, 0u, 0u, 0u};
      lds_char* v_last = lds + kLdsVBase + kLdsBuf(kStages - 1);
#pragma unroll
      for (int j = 0; j < kTileBytes / 16 / kThreads; ++j)
        *reinterpret_cast<__attribute__((address_space(3))) u32x4*>(v_last + (j * kThreads + tid) * 16) = zero;
    }
    if (tid == 0) flags[0] = 0;       // "a wave found an unsafe row sum": read behind the barrier that ends the loop
  }

  if (a.freqs != nullptr) {
    QueryRope rope;
    rope.freqs = a.freqs;
    rope.grid_w = a.grid_w; rope.frame_tokens = a.frame_tokens; rope.split_t = a.split_t; rope.split_h = a.split_h;
    rope.start_frame = row_start_frame(a, row);
    rope.norm_w = a.q_norm_w ? a.q_norm_w + head * kD + 8 * g : nullptr;
#pragma unroll
    for (int qt = 0; qt < 2; ++qt) {
      rope.inv_rms = a.q_norm_w ? a.q_inv_rms[(int64_t)row * a.q_tokens + q_tok[qt]] : 1.0f;
      load_query(rope, q_ptr[qt], q_tok[qt], g, qf[qt]);
    }
  }
  // the value is (re)defined in the register class every later use names, so it is never copied back and forth
#pragma unroll
  for (int qt = 0; qt < 2; ++qt)
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) asm volatile("" : "+a"(qf[qt][ks]));
  if (n > 0) {
    // every buffer a slot may read starts with real (finite) data, also where the tile does not exist
    issue_v(n > 1 ? 1 : n - 1, 1);
    issue_k(n > 2 ? 2 : n - 1, 2);
    issue_v(n > 2 ? 2 : n - 1, 2);
    issue_k(n > 3 ? 3 : n - 1, 3);
  }

  // ---- per-lane LDS read addresses ------------------------------------------
  c.ones = u32x4{0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u};
  asm volatile("" : "+a"(c.ones));      // (one register copy for the whole kernel: a constant formed in front of an asm MFMA is read too early)
  c.c2 = a.scale_log2;
  c.neg_ref[0] = c.neg_ref[1] = 0.f;
  c.g4 = 4 * g;
  if constexpr (kMask) {
    c.m_block = a.mask_block_tokens;
    c.m_div = read_div(a.div_mask_block);
    c.q_first = q_first + wave_u * kQBlock;
    c.m_first = __builtin_amdgcn_readfirstlane(row_chunk_start(a, row));
    c.m_hi = c.m_first + a.q_tokens;
    c.m_lo = __builtin_amdgcn_readfirstlane(c.m_first + (c.m_div(c.q_first) + 1) * c.m_block);
  }
  {
    // K (A operand): key = lane%16 of the 16-key tile, chunk = 4*ks + g
    const int base = n16 * 256 + ((g ^ swz16(n16)) << 4);
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) c.k_addr[ks] = lds_addr0 + (uint32_t)(base ^ (ks << 6));
    // V^T (A operand) through the transposing read: in each group of 16 lanes, lane i supplies the address of
    // key 4 g + i / 4, 8 bytes at d-offset 4 * (i % 4); it receives d = i, keys 4 g .. 4 g + 3
    const int r = 4 * g + (n16 >> 2);
    const int vbase_off = r * 256 + ((((n16 & 3) >> 1) ^ swz16(r)) << 4) + (n16 & 1) * 8;
#pragma unroll
    for (int db = 0; db < 8; ++db) c.v_addr[db] = lds_addr0 + kLdsVBase + (uint32_t)(vbase_off ^ (db << 5));
  }

#pragma unroll
  for (int db = 0; db < 8; ++db) oacc[db][0] = oacc[db][1] = f32x4{0.f, 0.f, 0.f, 0.f};
  f32x4 s[2][2][2];
  u32x4 p[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      p[i][j] = u32x4{0u, 0u, 0u, 0u};
      s[i][j][0] = s[i][j][1] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
  f32x4 lacc[2];                     // row sums, the same in every register and lane of the column
  lacc[0] = lacc[1] = f32x4{0.f, 0.f, 0.f, 0.f};
  l_sum[0] = l_sum[1] = 0.f;
  bool unsafe = false;

  // Tile T (64 keys) = blocks 2T, 2T+1, in K / V buffers T % 4.  Slot 2T needs
  // K tile T (second half) and V tile T-1 (second half); slot 2T+1 needs K tile
  // T+1 (first half) and V tile T (first half).  After slot 2T the buffers of
  // K tile T and V tile T-1 are free: that is where the one barrier per tile
  // sits, followed by the requests for K tile T+4 and V tile T+3.  The wait before
  // the barrier leaves the newest 2 * kPieces transfers of a wave (K tile T+3,
  // V tile T+2) in flight, so K tile T+2 and V tile T+1 have landed: slot 2T+2
  // may request slot 2T+3's first fragments ahead of barrier T+1.  Every tile runs
  // the same code; scores of keys at or beyond the end of the range are masked to
  // -inf, so their weights are exact zeros against whatever finite data the
  // buffers still hold.
  const int key_end = seq;
  Ahead ahead;
  auto land = [&](int T) {           // what must have landed by the barrier of tile T has
    if (T + 3 < n) {
      __builtin_amdgcn_s_waitcnt(0x0F70 | (2 * kPieces));   // vmcnt: one K and one V tile's worth per wave
    } else {
      __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0)
    }
    asm volatile("s_barrier" ::: "memory");
  };
  auto do_tile = [&](auto buf_c, int T) {
    constexpr int kB = decltype(buf_c)::value;              // T % kStages
    constexpr int kBNext = (kB + 1) % kStages, kBPrev = (kB + kStages - 1) % kStages;
    const int key0 = key0_of(tile_begin + T);
    slot<kMask, 0, kLdsBuf(kB) + kHalf, kLdsBuf(kBPrev) + kHalf, kLdsBuf(kBNext), kLdsBuf(kB), true, true, true, true>(
        c, qf, s, p, oacc, lacc, ahead, key0, key_end);
    land(T);
    if (T + 4 < n) issue_k(T + 4, kB);
    if (T + 3 < n) issue_v(T + 3, kBPrev);
    slot<kMask, 1, kLdsBuf(kBNext), kLdsBuf(kB), kLdsBuf(kBNext) + kHalf, kLdsBuf(kB) + kHalf, true, true, true, true>(
        c, qf, s, p, oacc, lacc, ahead, key0 + 32, key_end);
  };
  using B0 = std::integral_constant<int, 0>;
  using B1 = std::integral_constant<int, 1>;
  using B2 = std::integral_constant<int, 2>;
  using B3 = std::integral_constant<int, 3>;

  const bool idle = __builtin_amdgcn_readfirstlane(q_first + wave_block<kShare>(wave) * kQBlock >= q_end);       // no query row is this wave's
  // Behind the barrier of the last tile the K buffers are free (what the waves with a block of their own still read of them is
  // a tile that does not exist): there the waves that share a block leave their sums.
  auto parts_lie_in_lds = [&] {
    if constexpr (kShare > 0) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  };
  int seen = 0;
  if (n > 0) {
    // K tiles 0 and 1 and V tile 0 have landed once at most the four tiles requested behind them are in flight
    if ((unsigned)issuer < kIssuers) {
      __builtin_amdgcn_s_waitcnt(0x4070);   // vmcnt(16) = 4 * kPieces, and lgkmcnt(0) for the LDS clear
      static_assert(4 * kPieces == 16, "the wait above");
    } else {
      __builtin_amdgcn_s_waitcnt(0x0070);
    }
    __syncthreads();
    if (idle) {
      // No query row of this wave exists: it moves its share of every K / V tile and meets the others at every
      // barrier, but issues no LDS read, MFMA or softmax instruction (work on rows nobody reads would only lower
      // the clock for the rest).
      for (int T = 0; T < n; ++T) {
        land(T);
        if (T + 4 < n) issue_k(T + 4, T % kStages);
        if (T + 3 < n) issue_v(T + 3, (T + 3) % kStages);
      }
      parts_lie_in_lds();
    } else if (kShare > 0 && wave_u >= 4) {
      // (between the barriers of tiles T - 1 and T the K tiles T and T + 1 and the V tiles T - 1 and T lie in LDS)
      if constexpr (kShare > 0) {
        const int part = share_part<kShare>(wave_u);
        SharedBlock<kShare> b{c, qf, oacc};
        b.lacc[0] = b.lacc[1] = f32x4{0.f, 0.f, 0.f, 0.f};
        f32x4 first[2][2];
        {
          bf16x8 kf[2][4];
          b.template fetch_k<2>(0, kf);
          b.template scores<2>(kf, first);
        }
#pragma unroll
        for (int qt = 0; qt < 2; ++qt) {
          float ref = first[0][qt][0];
#pragma unroll
          for (int i = 0; i < 4; ++i) ref = vmax(ref, vmax(first[0][qt][i], first[1][qt][i]));
          ref = col_max(ref);
          ref = (ref > -0x1p120f && ref < 0x1p120f) ? ref : 0.f;      // also false for NaN
          c.neg_ref[qt] = -ref * c.c2;
        }
        const uint32_t mine = part * (SharedBlock<kShare>::kSubs * kSub);
        auto offset = [&](int T) { return (uint32_t)(T % kStages) * kTileBytes + mine; };
        auto first_key = [&](int T) { return key0_of(tile_begin + T) + part * (SharedBlock<kShare>::kSubs * 16); };
        auto end_tile = [&](int T) {
          land(T);
          if (T + 4 < n) issue_k(T + 4, T % kStages);
          if (T + 3 < n) issue_v(T + 3, (T + 3) % kStages);
        };
        constexpr int kSubs = SharedBlock<kShare>::kSubs;
        bf16x8 kf[kSubs][4], vf[8];
        f32x4 s[kSubs][2];
        b.template fetch_k<kSubs>(offset(0), kf);
        if constexpr (kShare == 2) {
          for (int T = 0; T < n; ++T) {
            const uint32_t off = offset(T);
            b.template scores<kSubs>(kf, s);
            b.fetch_v(off, off + kSub, vf);
            b.template fetch_k<kSubs>(offset(T + 1), kf);
            b.template weights<0>(s[0], first_key(T), seq);
            b.template weights<1>(s[1], first_key(T) + 16, seq);
            b.values(vf);
            b.k_has_been_read();
            b.v_has_been_read(vf);
            end_tile(T);
          }
        } else {
          // 16 keys of two tiles make one product; a last tile without a second one has zeros there, weights and values (its own
          // values again could hold an infinity, and that times zero is no number)
          for (int T = 0; T < n; T += 2) {
            const uint32_t off = offset(T);
            uint32_t off2 = off;
            b.template scores<kSubs>(kf, s);
            b.template fetch_k<kSubs>(offset(T + 1), kf);
            b.template weights<0>(s[0], first_key(T), seq);
            b.k_has_been_read();
            if (T + 1 < n) {
              end_tile(T);
              off2 = offset(T + 1);
              b.template scores<kSubs>(kf, s);
              b.template fetch_k<kSubs>(offset(T + 2), kf);
              b.fetch_v(off, off2, vf);
              b.template weights<1>(s[0], first_key(T + 1), seq);
            } else {
              b.p[0][2] = b.p[0][3] = b.p[1][2] = b.p[1][3] = 0u;
              b.fetch_v(off, off2, vf);
#pragma unroll
              for (int db = 0; db < 8; ++db) vf[db] = __builtin_shufflevector(vf[db], bf16x8{}, 0, 1, 2, 3, 8, 9, 10, 11);
            }
            b.values(vf);
            b.k_has_been_read();
            b.v_has_been_read(vf);
            end_tile(T + 1 < n ? T + 1 : T);
          }
        }
        // all but the first leave their sums, and the first adds them up in the waves' order
        auto place = [&](int of_wave, int j) {
          return reinterpret_cast<__attribute__((address_space(3))) f32x4*>(lds + (of_wave - 4) * kTileBytes + j * 1024 + lane * 16);
        };
        auto place_l = [&](int of_wave) {
          return reinterpret_cast<__attribute__((address_space(3))) float*>(lds + kLdsBytes + (of_wave - 4) * 512 + lane * 8);
        };
        if (part != 0) {
#pragma unroll
          for (int db = 0; db < 8; ++db)
#pragma unroll
            for (int qt = 0; qt < 2; ++qt) *place(wave_u, 2 * db + qt) = oacc[db][qt];
#pragma unroll
          for (int qt = 0; qt < 2; ++qt) place_l(wave_u)[qt] = b.lacc[qt][0];
        }
        parts_lie_in_lds();
        if (part == 0) {
          l_sum[0] = b.lacc[0][0];
          l_sum[1] = b.lacc[1][0];
#pragma unroll
          for (int w = 1; w < kShare; ++w) {
#pragma unroll
            for (int db = 0; db < 8; ++db)
#pragma unroll
              for (int qt = 0; qt < 2; ++qt) oacc[db][qt] += *place(wave_u + w, 2 * db + qt);
#pragma unroll
            for (int qt = 0; qt < 2; ++qt) l_sum[qt] += place_l(wave_u + w)[qt];
          }
          const bool ok = l_sum[0] >= 0x1p-100f && l_sum[0] <= 0x1p100f && l_sum[1] >= 0x1p-100f && l_sum[1] <= 0x1p100f;
          unsafe = __builtin_amdgcn_ballot_w64(!ok) != 0;
        }
      }
    } else {
      // S(0) alone fills the pipeline, and its largest score becomes the query's exponent reference
#pragma unroll
      for (int g = 0; g < kAhead; ++g) {
        ahead.k[g] = read_k<kLdsBuf(0)>(c, g);
        ahead.v[g] = read_v<kLdsBuf(kStages - 1) + kHalf>(c, g);
      }
      slot<kMask, 1, kLdsBuf(0), kLdsBuf(kStages - 1) + kHalf, kLdsBuf(0) + kHalf, kLdsBuf(kStages - 1) + kHalf, true, false, false, true>(
          c, qf, s, p, oacc, lacc, ahead, 0, key_end);
      mfma_drain<1>(oacc, s);
#pragma unroll
      for (int qt = 0; qt < 2; ++qt) {
        float ref = s[0][0][qt][0];
#pragma unroll
        for (int i = 0; i < 4; ++i) ref = vmax(ref, vmax(s[0][0][qt][i], s[0][1][qt][i]));
        ref = col_max(ref);
        ref = (ref > -0x1p120f && ref < 0x1p120f) ? ref : 0.f;      // also false for NaN
        c.neg_ref[qt] = -ref * c.c2;
      }
      // Four tiles per trip, one per buffer; the last trip stops after the last
      // real tile.  The skipped tiles sit behind uniform branches that no value
      // is changed on, so the accumulators stay where they are on either way.
      for (int T = 0; T < n; T += 4) {
        do_tile(B0{}, T);
        if (T + 1 < n) {
          do_tile(B1{}, T + 1);
          if (T + 2 < n) {
            do_tile(B2{}, T + 2);
            if (T + 3 < n) do_tile(B3{}, T + 3);
          }
        }
      }
      parts_lie_in_lds();
      // PV of the last block (odd -> p[1], second half of the last tile's V
      // buffer) empties the pipeline.  The code addresses V buffer kStages - 1; the lane
      // addresses are moved when the last tile sits in another buffer.
      {
        // (what was requested for a slot that does not come - its K fragment - must land before its registers are
        // used for anything else)
        asm volatile("s_waitcnt lgkmcnt(0)");
#pragma unroll
        for (int g = 0; g < kAhead; ++g) asm volatile("" : "+v"(ahead.k[g]), "+v"(ahead.v[g]));
        seen = look.begin();
        // (in place and back again: a copy of the addresses does not fit the registers)
        const uint32_t shift = (uint32_t)(((n - 1) % kStages - (kStages - 1)) * kTileBytes);
#pragma unroll
        for (int db = 0; db < 8; ++db) c.v_addr[db] += shift;
        slot<kMask, 0, 0, kLdsBuf(kStages - 1) + kHalf, 0, 0, false, true, false, false>(
            c, qf, s, p, oacc, lacc, ahead, 0, key_end);
#pragma unroll
        for (int db = 0; db < 8; ++db) c.v_addr[db] -= shift;
      }
      mfma_drain<0>(oacc, s);
      asm volatile("" : "+a"(lacc[0]), "+a"(lacc[1]));
      l_sum[0] = lacc[0][0];
      l_sum[1] = lacc[1][0];
      // Checked once, after the last tile: a sum that overflowed stays inf or NaN, one
      // that underflowed stays tiny.
      bool ok = true;
#pragma unroll
      for (int qt = 0; qt < 2; ++qt) {
        bool fine = l_sum[qt] >= 0x1p-100f && l_sum[qt] <= 0x1p100f;
        if constexpr (kMask) {
          // (zero is right where every key of this range is hidden from the query; a range that goes on from the
          // last key to the first one holds some that are not)
          const int m_lo = c.m_first + (c.m_div(q_row + 16 * qt) + 1) * c.m_block;
          const int last = key0_of(tile_end - 1) + kKTile;
          fine |= l_sum[qt] == 0.f && key0_of(tile_begin) >= m_lo && (last < seq ? last : seq) <= c.m_hi && last > key0_of(tile_begin);
        }
        ok &= fine;
      }
      unsafe = __builtin_amdgcn_ballot_w64(!ok) != 0;
    }

    // Did any wave of the workgroup see an unsafe row sum?  One barrier: behind it every wave is done
    // with the K / V buffers (the epilogue stages its output there) and the flag, cleared before the
    // loop, holds every wave's word.
    if (unsafe && lane == 0) flags[0] = 1;
    look.end(seen);
    __syncthreads();
    const int redo = flags[0];
    if (redo)
      exact_pass<kMask>(c, qf, oacc, l_sum, unsafe, kbase, vbase, k_tok_bytes, v_tok_bytes, f, tile_begin, n,
                 seq, key0_of, lds_addr0, issuer, lane);
  }
}

// A lane holds two query rows' values scattered over the 128 dims.  Every wave
// stages its 32-row block in its own 8 KB of the (now idle) LDS, 16-byte
// chunks XOR-swizzled by row, and writes whole rows of 256 bytes.  LDS
// operations of one wave complete in order, so the block needs no barrier of
// its own.
__device__ __forceinline__ void stage_out(lds_char* stage, int lane, int db, const f32x4 (&o)[2], const float (&inv)[2]) {
  const int n16 = lane & 15, g = lane >> 4;
#pragma unroll
  for (int qt = 0; qt < 2; ++qt) {
    u32x2 x;
    x[0] = pack_bf16x2(o[qt][0] * inv[qt], o[qt][1] * inv[qt]);
    x[1] = pack_bf16x2(o[qt][2] * inv[qt], o[qt][3] * inv[qt]);
    const int r = 16 * qt + n16, chunk = 2 * db + (g >> 1);
    *reinterpret_cast<__attribute__((address_space(3))) u32x2*>(stage + r * 256 + ((chunk ^ n16) << 4) + (g & 1) * 8) = x;
  }
}
__device__ __forceinline__ void write_block(late_args<AttnKernelArgs>& a, lds_char* stage, int q0, int head, int row, int lane) {
  const int n16 = lane & 15, g = lane >> 4;
  uint16_t* dst = a.out + row * a.o_st.row + head * a.o_st.head + (int64_t)q0 * a.o_st.token;
#pragma unroll
  for (int it = 0; it < 8; ++it) {
    const int rr = 4 * it + g;
    const u32x4 x = *reinterpret_cast<__attribute__((address_space(3))) const u32x4*>(
        stage + rr * 256 + ((n16 ^ (rr & 15)) << 4));
    if (q0 + rr < a.q_tokens) *reinterpret_cast<u32x4*>(dst + rr * a.o_st.token + n16 * 8) = x;
  }
}

}  // namespace m16
}  // namespace attn
}  // namespace sdv2

#endif  // SDV2KV_ATTN_M16_DEVICE_H
