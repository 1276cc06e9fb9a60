// Attention of a chunk's queries against an fp32 ring KV cache, computed in
// fp32 throughout, for gfx950 (MI355X).
//
// Stands in for what the reference computes on fp32 tensors at
// models/wan/causal_model.py:111-157 (attention_with_kvcache_fallback: scaled
// dot product attention of q against k_cache[:, :seq_len], no mask inside the
// chunk) - the configuration the reference itself can run on a CPU.  Products
// and sums are fp32 (the fp32 matrix instruction multiplies and adds in fp32),
// the softmax keeps a running maximum per query row, and nothing is rounded
// below fp32 anywhere.
//
// What bounds it: the fp32 matrix pipe, 64 flop per cycle and SIMD (157 TFLOP/s
// nominal; the vendor's fp32 GEMM reaches 154).  One v_mfma_f32_32x32x2_f32
// takes 64 cycles and one 4-byte register per lane and operand, so LDS reads
// (one 16-byte read per lane feeds four of them), the softmax (some 300 vector
// instructions per 128 matrix instructions) and the tile loads all fit beside
// it; what has to be got right is that every SIMD has two waves and that the
// grid packs evenly onto the CUs.
//
// Work decomposition: workgroup = 4 waves = 128 query rows of one (row, head),
// wave w owns the 32-row block 32 w..32 w + 31, two workgroups per CU (64 KB of
// LDS each): one wave's softmax and barriers run under the other's matrix
// instructions.  Keys stream through LDS 32 at a time, double-buffered, by
// transfers that take no register (as the 32 registers of a tile on its way are
// what the two-level sums below live in).  One or two 32-row blocks past the last
// whole 128 rows would keep one or two of the four SIMDs busy for a workgroup's
// time: there the four waves deal out the keys of the same blocks among themselves
// and meet in LDS.
//
// The call's items (query tile of a (row, head), rest) lie end to end, as long as
// their key tiles take, and are cut into equal shares for two workgroups on every CU
// (f32_plan, attn_f32_plan.h): with key ranges of one length for all, 1560 x 12
// queries were 468 workgroups for 512 places, 36 of them for 24 rows.  Each piece
// leaves its unnormalised output, maximum and sum in the workspace, and the
// workgroup that draws the last ticket of its item combines them in the order of
// the keys, so the result does not depend on which one that is.  A caller without
// a workspace gets one workgroup per item.
//
// Sums are kept in two levels: a tile's weights, and its weights times values, are
// summed from zero and added to the long sums once a tile, in the multiplication
// that makes those relative to the new maximum.  A piece may be longer than it was
// (an item of 225 tiles is walked whole where it was cut in three), and the error
// against 64 bits is half of what it was all the same: rms 1.9e-8 -> 0.9e-8 on
// 1560 queries against 6240 keys, 1.5e-8 -> 0.9e-8 on 3600 against 7200.
//
// Matrix layout (D = A(32x2) * B(2x32) + C; the two k values of an instruction
// sit in the two halves of the wave):
//   S^T = K Q^T    A = K: lane holds key lane % 32; B = Q: lane holds query
//                  lane % 32.  The contraction may run over the head dimensions
//                  in any order: step (t, e) takes 8 t + e in the lower half
//                  and 8 t + 4 + e in the upper one, so a lane's operands of
//                  four steps are 16 contiguous bytes.
//   O^T = V^T P^T  B = P^T is the S^T accumulator register as it stands
//                  (register 4 g + j: keys 8 g + j and 8 g + 4 + j in the two
//                  halves); A = V of those two keys.  Accumulator db collects the
//                  dimensions 64 (db / 2) + 2 m + db % 2, m = 0..31, so one 8-byte
//                  read of V feeds two accumulators and two of a lane's results are
//                  16 contiguous bytes of an output row.
//
// Against equal key ranges, same box: 1560 queries x 12 heads against 6240 keys 554 ->
// 463 us (108 -> 129 TFLOP/s), 9360 keys 812 -> 685, 2 x 1740 against 8700 1468 -> 1405,
// 780 x 40 against 4000 649 -> 503, 4 x 29 x 40 against 19282 993 -> 713; 60 shapes of
// 20 to 4700 queries 10 % less on average, calls of some 30 us within a microsecond of
// what they took, but for one of less than 64 rows against 500 keys (27 -> 31).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>

#include "sdv2kv.h"
#include "sdv2kv_profile.h"
#include "sdv2kv_internal.h"
#include "attn_device.h"
#include "attn_f32_plan.h"

namespace {

using sdv2::attn::EvenPlanF32;
using sdv2::attn::FastDiv;
using sdv2::attn::ItemKind;
using sdv2::attn::dma16;
using sdv2::attn::first_workgroup;
using sdv2::attn::kWholeTileF32;
using sdv2::attn::last_workgroup;
using sdv2::attn::late_args;
using sdv2::attn::read_div;
using sdv2::attn::read_late;
using sdv2::attn::rest_kind_f32;

typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(2))) float f32x2;

constexpr int kD = SDV2_HEAD_DIM;     // 128
constexpr int kWaves = 4;
constexpr int kThreads = kWaves * 64;
constexpr int kQBlock = 32;           // query rows per wave
constexpr int kQTile = kWaves * kQBlock;
constexpr int kKeys = 32;             // keys per tile
// Tiles come from memory without a register: 16-byte chunk c of row r of K lies at position c ^ r % 16, so that eight
// lanes' reads of "their" key rows never meet in a bank.  V is read along a row and lies as it is.
constexpr int kTileBytes = kKeys * kD * 4;            // 16 KB
constexpr int kLdsBytes = 4 * kTileBytes + 16;        // two buffers of K, two of V, one flag word
constexpr int kMaxDevices = 64;
constexpr int kCus = 256;
constexpr float kLog2e = 1.4426950408889634f;
// Ticket words at the head of the workspace, as in the bf16 kernel (one
// workspace serves both): a fixed region, all zero between calls.
constexpr int kMaxTickets = 16384;
constexpr int kMostPieces = 16;                       // that an item is cut into, or about that
constexpr int kBlockFloats = kQBlock * kD;            // a block's partial output

struct AttnF32Args {
  const float* q;
  const float* k;
  const float* v;
  float* out;
  const int32_t* seq_lens;
  sdv2_stride3 q_st, k_st, v_st, o_st;
  int32_t rows, q_tokens, heads, max_seq_len;
  float scale_log2;            // softmax_scale * log2(e)
  int32_t mask_block_tokens;
  EvenPlanF32 plan;
  FastDiv div_items, div_heads;                  // by the items of a (row, head); by heads
  int32_t* tickets;            // [row][head][item]
  // two places for each workgroup: the rest or the middle of an item, and the start of one that others go on with
  float* part_o;               // [place][wave][16 KB]: sums of weights times values, in register order
  float* part_m;               // [place][wave][32]: running maximum, log2 units
  float* part_l;               // [place][wave][32]: sum of weights
  sdv2::ChunkStarts chunk_starts;   // with the mask inside the chunk
};

__device__ __forceinline__ float half_max(float x) {
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float half_sum(float x) {
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Partial results cross XCDs: device-coherent accesses, ordered by the ticket
// (stores are acknowledged before it is drawn).
__device__ __forceinline__ void store_coherent(float* p, float x) {
  __hip_atomic_store(reinterpret_cast<uint32_t*>(p), __float_as_uint(x), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float load_coherent(const float* p) {
  return __uint_as_float(
      __hip_atomic_load(reinterpret_cast<const uint32_t*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}
// (a store of 16 bytes reads its data up to two cycles after its issue, which the compiler does not know of a store
// inside a statement: what comes behind may be an instruction that writes those registers)
__device__ __forceinline__ void store_coherent16(float* p, const f32x4& x) {
  asm volatile("global_store_dwordx4 %0, %1, off sc1\n\ts_nop 1" : : "v"(p), "v"(x) : "memory");
}
// eight 16-byte pieces 1 KB apart, issued and waited for in one statement (in
// between the compiler must not touch the destination registers)
__device__ __forceinline__ void load_coherent_x8(const float* p, f32x4 (&w)[8]) {
  asm volatile(
      "global_load_dwordx4 %0, %8, off sc1\n\t"
      "global_load_dwordx4 %1, %8, off offset:1024 sc1\n\t"
      "global_load_dwordx4 %2, %8, off offset:2048 sc1\n\t"
      "global_load_dwordx4 %3, %8, off offset:3072 sc1\n\t"
      "global_load_dwordx4 %4, %9, off sc1\n\t"
      "global_load_dwordx4 %5, %9, off offset:1024 sc1\n\t"
      "global_load_dwordx4 %6, %9, off offset:2048 sc1\n\t"
      "global_load_dwordx4 %7, %9, off offset:3072 sc1\n\t"
      "s_waitcnt vmcnt(0)"
      : "=&v"(w[0]), "=&v"(w[1]), "=&v"(w[2]), "=&v"(w[3]), "=&v"(w[4]), "=&v"(w[5]), "=&v"(w[6]), "=&v"(w[7])
      : "v"(p), "v"(p + 1024)
      : "memory");
}

// as dma16, from an address of this lane's
__device__ __forceinline__ void dma16_far(const char* p, uint32_t lds_dst) {
  asm volatile(
      "s_mov_b32 m0, %1\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %0, off"
      :
      : "v"(p), "s"(lds_dst)
      : "memory");
}

// One item of the work: 128 query rows of a (row, head), or what is left past the last whole 128.
struct Piece {
  int row, head, item;         // query rows item * 128 .. of (row, head)
  int tile0, tile1;            // key tiles
};

// What the waves of a workgroup hold of a piece: wave w's block of 32 queries, the lane's columns.
struct Sums {
  f32x16 o[4];                 // sums of weights times values
  float m, l;                  // running maximum of the row's scores, log2 units; this lane's share of the row sum
};

// The chunk's own later blocks, hidden from a query when the mask inside the chunk is on.
struct Hidden {
  int lo, hi;
};
__device__ __forceinline__ Hidden hidden_keys(late_args<AttnF32Args>& a, int row, int q_row) {
  Hidden h{0x7fffffff, 0};
  if (a.mask_block_tokens > 0) {
    const int first = sdv2::row_chunk_start<offsetof(AttnF32Args, chunk_starts)>(a.chunk_starts.device, row);
    h.hi = first + a.q_tokens;
    h.lo = first + (q_row / a.mask_block_tokens + 1) * a.mask_block_tokens;
  }
  return h;
}

__device__ __forceinline__ void load_query(late_args<AttnF32Args>& a, int row, int head, int q_row, int hf, float (&qf)[kD / 2]) {
  // the query row as the B operand (rows past the last query repeat it; their results are not stored)
  const int t = q_row < a.q_tokens ? q_row : a.q_tokens - 1;
  const float* qp = a.q + row * a.q_st.row + head * a.q_st.head + (int64_t)t * a.q_st.token + 4 * hf;
#pragma unroll
  for (int c = 0; c < kD / 8; ++c) {
    const f32x4 x = *reinterpret_cast<const f32x4*>(qp + 8 * c);
#pragma unroll
    for (int e = 0; e < 4; ++e) qf[4 * c + e] = x[e];
  }
}

__device__ __forceinline__ void clear(Sums& z) {
#pragma unroll
  for (int db = 0; db < 4; ++db)
#pragma unroll
    for (int i = 0; i < 16; ++i) z.o[db][i] = 0.f;
  z.m = -INFINITY;
  z.l = 0.f;
}

// scores of a tile -> weights; returns what makes the sums of values so far relative to the new maximum
__device__ __forceinline__ float soften(f32x16& s, Sums& z, int key0, int seq, const Hidden& h, int hf, float scale_log2) {
  float m_tile = -INFINITY;
  // the last tile, and tiles that touch the hidden range of any query of the block
  if (key0 + kKeys > seq || (key0 + kKeys > h.lo && key0 < h.hi)) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int key = key0 + 8 * (i >> 2) + 4 * hf + (i & 3);
      if (key >= seq || (key >= h.lo && key < h.hi)) s[i] = -INFINITY;
    }
  }
#pragma unroll
  for (int i = 0; i < 16; ++i) m_tile = fmaxf(m_tile, s[i]);
  const float m_new = fmaxf(z.m, half_max(m_tile) * scale_log2);         // (a positive scale)
  // -inf only while every key so far was hidden from this query: nothing has been summed yet
  const float ref = m_new == -INFINITY ? 0.f : m_new;
  const float alpha = __builtin_amdgcn_exp2f(z.m - ref);           // 0 for the first visible keys
  z.m = m_new;
#pragma unroll
  for (int i = 0; i < 16; ++i) s[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[i], scale_log2, -ref));
  // the tile's own sum first, in pairs: one rounding of the long sum per tile
  float sum[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) sum[i] = s[i] + s[i + 8];
#pragma unroll
  for (int n = 4; n > 0; n >>= 1)
#pragma unroll
    for (int i = 0; i < n; ++i) sum[i] += sum[i + n];
  z.l = __builtin_fmaf(z.l, alpha, sum[0]);
  return alpha;
}

// LDS reads run two ahead of the four matrix instructions that each feeds (left alone, every one is waited for where it
// is issued: 10 % of a workgroup that has its CU to itself)
__device__ __forceinline__ void reads_ahead() {
  constexpr int kReads = 16, kMatrix = 0x8, kLdsRead = 0x100;
  __builtin_amdgcn_sched_group_barrier(kLdsRead, 2, 0);
#pragma unroll
  for (int i = 0; i < kReads; ++i) {
    __builtin_amdgcn_sched_group_barrier(kMatrix, 4, 0);
    if (i + 2 < kReads) __builtin_amdgcn_sched_group_barrier(kLdsRead, 1, 0);
  }
}

// sums so far + weights of a tile times its values: two accumulators at a time, from zero, so that the long sums are
// rounded once a tile (the multiplication by alpha, which every tile pays, takes the addition in).
// value(half, i): dimensions 64 half + 2 (lane % 32) and the one behind it of the key of accumulator register i
template <typename Value>
__device__ __forceinline__ void add_values(const f32x16& s, float alpha, Sums& z, Value value) {
#pragma unroll
  for (int half = 0; half < 2; ++half) {
    // (one read must not take the values of both halves: there are no registers for the later ones)
    if (half) asm volatile("" ::: "memory");
    f32x16 t0, t1;
#pragma unroll
    for (int i = 0; i < 16; ++i) t0[i] = t1[i] = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const f32x2 vf = value(half, i);
      t0 = __builtin_amdgcn_mfma_f32_32x32x2f32(vf[0], s[i], t0, 0, 0, 0);
      t1 = __builtin_amdgcn_mfma_f32_32x32x2f32(vf[1], s[i], t1, 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      z.o[2 * half][i] = __builtin_fmaf(z.o[2 * half][i], alpha, t0[i]);
      z.o[2 * half + 1][i] = __builtin_fmaf(z.o[2 * half + 1][i], alpha, t1[i]);
    }
  }
}

// A piece of a whole query tile: all waves stream the same keys through LDS.
__device__ __forceinline__ void stream_tiles(late_args<AttnF32Args>& a, float* lds, const Piece& w, int seq, bool idle, int tid, Sums& z) {
  const int lane = tid & 63, l32 = lane & 31, hf = lane >> 5, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int q_row = w.item * kQTile + wave * kQBlock + l32;
  const Hidden hidden = hidden_keys(a, w.row, q_row);

  // Wave w brings rows 8 w .. 8 w + 7 of either matrix, two in each transfer.  A whole tile is fetched from a scalar base
  // and one offset per lane; the last one, and token strides beyond 32 bits, take the general form, where keys past the
  // valid length repeat the last valid one (their scores are masked).
  const int64_t k_token = a.k_st.token, v_token = a.v_st.token;
  const float* const kp = a.k + w.row * a.k_st.row + w.head * a.k_st.head;
  const float* const vp = a.v + w.row * a.v_st.row + w.head * a.v_st.head;
  const float scale_log2 = a.scale_log2;
  const bool near = k_token < (1 << 24) && v_token < (1 << 24);
  const uint32_t lds0 = (uint32_t)(uintptr_t)(sdv2::attn::lds_char*)lds + wave * 4096;
  const uint32_t k_chunk = 16 * (l32 ^ hf ^ (wave & 1) << 3), k_row = hf * (uint32_t)k_token * 4, v_off = hf * (uint32_t)v_token * 4 + 16 * l32;
  auto issue = [&](int tile) {
    const uint32_t dst = lds0 + ((tile - w.tile0) & 1) * kTileBytes;
    const int key0 = tile * kKeys + wave * 8;
    if (near && (tile + 1) * kKeys <= seq) {
      const float* const kt = kp + key0 * k_token;
      const float* const vt = vp + key0 * v_token;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        dma16(reinterpret_cast<const char*>(kt + 2 * j * k_token), (k_chunk ^ (32 * j)) + k_row, dst + 1024 * j);
        dma16(reinterpret_cast<const char*>(vt + 2 * j * v_token), v_off, dst + 2 * kTileBytes + 1024 * j);
      }
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int64_t key = key0 + 2 * j + hf < seq ? key0 + 2 * j + hf : seq - 1;
        dma16_far(reinterpret_cast<const char*>(kp + key * k_token) + (k_chunk ^ (32 * j)), dst + 1024 * j);
        dma16_far(reinterpret_cast<const char*>(vp + key * v_token) + 16 * l32, dst + 2 * kTileBytes + 1024 * j);
      }
    }
  };
  if (w.tile0 < w.tile1) issue(w.tile0);
  float qf[kD / 2];
  load_query(a, w.row, w.head, q_row, hf, qf);

  // tile `tile` is there for all waves, and the next one on its way into the other buffer (whose readers, a tile ago, are
  // behind this barrier)
  auto advance = [&](int tile) {
    __builtin_amdgcn_s_waitcnt(0x0F70);       // vmcnt(0)
    __syncthreads();
    if (tile + 1 < w.tile1) issue(tile + 1);
  };
  // chunk 2 c + hf of row l32 lies at position (2 c + hf) ^ l32 % 16
  const char* const k_s = reinterpret_cast<const char*>(lds);
  const uint32_t k_read = l32 * 512 + 16 * (hf ^ (l32 & 15));
  if (idle)
    for (int tile = w.tile0; tile < w.tile1; ++tile) advance(tile);
  else for (int tile = w.tile0; tile < w.tile1; ++tile) {
    const int buf = (tile - w.tile0) & 1;
    advance(tile);
    f32x16 s;
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = 0.f;
    // the matrix instructions go ahead of the other workgroup's softmax on this SIMD (0.7 %)
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int c = 0; c < kD / 8; ++c) {
      const f32x4 kf = *reinterpret_cast<const f32x4*>(k_s + ((k_read + buf * kTileBytes) ^ (32 * (c & 7))) + 256 * (c >> 3));
#pragma unroll
      for (int e = 0; e < 4; ++e) s = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[e], qf[4 * c + e], s, 0, 0, 0);
    }
    reads_ahead();
    __builtin_amdgcn_s_setprio(0);
    const float alpha = soften(s, z, tile * kKeys, seq, hidden, hf, scale_log2);
    __builtin_amdgcn_s_setprio(1);
    const float* vr = lds + (2 * kTileBytes + buf * kTileBytes) / 4 + 4 * hf * kD + 2 * l32;
    add_values(s, alpha, z, [&](int half, int i) {
      return *reinterpret_cast<const f32x2*>(vr + (8 * (i >> 2) + (i & 3)) * kD + 64 * half);
    });
    reads_ahead();
    __builtin_amdgcn_s_setprio(0);
  }
  z.l = half_sum(z.l);
}

// A piece of the one or two blocks past the last whole query tile: the waves of a block deal its key tiles out among
// themselves, read them from memory as the matrix instructions take them, and meet in LDS.  The first `blocks` waves
// return with the sums.
__device__ __forceinline__ void stream_rest(late_args<AttnF32Args>& a, float* lds, const Piece& w, int seq, int blocks, int tid, Sums& z) {
  const int wave = tid >> 6, lane = tid & 63, l32 = lane & 31, hf = lane >> 5;
  const int ways = kWaves / blocks, block = wave % blocks;
  const int q_row = w.item * kQTile + block * kQBlock + l32;
  const Hidden hidden = hidden_keys(a, w.row, q_row);
  const int64_t k_token = a.k_st.token, v_token = a.v_st.token;
  const float* const kp = a.k + w.row * a.k_st.row + w.head * a.k_st.head + 4 * hf;
  const float* const vp = a.v + w.row * a.v_st.row + w.head * a.v_st.head + 2 * l32;
  const float scale_log2 = a.scale_log2;
  float qf[kD / 2];
  load_query(a, w.row, w.head, q_row, hf, qf);
  for (int tile = w.tile0 + wave / blocks; tile < w.tile1; tile += ways) {
    const int key0 = tile * kKeys;
    const int64_t key = key0 + l32 < seq ? key0 + l32 : seq - 1;
    const float* kr = kp + key * k_token;
    f32x4 kf[kD / 8];
#pragma unroll
    for (int c = 0; c < kD / 8; ++c) kf[c] = *reinterpret_cast<const f32x4*>(kr + 8 * c);
    f32x16 s;
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = 0.f;
#pragma unroll
    for (int c = 0; c < kD / 8; ++c)
#pragma unroll
      for (int e = 0; e < 4; ++e) s = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[c][e], qf[4 * c + e], s, 0, 0, 0);
    f32x2 vf[2][16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int at = key0 + 8 * (i >> 2) + 4 * hf + (i & 3);
      const float* const vr = vp + (at < seq ? at : seq - 1) * v_token;
      vf[0][i] = *reinterpret_cast<const f32x2*>(vr);
      vf[1][i] = *reinterpret_cast<const f32x2*>(vr + 64);
    }
    const float alpha = soften(s, z, key0, seq, hidden, hf, scale_log2);
    // (a wave has a quarter or half of the keys: nothing is gained by sums of each tile's own, and no register is free)
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
      for (int i = 0; i < 16; ++i) z.o[db][i] *= alpha;
#pragma unroll
    for (int i = 0; i < 16; ++i)
#pragma unroll
      for (int db = 0; db < 4; ++db)
        z.o[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(vf[db >> 1][i][db & 1], s[i], z.o[db], 0, 0, 0);
  }
  z.l = half_sum(z.l);

  // [wave past the first ones][register quad][lane][4], and behind the three of them the maxima and sums
  float* const part = lds + (wave - blocks) * kBlockFloats + 4 * lane;
  float* const stats = lds + 3 * kBlockFloats;
  if (wave >= blocks) {
#pragma unroll
    for (int i = 0; i < 16; ++i) *reinterpret_cast<f32x4*>(part + 256 * i) = f32x4{z.o[0][i], z.o[1][i], z.o[2][i], z.o[3][i]};
    if (hf == 0) {
      stats[(wave - blocks) * 64 + l32] = z.m;
      stats[(wave - blocks) * 64 + 32 + l32] = z.l;
    }
  }
  __syncthreads();
  if (wave < blocks) {
    for (int other = wave; other < kWaves - blocks; other += blocks) {
      const float m = stats[other * 64 + l32], l = stats[other * 64 + 32 + l32];
      const float top = fmaxf(z.m, m);
      const float mine = z.m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(z.m - top);
      const float its = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - top);
      const float* const src = lds + other * kBlockFloats + 4 * lane;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const f32x4 x = *reinterpret_cast<const f32x4*>(src + 256 * i);
#pragma unroll
        for (int db = 0; db < 4; ++db) z.o[db][i] = __builtin_fmaf(its, x[db], mine * z.o[db][i]);
      }
      z.l = __builtin_fmaf(its, l, mine * z.l);
      z.m = top;
    }
  }
}

__global__ __launch_bounds__(kThreads, 2)
void swa_attn_fwd_f32_kernel(const AttnF32Args args) {
  extern __shared__ __attribute__((aligned(16))) float lds_f32[];
  int* const flag = reinterpret_cast<int*>(lds_f32 + kLdsBytes / 4 - 4);

  // XCD x (workgroup id mod 8) takes the x-th eighth of the shares: the workgroups that read the same keys share an L2.
  const int wg = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  int begin = 0, end = 0, off = 0, pair = 0, item = 0;
  {
    late_args<AttnF32Args>& a = read_late<AttnF32Args>();
    const int per_pair = a.plan.whole_tiles + (a.plan.rest_blocks > 0);
    if (a.plan.share == 0) {                     // uncut: one item each
      if (wg >= a.plan.pairs * per_pair) return;
      pair = read_div(a.div_items)(wg);
      item = wg - pair * per_pair;
    } else {
      begin = wg * a.plan.share;
      if (begin >= a.plan.total) return;
      end = begin + a.plan.share < a.plan.total ? begin + a.plan.share : a.plan.total;
      pair = read_div(a.plan.div_pair)(begin);
      off = pair * a.plan.pair_units;
      item = read_div(a.plan.div_whole)(begin - off);
      item = item < a.plan.whole_tiles ? item : a.plan.whole_tiles;
      off += item * a.plan.whole_units;
    }
  }
  for (bool again = false;; again = true) {
    late_args<AttnF32Args>& a = read_late<AttnF32Args>();
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int lane = tid & 63, l32 = lane & 31, hf = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int whole_tiles = a.plan.whole_tiles, rest_blocks = a.plan.rest_blocks, share = a.plan.share;
    const bool is_rest = item >= whole_tiles;
    const ItemKind kind = is_rest ? rest_kind_f32(rest_blocks) : ItemKind{a.plan.whole_start, kWholeTileF32.per_tile};
    const int next_off = off + kind.units(a.plan.tiles);
    Piece w;
    w.tile0 = share ? kind.tile_at(begin - off, a.plan.tiles) : 0;
    w.tile1 = share ? kind.tile_at(end - off, a.plan.tiles) : a.plan.tiles;
    if (w.tile1 > w.tile0 || share == 0) {
      w.item = item;
      w.row = read_div(a.div_heads)(pair);
      w.head = pair - w.row * a.heads;
      if (again) __syncthreads();                // every wave is done with the LDS of the piece before
      const bool whole = w.tile0 == 0 && w.tile1 == a.plan.tiles;
      int seq = a.seq_lens ? a.seq_lens[w.row] : a.max_seq_len;
      seq = seq < a.max_seq_len ? seq : a.max_seq_len;
      seq = seq < 0 ? 0 : seq;
      // (a row may hold fewer keys than the longest one)
      const int tiles = (seq + kKeys - 1) / kKeys;
      w.tile0 = w.tile0 < tiles ? w.tile0 : tiles;
      w.tile1 = w.tile1 < tiles ? w.tile1 : tiles;

      // a wave whose block lies past the last query moves its share of the tiles and meets the barriers
      const bool idle = item * kQTile + wave * kQBlock >= a.q_tokens;
      Sums z;
      clear(z);
      if (is_rest) stream_rest(a, lds_f32, w, seq, rest_blocks, tid, z);
      else stream_tiles(a, lds_f32, w, seq, idle, tid, z);

      late_args<AttnF32Args>& b = read_late<AttnF32Args>();
      bool write = !idle;
      if (!whole) {
        const FastDiv div_share = read_div(b.plan.div_share);
        const int first_wg = first_workgroup(div_share, kind, off);
        const int parts = last_workgroup(div_share, kind, off, b.plan.tiles) - first_wg + 1;
        // A workgroup has a piece of two cut items at most: the one that began before its share, and the one that it begins.
        auto block_of = [&](int of) { return (int64_t)(2 * of + (of == first_wg)) * kWaves + wave; };
        if (!idle) {
          float* dst = b.part_o + block_of(wg) * kBlockFloats + 4 * lane;
#pragma unroll
          for (int i = 0; i < 16; ++i) store_coherent16(dst + 256 * i, f32x4{z.o[0][i], z.o[1][i], z.o[2][i], z.o[3][i]});
          if (hf == 0) {
            store_coherent(b.part_m + block_of(wg) * kQBlock + l32, z.m);
            store_coherent(b.part_l + block_of(wg) * kQBlock + l32, z.l);
          }
        }
        __builtin_amdgcn_s_waitcnt(0x0F70);       // vmcnt(0): the stores are acknowledged
        __syncthreads();
        if (tid == 0) {
          int32_t* ticket = b.tickets + pair * (whole_tiles + (rest_blocks > 0)) + item;
          const int drawn = __hip_atomic_fetch_add(ticket, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          const int last = drawn == parts - 1;
          if (last) __hip_atomic_store(ticket, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          *flag = last;
        }
        __syncthreads();
        write = write && *flag != 0;
        if (write) {
          // out = sum_s 2^(m_s - top) O_s / sum_s 2^(m_s - top) l_s.  Every trip to memory costs the same few
          // microseconds: the statistics of up to eight pieces travel together, then half a block at a time.
          constexpr int kBatch = 8;
          float ms[kBatch], ls[kBatch];
          auto stats = [&](int s0) {
#pragma unroll
            for (int u = 0; u < kBatch; ++u) {
              const int64_t blk = block_of(first_wg + (s0 + u < parts ? s0 + u : parts - 1));     // (past the last: repeats it)
              ms[u] = load_coherent(b.part_m + blk * kQBlock + l32);
              ls[u] = load_coherent(b.part_l + blk * kQBlock + l32);
            }
          };
          stats(0);
          float top = -INFINITY;
#pragma unroll
          for (int u = 0; u < kBatch; ++u) top = fmaxf(top, ms[u]);
          for (int sp = kBatch; sp < parts; ++sp) top = fmaxf(top, load_coherent(b.part_m + block_of(first_wg + sp) * kQBlock + l32));
          clear(z);
          for (int s0 = 0; s0 < parts; s0 += kBatch) {
            if (s0 > 0) stats(s0);
#pragma unroll
            for (int u = 0; u < kBatch; ++u) {
              if (s0 + u < parts) {
                const float weight = ms[u] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(ms[u] - top);
                z.l += weight * ls[u];
                const float* src = b.part_o + block_of(first_wg + s0 + u) * kBlockFloats + 4 * lane;
#pragma unroll
                for (int half = 0; half < 2; ++half) {
                  f32x4 x[8];
                  load_coherent_x8(src + 2048 * half, x);
#pragma unroll
                  for (int j = 0; j < 8; ++j)
#pragma unroll
                    for (int db = 0; db < 4; ++db) z.o[db][8 * half + j] = __builtin_fmaf(weight, x[j][db], z.o[db][8 * half + j]);
                }
              }
            }
          }
        }
      }

      const int q_row = item * kQTile + wave * kQBlock + l32;
      if (write && q_row < b.q_tokens) {
        const float inv = z.l > 0.f ? 1.0f / z.l : 0.f;       // no visible key: zeros, as the bf16 kernel writes
        float* op = b.out + w.row * b.o_st.row + w.head * b.o_st.head + (int64_t)q_row * b.o_st.token + 8 * hf;
#pragma unroll
        for (int half = 0; half < 2; ++half)
#pragma unroll
          for (int i = 0; i < 16; i += 2)
            *reinterpret_cast<f32x4*>(op + 64 * half + 16 * (i >> 2) + 2 * (i & 3)) =
                f32x4{z.o[2 * half][i] * inv, z.o[2 * half + 1][i] * inv, z.o[2 * half][i + 1] * inv, z.o[2 * half + 1][i + 1] * inv};
      }
    }
    if (next_off >= end) return;
    off = next_off;
    if (++item == whole_tiles + (rest_blocks > 0)) {
      item = 0;
      ++pair;
    }
  }
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }
bool stride_ok(const sdv2_stride3& s) { return s.row % 4 == 0 && s.token % 4 == 0 && s.head % 4 == 0; }
size_t align_up(size_t x, size_t a) { return (x + a - 1) / a * a; }

// The items of a call, and - true is returned - shares of them.  The waves of a CU share its matrix pipes, so a call
// lasts as long as the CU with the most to do: its tiles, and what is not a tile.  Three ways are compared, in sixteenths
// of the 3.9 us a tile takes:
//   one item for each workgroup     19 us (13 with two on a CU) besides the tiles
//   equal shares for one or two workgroups on every CU, which may hold the end of one item and the start of the next:
//                                   21-25 us, and 12 for each item of a workgroup that hides them behind no other one
//                                   (3 x 3707 x 40 queries against 289 keys 614 us uncut, 685 in 256 shares)
//   all items in the same number of pieces, one for each workgroup: 23 us, 33 with two on a CU, and what a short call
//                                   fares better with (3 x 108 x 12 against 2062 keys 59 us in 7 pieces, 71 in 14)
// A workgroup that has its CU to itself runs a tenth below its share where the keys come from memory (2876 x 9 against
// 7507 keys 829 us on 256 workgroups, 745 on 512).
bool f32_plan(int32_t rows, int32_t q_tokens, int32_t heads, int32_t max_seq_len, EvenPlanF32* e) {
  *e = EvenPlanF32{};
  const int64_t pairs = (int64_t)rows * heads;
  e->whole_tiles = q_tokens / kQTile;
  e->rest_blocks = (q_tokens % kQTile + kQBlock - 1) / kQBlock;
  if (e->rest_blocks > sdv2::attn::kMostRestBlocksF32) {
    ++e->whole_tiles;
    e->rest_blocks = 0;
  }
  e->tiles = (max_seq_len + kKeys - 1) / kKeys;
  const int64_t items = pairs * (e->whole_tiles + (e->rest_blocks > 0));
  if (items > (1 << 28)) return false;
  e->pairs = (int)pairs;
  e->workgroups = (int)(8 * ((items + 7) / 8));
  const int per_tile = kWholeTileF32.per_tile;
  if (items > kMaxTickets || e->tiles >= (1 << 24) || items * (kWholeTileF32.units(e->tiles) + kMostPieces) >= (1 << 30)) return false;

  const int whole = kWholeTileF32.units(e->tiles);
  e->rest_units = e->rest_blocks > 0 ? rest_kind_f32(e->rest_blocks).units(e->tiles) : 0;
  // in sixteenths of 3.9 us, a tile of one workgroup; `more` for what is not a tile
  auto cost = [&](int64_t workgroups, int64_t units, int per_cu_more, int more) {
    const int64_t per_cu = (workgroups + kCus - 1) / kCus;
    return (20 * per_cu + 2 * (per_cu & 1)) * units / 20 + per_cu * per_cu_more + more;
  };
  int64_t best = cost(items, whole, 0, 40);
  auto consider = [&](int whole_units, int share, int per_cu_more, int more) {
    const int total = (int)pairs * (e->whole_tiles * whole_units + e->rest_units);
    const int workgroups = (total + share - 1) / share;
    const int64_t c = cost(workgroups, share, per_cu_more, more);
    if (c >= best) return;
    best = c;
    e->whole_units = whole_units;
    e->share = share;
    e->total = total;
    e->workgroups = 8 * ((workgroups + 7) / 8);
  };
  const int total = (int)pairs * (e->whole_tiles * whole + e->rest_units);
  const int least = kWholeTileF32.units(4) > whole / kMostPieces ? kWholeTileF32.units(4) : whole / kMostPieces;
  for (int workgroups : {kCus, 2 * kCus}) {
    const int share = (total + workgroups - 1) / workgroups;
    // (starts and ends within a share are hidden only where another workgroup has the CU too)
    consider(whole, share < least ? least : share, 0, workgroups == kCus ? 60 + 50 * (share / whole + 1) : 110);
  }
  // (every piece has its start: only what makes the borders of shares and items fall together is added to the tiles)
  if (e->rest_blocks == 0)
    for (int pieces = 2; pieces <= kMostPieces && e->tiles / pieces >= 4; ++pieces) {
      const int share = (per_tile * e->tiles + pieces - 1) / pieces;
      consider(share * pieces, share, 70, 25);
    }
  if (e->share == 0) return false;
  e->whole_start = e->whole_units - per_tile * e->tiles;
  e->pair_units = e->whole_tiles * e->whole_units + e->rest_units;
  e->div_share = FastDiv::by((uint32_t)e->share);
  e->div_whole = FastDiv::by((uint32_t)e->whole_units);
  e->div_pair = FastDiv::by((uint32_t)e->pair_units);
  return true;
}

struct WorkspaceLayout {
  size_t part_o, part_m, part_l, total;
};
WorkspaceLayout workspace_layout(const EvenPlanF32& e) {
  const size_t blocks = (size_t)2 * e.workgroups * kWaves;
  WorkspaceLayout w;
  w.part_o = (size_t)kMaxTickets * sizeof(int32_t);
  w.part_m = w.part_o + blocks * kBlockFloats * sizeof(float);
  w.part_l = w.part_m + align_up(blocks * kQBlock * sizeof(float), 256);
  w.total = w.part_l + align_up(blocks * kQBlock * sizeof(float), 256);
  return w;
}

}  // namespace

extern "C" size_t sdv2_swa_attn_f32_workspace_bytes(int32_t rows, int32_t q_tokens, int32_t heads, int32_t max_seq_len) {
  if (rows <= 0 || q_tokens <= 0 || heads <= 0 || max_seq_len <= 0) return 0;
  EvenPlanF32 plan;
  return f32_plan(rows, q_tokens, heads, max_seq_len, &plan) ? workspace_layout(plan).total : 0;
}

int sdv2::attn_fwd_f32(const sdv2_attn_params* p, void* workspace, size_t workspace_bytes) {
  if (p->head_dim != kD) return SDV2_ERR_UNSUPPORTED;
  if (p->rows < 0 || p->q_tokens < 0 || p->heads <= 0 || p->max_seq_len < 0) return SDV2_ERR_INVALID_ARG;
  if (p->rows == 0 || p->q_tokens == 0) return SDV2_OK;
  if (!p->q || !p->k_cache || !p->v_cache || !p->out) return SDV2_ERR_INVALID_ARG;
  if (!aligned16(p->q) || !aligned16(p->k_cache) || !aligned16(p->v_cache) || !aligned16(p->out))
    return SDV2_ERR_INVALID_ARG;
  if (!stride_ok(p->q_stride) || !stride_ok(p->k_stride) || !stride_ok(p->v_stride) || !stride_ok(p->out_stride))
    return SDV2_ERR_INVALID_ARG;
  if (p->rows > 65535 || p->heads > 65535) return SDV2_ERR_INVALID_ARG;
  if (p->rope_freqs || p->q_norm_weight || p->q_inv_rms)
    return SDV2_ERR_UNSUPPORTED;                        // fp32 queries arrive normalised and rotated (the append returns them)
  if (p->mask_block_tokens < 0) return SDV2_ERR_INVALID_ARG;

  AttnF32Args a{};
  a.q = static_cast<const float*>(p->q);
  a.k = static_cast<const float*>(p->k_cache);
  a.v = static_cast<const float*>(p->v_cache);
  a.out = static_cast<float*>(p->out);
  a.seq_lens = p->seq_lens;
  a.q_st = p->q_stride; a.k_st = p->k_stride; a.v_st = p->v_stride; a.o_st = p->out_stride;
  a.rows = p->rows; a.q_tokens = p->q_tokens; a.heads = p->heads; a.max_seq_len = p->max_seq_len;
  a.scale_log2 = (p->softmax_scale > 0.f ? p->softmax_scale : 0.08838834764831845f) * kLog2e;  // 1/sqrt(128)
  if (p->mask_block_tokens > 0 && p->mask_block_tokens < p->q_tokens) {
    const int status = sdv2::set_chunk_starts(*p, &a.chunk_starts);
    if (status != SDV2_OK) return status;
    a.mask_block_tokens = p->mask_block_tokens;
  }
  if ((int64_t)p->rows * p->heads * ((p->q_tokens + kQTile - 1) / kQTile) > (1 << 28)) return SDV2_ERR_INVALID_ARG;
  const bool cut = f32_plan(p->rows, p->q_tokens, p->heads, p->max_seq_len, &a.plan);
  const int per_pair = a.plan.whole_tiles + (a.plan.rest_blocks > 0);
  a.div_items = FastDiv::by((uint32_t)per_pair);
  a.div_heads = FastDiv::by((uint32_t)p->heads);
  if (cut) {
    const WorkspaceLayout w = workspace_layout(a.plan);
    if (workspace && workspace_bytes >= w.total && (reinterpret_cast<uintptr_t>(workspace) & 255) == 0) {
      char* ws = static_cast<char*>(workspace);
      a.tickets = reinterpret_cast<int32_t*>(ws);
      a.part_o = reinterpret_cast<float*>(ws + w.part_o);
      a.part_m = reinterpret_cast<float*>(ws + w.part_m);
      a.part_l = reinterpret_cast<float*>(ws + w.part_l);
    } else {
      // nowhere for the pieces to meet: every workgroup walks one item from end to end
      a.plan.share = 0;
      a.plan.workgroups = 8 * ((a.plan.pairs * per_pair + 7) / 8);
    }
  }

  static std::atomic<bool> lds_ready[kMaxDevices];
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= kMaxDevices) return SDV2_ERR_LAUNCH;
  if (!lds_ready[device].load(std::memory_order_acquire)) {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(swa_attn_fwd_f32_kernel),
                            hipFuncAttributeMaxDynamicSharedMemorySize, kLdsBytes) != hipSuccess)
      return SDV2_ERR_LAUNCH;
    lds_ready[device].store(true, std::memory_order_release);
  }
  sdv2::launch_timed(SDV2_KERNEL_ATTENTION, swa_attn_fwd_f32_kernel, dim3((unsigned)a.plan.workgroups), dim3(kThreads),
                     kLdsBytes, static_cast<hipStream_t>(p->stream), a);
  if (hipGetLastError() != hipSuccess) return SDV2_ERR_LAUNCH;
  return SDV2_OK;
}
