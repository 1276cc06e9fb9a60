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
// wave w owns the 32-row block 32 w..32 w + 31, two workgroups per CU (67 KB of
// LDS each): one wave's softmax, loads and barriers run under the other's matrix
// instructions.  Keys stream through LDS 32 at a time, double-buffered.  The key
// range of a (row, head) is cut into as many pieces as pack the CUs best
// (f32_splits); each piece leaves its unnormalised output, maximum and sum in
// the workspace, and the workgroup that draws the last ticket of its query tile
// combines them in their fixed order, so the result does not depend on which one
// that is.  A caller without a workspace gets one piece per (row, head).
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
//                  dimensions 4 m + db, m = 0..31, so one 16-byte read of V feeds
//                  the four accumulators and a lane's results are 16 contiguous
//                  bytes of an output row.
//
// 1560 queries x 12 heads against 6240 keys: 2056 us -> 540 us
// (29 -> 111 TFLOP/s; 126 on 2 x 1740 queries against 8700 keys, where the grid
// packs better, with the matrix pipe 80 % busy at the 2.2 GHz the chip then
// holds); the kernel before it kept the products on the vector ALU, at 64 rows
// per workgroup without a key split.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>

#include "sdv2kv.h"
#include "sdv2kv_profile.h"
#include "sdv2kv_internal.h"

namespace {

typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) float f32x4;

constexpr int kD = SDV2_HEAD_DIM;     // 128
constexpr int kWaves = 4;
constexpr int kThreads = kWaves * 64;
constexpr int kQBlock = 32;           // query rows per wave
constexpr int kQTile = kWaves * kQBlock;
constexpr int kKeys = 32;             // keys per tile
// A lane reads 16 bytes of "its" key row of K: rows start 4 banks apart, so that eight lanes' reads never meet in a
// bank, and every read of a tile is one base register plus an immediate.  V is read along a row and needs no padding.
constexpr int kKStride = kD + 4;
constexpr int kKTileFloats = kKeys * kKStride, kVTileFloats = kKeys * kD;
constexpr int kPieces = kKeys * kD / 4 / kThreads;    // 16-byte pieces per thread and matrix tile: 4
constexpr int kLdsBytes = 2 * (kKTileFloats + kVTileFloats) * 4 + 16;   // two buffers of each, one flag word
constexpr int kMaxDevices = 64;
constexpr int kCus = 256;
constexpr float kLog2e = 1.4426950408889634f;
// Ticket words at the head of the workspace, as in the bf16 kernel (one
// workspace serves both): a fixed region, all zero between calls.
constexpr int kMaxTickets = 16384;
constexpr int kMaxSplits = 16;
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
  int32_t splits, q_tiles, q_blocks;
  int32_t* tickets;            // [row][head][query tile]
  float* part_o;               // [split][row][head][block][16 KB]: sums of weights times values, in register order
  float* part_m;               // [split][row][head][block][32]: running maximum, log2 units
  float* part_l;               // [split][row][head][block][32]: sum of weights
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
__device__ __forceinline__ void store_coherent16(float* p, const f32x4& x) {
  asm volatile("global_store_dwordx4 %0, %1, off sc1" : : "v"(p), "v"(x) : "memory");
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

__global__ __launch_bounds__(kThreads, 2)
void swa_attn_fwd_f32_kernel(const AttnF32Args a) {
  extern __shared__ __attribute__((aligned(16))) float lds_f32[];
  float* const k_s = lds_f32;                       // [2][kKeys][kKStride]
  float* const v_s = lds_f32 + 2 * kKTileFloats;    // [2][kKeys][kD]
  int* const flag = reinterpret_cast<int*>(v_s + 2 * kVTileFloats);

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int l32 = lane & 31, hf = lane >> 5;

  // XCD x (workgroup id mod 8) takes the x-th eighth of the (row, head, split,
  // query tile) list: the workgroups that read the same keys share one L2.
  int qtile, head, row, split;
  {
    const int total = a.rows * a.heads * a.splits * a.q_tiles;
    const int xcd = blockIdx.x & 7;
    const int first = (int)(((int64_t)xcd * total) >> 3), end = (int)(((int64_t)(xcd + 1) * total) >> 3);
    int item = first + (blockIdx.x >> 3);
    if (item >= end) return;
    qtile = item % a.q_tiles;
    item /= a.q_tiles;
    split = item % a.splits;
    item /= a.splits;
    head = item % a.heads;
    row = item / a.heads;
  }

  int seq = a.seq_lens ? a.seq_lens[row] : a.max_seq_len;
  seq = seq < a.max_seq_len ? seq : a.max_seq_len;
  seq = seq < 0 ? 0 : seq;
  const int tiles = (seq + kKeys - 1) / kKeys;
  const int per_split = (tiles + a.splits - 1) / a.splits;
  const int tile0 = split * per_split;
  const int tile1 = tile0 + per_split < tiles ? tile0 + per_split : tiles;

  const int q_row = qtile * kQTile + wave * kQBlock + l32;
  // a wave whose block lies past the last query moves its share of the tiles and meets the barriers
  const bool idle = __builtin_amdgcn_readfirstlane(qtile * kQTile + wave * kQBlock >= a.q_tokens);

  // the chunk's own later blocks, hidden from this lane's query when the mask inside the chunk is on
  int m_lo = 0x7fffffff, m_hi = 0;
  if (a.mask_block_tokens > 0) {
    const int first = sdv2::row_chunk_start<offsetof(AttnF32Args, chunk_starts)>(a.chunk_starts.device, row);
    m_hi = first + a.q_tokens;
    m_lo = first + (q_row / a.mask_block_tokens + 1) * a.mask_block_tokens;
  }

  // This thread's pieces of a tile: piece n is chunk tid % 32 of key tid / 32 + 8 n (both matrices).  A whole tile is
  // fetched from a scalar base plus a 32-bit offset per piece, formed once (64-bit products per load are a tenth of
  // the vector work of a tile); the last one, and token strides beyond 32 bits, take the general form, where keys
  // past the valid length repeat the last valid one (their scores are masked).
  const float* const kp = a.k + row * a.k_st.row + head * a.k_st.head;
  const float* const vp = a.v + row * a.v_st.row + head * a.v_st.head;
  const bool near = a.k_st.token < (1 << 24) && a.v_st.token < (1 << 24);
  uint32_t k_off[kPieces], v_off[kPieces];
#pragma unroll
  for (int n = 0; n < kPieces; ++n) {
    k_off[n] = ((tid >> 5) + 8 * n) * (uint32_t)a.k_st.token + 4 * (tid & 31);
    v_off[n] = ((tid >> 5) + 8 * n) * (uint32_t)a.v_st.token + 4 * (tid & 31);
  }
  f32x4 k_next[kPieces], v_next[kPieces];
  auto fetch = [&](int tile) {
    if (near && (tile + 1) * kKeys <= seq) {
      const float* const kt = kp + (int64_t)tile * kKeys * a.k_st.token;
      const float* const vt = vp + (int64_t)tile * kKeys * a.v_st.token;
#pragma unroll
      for (int n = 0; n < kPieces; ++n) {
        k_next[n] = *reinterpret_cast<const f32x4*>(kt + k_off[n]);
        v_next[n] = *reinterpret_cast<const f32x4*>(vt + v_off[n]);
      }
    } else {
#pragma unroll
      for (int n = 0; n < kPieces; ++n) {
        int64_t key = tile * kKeys + (tid >> 5) + 8 * n;
        key = key < seq ? key : seq - 1;
        k_next[n] = *reinterpret_cast<const f32x4*>(kp + key * a.k_st.token + 4 * (tid & 31));
        v_next[n] = *reinterpret_cast<const f32x4*>(vp + key * a.v_st.token + 4 * (tid & 31));
      }
    }
  };
  auto park = [&](int buf) {
#pragma unroll
    for (int n = 0; n < kPieces; ++n) {
      const int r = (tid >> 5) + 8 * n;
      *reinterpret_cast<f32x4*>(k_s + buf * kKTileFloats + r * kKStride + 4 * (tid & 31)) = k_next[n];
      *reinterpret_cast<f32x4*>(v_s + buf * kVTileFloats + r * kD + 4 * (tid & 31)) = v_next[n];
    }
  };
  if (tile0 < tile1) fetch(tile0);

  // the query row as the B operand (rows past the last query repeat it; their results are not stored)
  float qf[kD / 2];
  {
    const int t = q_row < a.q_tokens ? q_row : a.q_tokens - 1;
    const float* qp = a.q + row * a.q_st.row + head * a.q_st.head + (int64_t)t * a.q_st.token + 4 * hf;
#pragma unroll
    for (int c = 0; c < kD / 8; ++c) {
      const f32x4 x = *reinterpret_cast<const f32x4*>(qp + 8 * c);
#pragma unroll
      for (int e = 0; e < 4; ++e) qf[4 * c + e] = x[e];
    }
  }

  f32x16 o[4];
#pragma unroll
  for (int db = 0; db < 4; ++db)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[db][i] = 0.f;
  float m_run = -INFINITY;     // running maximum of the row's scores, log2 units
  float l_run = 0.f;           // this lane's share of the row sum

  auto advance = [&](int tile) {
    park((tile - tile0) & 1);  // (its last readers, two tiles ago, are behind the barrier of the previous trip)
    __syncthreads();
    if (tile + 1 < tile1) fetch(tile + 1);
  };
  if (idle)
    for (int tile = tile0; tile < tile1; ++tile) advance(tile);
  else for (int tile = tile0; tile < tile1; ++tile) {
    const int buf = (tile - tile0) & 1;
    advance(tile);
    f32x16 s;
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = 0.f;
    // the matrix instructions go ahead of the other workgroup's softmax on this SIMD (0.7 %)
    __builtin_amdgcn_s_setprio(1);
    const float* kr = k_s + buf * kKTileFloats + l32 * kKStride + 4 * hf;
#pragma unroll
    for (int c = 0; c < kD / 8; ++c) {
      const f32x4 kf = *reinterpret_cast<const f32x4*>(kr + 8 * c);
#pragma unroll
      for (int e = 0; e < 4; ++e) s = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[e], qf[4 * c + e], s, 0, 0, 0);
    }

    __builtin_amdgcn_s_setprio(0);

    const int key0 = tile * kKeys;
    float m_tile = -INFINITY;
    // the last tile, and tiles that touch the hidden range of any query of the block
    if (key0 + kKeys > seq || (key0 + kKeys > m_lo && key0 < m_hi)) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int key = key0 + 8 * (i >> 2) + 4 * hf + (i & 3);
        if (key >= seq || (key >= m_lo && key < m_hi)) s[i] = -INFINITY;
      }
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) m_tile = fmaxf(m_tile, s[i]);
    const float m_new = fmaxf(m_run, half_max(m_tile) * a.scale_log2);         // (a positive scale)
    // -inf only while every key so far was hidden from this query: nothing has been summed yet
    const float ref = m_new == -INFINITY ? 0.f : m_new;
    // (every tile, needed or not: a branch around these 64 multiplies costs the accumulators a copy)
    const float alpha = __builtin_amdgcn_exp2f(m_run - ref);           // 0 for the first visible keys
    m_run = m_new;
    l_run *= alpha;
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
      for (int i = 0; i < 16; ++i) o[db][i] *= alpha;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      s[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[i], a.scale_log2, -ref));
      l_run += s[i];
    }

    __builtin_amdgcn_s_setprio(1);
    const float* vr = v_s + buf * kVTileFloats + 4 * hf * kD + 4 * l32;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const f32x4 vf = *reinterpret_cast<const f32x4*>(vr + (8 * (i >> 2) + (i & 3)) * kD);
#pragma unroll
      for (int db = 0; db < 4; ++db) o[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(vf[db], s[i], o[db], 0, 0, 0);
    }
    __builtin_amdgcn_s_setprio(0);
  }

  float l = half_sum(l_run);
  if (a.splits > 1) {
    const int64_t slab = (int64_t)a.rows * a.heads * a.q_blocks;
    const int64_t blk0 = ((int64_t)row * a.heads + head) * a.q_blocks + qtile * kWaves + wave;
    if (!idle) {
      const int64_t blk = split * slab + blk0;
      float* dst = a.part_o + blk * kBlockFloats + 4 * lane;
#pragma unroll
      for (int i = 0; i < 16; ++i) store_coherent16(dst + 256 * i, f32x4{o[0][i], o[1][i], o[2][i], o[3][i]});
      if (hf == 0) {
        store_coherent(a.part_m + blk * kQBlock + l32, m_run);
        store_coherent(a.part_l + blk * kQBlock + l32, l);
      }
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);       // vmcnt(0): the stores are acknowledged
    __syncthreads();
    if (tid == 0) {
      int32_t* ticket = a.tickets + ((int64_t)row * a.heads + head) * a.q_tiles + qtile;
      const int drawn = __hip_atomic_fetch_add(ticket, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const int last = drawn == a.splits - 1;
      if (last) __hip_atomic_store(ticket, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      *flag = last;
    }
    __syncthreads();
    if (*flag == 0 || idle) return;
    // out = sum_s 2^(m_s - top) O_s / sum_s 2^(m_s - top) l_s.  Every trip to memory costs the same few
    // microseconds: the statistics of up to eight ranges travel together, then half a block at a time.
    constexpr int kBatch = 8;
    float ms[kBatch], ls[kBatch];
    auto stats = [&](int s0) {
#pragma unroll
      for (int u = 0; u < kBatch; ++u) {
        const int64_t blk = (s0 + u < a.splits ? s0 + u : a.splits - 1) * slab + blk0;     // (past the last: repeats it)
        ms[u] = load_coherent(a.part_m + blk * kQBlock + l32);
        ls[u] = load_coherent(a.part_l + blk * kQBlock + l32);
      }
    };
    stats(0);
    float top = -INFINITY;
#pragma unroll
    for (int u = 0; u < kBatch; ++u) top = fmaxf(top, ms[u]);
    for (int sp = kBatch; sp < a.splits; ++sp)
      top = fmaxf(top, load_coherent(a.part_m + (sp * slab + blk0) * kQBlock + l32));
    l = 0.f;
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
      for (int i = 0; i < 16; ++i) o[db][i] = 0.f;
    for (int s0 = 0; s0 < a.splits; s0 += kBatch) {
      if (s0 > 0) stats(s0);
#pragma unroll
      for (int u = 0; u < kBatch; ++u) {
        if (s0 + u < a.splits) {
          const float w = ms[u] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(ms[u] - top);
          l += w * ls[u];
          const float* src = a.part_o + ((s0 + u) * slab + blk0) * kBlockFloats + 4 * lane;
#pragma unroll
          for (int half = 0; half < 2; ++half) {
            f32x4 x[8];
            load_coherent_x8(src + 2048 * half, x);
#pragma unroll
            for (int j = 0; j < 8; ++j)
#pragma unroll
              for (int db = 0; db < 4; ++db) o[db][8 * half + j] = __builtin_fmaf(w, x[j][db], o[db][8 * half + j]);
          }
        }
      }
    }
  } else if (idle) {
    return;
  }

  const float inv = l > 0.f ? 1.0f / l : 0.f;       // no visible key: zeros, as the bf16 kernel writes
  if (q_row < a.q_tokens) {
    float* op = a.out + row * a.o_st.row + head * a.o_st.head + (int64_t)q_row * a.o_st.token + 16 * hf;
#pragma unroll
    for (int i = 0; i < 16; ++i)
      *reinterpret_cast<f32x4*>(op + 32 * (i >> 2) + 4 * (i & 3)) =
          f32x4{o[0][i] * inv, o[1][i] * inv, o[2][i] * inv, o[3][i] * inv};
  }
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }
bool stride_ok(const sdv2_stride3& s) { return s.row % 4 == 0 && s.token % 4 == 0 && s.head % 4 == 0; }
size_t align_up(size_t x, size_t a) { return (x + a - 1) / a * a; }

// Key ranges per (row, head).  The waves of a CU share its matrix pipes, so a
// call lasts as long as the CU with the most workgroups: ceil(workgroups / 256)
// times the length of one, which is its tiles plus about two tile times of start
// and end (query load, first tile, partial results).  The smallest such product
// wins, the smaller count on a tie.  A workgroup that has its CU to itself hides
// nothing of its softmax and loads and runs some 15 % below its share.
int f32_splits(int32_t rows, int32_t q_tokens, int32_t heads, int32_t max_seq_len) {
  const int64_t columns = (int64_t)rows * heads * ((q_tokens + kQTile - 1) / kQTile);
  if (columns > kMaxTickets) return 1;
  const int tiles = (max_seq_len + kKeys - 1) / kKeys;
  int best = 1;
  int64_t best_cost = INT64_MAX;
  for (int s = 1; s <= kMaxSplits && (s == 1 || tiles / s >= 4); ++s) {
    const int64_t per_cu = (columns * s + kCus - 1) / kCus;
    const int64_t cost = (20 * per_cu + 3 * (per_cu & 1)) * ((tiles + s - 1) / s + 2);
    if (cost < best_cost) { best_cost = cost; best = s; }
  }
  return best;
}

struct WorkspaceLayout {
  size_t part_o, part_m, part_l, total;
};
WorkspaceLayout workspace_layout(int32_t rows, int32_t q_tokens, int32_t heads, int32_t splits) {
  const size_t blocks = (size_t)splits * rows * heads * ((q_tokens + kQBlock - 1) / kQBlock);
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
  const int splits = f32_splits(rows, q_tokens, heads, max_seq_len);
  return splits > 1 ? workspace_layout(rows, q_tokens, heads, splits).total : 0;
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
  a.q_tiles = (p->q_tokens + kQTile - 1) / kQTile;
  a.q_blocks = (p->q_tokens + kQBlock - 1) / kQBlock;
  a.splits = 1;
  const int splits = f32_splits(p->rows, p->q_tokens, p->heads, p->max_seq_len);
  if (splits > 1 && workspace) {
    const WorkspaceLayout w = workspace_layout(p->rows, p->q_tokens, p->heads, splits);
    if (workspace_bytes >= w.total && (reinterpret_cast<uintptr_t>(workspace) & 255) == 0) {
      char* ws = static_cast<char*>(workspace);
      a.splits = splits;
      a.tickets = reinterpret_cast<int32_t*>(ws);
      a.part_o = reinterpret_cast<float*>(ws + w.part_o);
      a.part_m = reinterpret_cast<float*>(ws + w.part_m);
      a.part_l = reinterpret_cast<float*>(ws + w.part_l);
    }
  }
  const int64_t items = (int64_t)p->rows * p->heads * a.q_tiles * a.splits;
  if (items > (1 << 28)) return SDV2_ERR_INVALID_ARG;

  static std::atomic<bool> lds_ready[kMaxDevices];
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= kMaxDevices) return SDV2_ERR_LAUNCH;
  if (!lds_ready[device].load(std::memory_order_acquire)) {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(swa_attn_fwd_f32_kernel),
                            hipFuncAttributeMaxDynamicSharedMemorySize, kLdsBytes) != hipSuccess)
      return SDV2_ERR_LAUNCH;
    lds_ready[device].store(true, std::memory_order_release);
  }
  sdv2::launch_timed(SDV2_KERNEL_ATTENTION, swa_attn_fwd_f32_kernel, dim3((unsigned)(8 * ((items + 7) / 8))), dim3(kThreads),
                     kLdsBytes, static_cast<hipStream_t>(p->stream), a);
  if (hipGetLastError() != hipSuccess) return SDV2_ERR_LAUNCH;
  return SDV2_OK;
}
