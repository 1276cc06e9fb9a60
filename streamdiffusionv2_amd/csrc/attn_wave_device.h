// One 32-row query block of the bf16 attention as the work of a whole workgroup (gfx950
// only): its 8 waves take the keys 32 at a time in turn, each by itself, and meet once, in
// LDS, at the end.  For small calls (swa_attn_fwd_wave.hip), and for the few query rows
// past the last whole query tile of a larger one (swa_attn_fwd_even.hip).
//
// A wave's K and V blocks sit in 16 KB of LDS of its own; the next K block is requested
// as soon as the fragments of this one are in registers, the next V block likewise.
// (K fragments straight from memory into registers, which would leave room for a block
// more in flight, are 64-byte pieces of 16 rows: 2.2 us per 256 keys and workgroup.)
//
// Or two workgroups share a query block, each with half of V's columns (kParts = 2): both take all of K, nothing has to meet
// between them, and each brings three quarters of the bytes; every number is the one a workgroup by itself comes to.
//
// Matrix layout (v_mfma_f32_16x16x32_bf16) and V^T fragments as in swa_attn_fwd_m16.hip.
// Softmax: exp2 of the scaled scores against a running maximum per query and wave.
#ifndef SDV2KV_ATTN_WAVE_DEVICE_H
#define SDV2KV_ATTN_WAVE_DEVICE_H

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "sdv2kv.h"
#include "sdv2kv_internal.h"
#include "rope_device.h"
#include "attn_device.h"

namespace sdv2 {
namespace attn {
namespace wave {

constexpr int kWaves = 8;
constexpr int kThreads = kWaves * 64;
constexpr int kKeys = 32;                          // keys of a block
constexpr int kSub = 16 * 256;                     // bytes of 16 keys
constexpr int kBlockBytes = kKeys * 256;
constexpr int kWaveLds = 2 * kBlockBytes;          // a K and a V block; at the end the wave's 32 x 128 fp32 result
static_assert(kWaveLds == kQBlock * kD * 4, "the result takes the place of the blocks");
constexpr int kLdsStats = kWaves * kWaveLds;       // [wave][query] (largest score, row sum)
constexpr int kLdsBytes = kLdsStats + kWaves * kQBlock * 8;

typedef __attribute__((address_space(3))) f32x4 lds_f32x4;
typedef __attribute__((address_space(3))) f32x2 lds_f32x2;

// Fragments of the block in LDS, waited for in the statement that reads them (the compiler would wait for every
// transfer into LDS that is in flight).
// All of K: key 16 kt + lane % 16, d-step ks; address `at ^ (ks << 6)`, second 16 keys kSub further on
__device__ __forceinline__ void read_k_now(uint32_t at, u32x4 (&k)[2][4]) {
  asm volatile(
      "ds_read_b128 %0, %8\n\t"
      "ds_read_b128 %1, %9\n\t"
      "ds_read_b128 %2, %10\n\t"
      "ds_read_b128 %3, %11\n\t"
      "ds_read_b128 %4, %8 offset:%12\n\t"
      "ds_read_b128 %5, %9 offset:%12\n\t"
      "ds_read_b128 %6, %10 offset:%12\n\t"
      "ds_read_b128 %7, %11 offset:%12\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(k[0][0]), "=&v"(k[0][1]), "=&v"(k[0][2]), "=&v"(k[0][3]), "=&v"(k[1][0]), "=&v"(k[1][1]), "=&v"(k[1][2]),
        "=&v"(k[1][3])
      : "v"(at), "v"(at ^ 64u), "v"(at ^ 128u), "v"(at ^ 192u), "n"(kSub)
      : "memory");
}
// Four V^T fragments: dimension blocks db .. db + 3, address `at ^ (db << 5)`, second 16 keys as far on as 16 rows take
template <int kParts>
__device__ __forceinline__ void read_v_now(uint32_t at, bf16x8 (&f)[4]) {
  u32x2 lo[4], hi[4];
  asm volatile(
      "ds_read_b64_tr_b16 %0, %8\n\t"
      "ds_read_b64_tr_b16 %1, %8 offset:%12\n\t"
      "ds_read_b64_tr_b16 %2, %9\n\t"
      "ds_read_b64_tr_b16 %3, %9 offset:%12\n\t"
      "ds_read_b64_tr_b16 %4, %10\n\t"
      "ds_read_b64_tr_b16 %5, %10 offset:%12\n\t"
      "ds_read_b64_tr_b16 %6, %11\n\t"
      "ds_read_b64_tr_b16 %7, %11 offset:%12\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(lo[0]), "=&v"(hi[0]), "=&v"(lo[1]), "=&v"(hi[1]), "=&v"(lo[2]), "=&v"(hi[2]), "=&v"(lo[3]), "=&v"(hi[3])
      : "v"(at), "v"(at ^ 32u), "v"(at ^ 64u), "v"(at ^ 96u), "n"(kSub / kParts)
      : "memory");
#pragma unroll
  for (int i = 0; i < 4; ++i) f[i] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo[i], hi[i], 0, 1, 2, 3));
}

// All but the newest block (kTransfers, if there is one) have landed
template <int kTransfers>
__device__ __forceinline__ void land(bool newer) {
  if (newer) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kTransfers) : "memory");
  else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}
// Where 16-byte chunk c of row r of half of V is stored: position c ^ swz_half(r).  Two rows lie side by side in the banks, and
// the four of a parity among eight consecutive rows, two chunks of each read together, must not meet.
__device__ __forceinline__ int swz_half(int r) { return (r >> 1 & 3) << 1; }
// A query that arrives rotated, ahead of everything else: it has landed with the first block
__device__ __forceinline__ void load_rotated(bf16x8 (&qf)[2][4], const uint16_t* p0, const uint16_t* p1) {
  asm volatile(
      "global_load_dwordx4 %0, %8, off\n\t"
      "global_load_dwordx4 %1, %8, off offset:64\n\t"
      "global_load_dwordx4 %2, %8, off offset:128\n\t"
      "global_load_dwordx4 %3, %8, off offset:192\n\t"
      "global_load_dwordx4 %4, %9, off\n\t"
      "global_load_dwordx4 %5, %9, off offset:64\n\t"
      "global_load_dwordx4 %6, %9, off offset:128\n\t"
      "global_load_dwordx4 %7, %9, off offset:192 ; Q requested"
      : "=&v"(qf[0][0]), "=&v"(qf[0][1]), "=&v"(qf[0][2]), "=&v"(qf[0][3]), "=&v"(qf[1][0]), "=&v"(qf[1][1]),
        "=&v"(qf[1][2]), "=&v"(qf[1][3])
      : "v"(p0), "v"(p1)
      : "memory");
}

// Queries q0 .. q0 + 31 of (row, head) against 32-key blocks [first_block, end_block) of those they see.  Every thread
// gets eight columns, 8 (tid % 16) and on, of row tid / 16 of the normalised result; of two parts four, 64 part + 4 (tid %
// 16) and on.  kEarly: a query that arrives
// rotated is requested ahead of the first keys and waited for with them, which rests on the compiler leaving its
// registers alone until then (checked on the assembly of the kernel that uses it).
template <bool kMask, bool kRope, bool kEarly, int kParts = 1, typename Args>
__device__ __forceinline__ void stream_block(Args& a, lds_char* lds, int head, int row, int q0, int first_block, int end_block,
                                             f32x4 (&sum)[2 / kParts], int part = 0) {
  static_assert(kParts == 1 || kParts == 2, "columns of V");
  constexpr int kDb = 8 / kParts, kVTransfers = 8 / kParts, kVRow = 256 / kParts;       // dimension blocks, transfers and bytes of a row of V
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n16 = lane & 15, g = lane >> 4;

  int seq = a.seq_lens ? a.seq_lens[row] : a.max_seq_len;
  seq = seq < a.max_seq_len ? seq : a.max_seq_len;
  seq = seq < 0 ? 0 : seq;
  int nblocks = (seq + kKeys - 1) / kKeys;
  // With the mask inside the chunk: this lane's queries do not see keys [m_lo, m_hi), and the blocks
  // [hole, hole + skipped) are hidden from all of the workgroup's queries (from the last one, that is) and left out.
  int m_lo[2] = {0, 0}, m_lo_first = 0, m_hi = 0, hole = 0x7fffffff, skipped = 0;
  if constexpr (kMask) {
    const int first = row_chunk_start(a, row), bt = a.mask_block_tokens;
    const int q_last = q0 + kQBlock < a.q_tokens ? q0 + kQBlock - 1 : a.q_tokens - 1;
    m_hi = first + a.q_tokens;
    m_lo_first = first + (q0 / bt + 1) * bt;
#pragma unroll
    for (int qt = 0; qt < 2; ++qt) m_lo[qt] = first + ((q0 + 16 * qt + n16) / bt + 1) * bt;
    const int h0 = (first + (q_last / bt + 1) * bt + kKeys - 1) / kKeys, h1 = m_hi >= seq ? nblocks : m_hi / kKeys;
    if (h1 > h0) {
      hole = h0;
      skipped = h1 - h0;
      nblocks -= skipped;
    }
  }
  nblocks = nblocks < end_block ? nblocks : end_block;
  const int block0 = first_block + wave;
  auto key0_of = [&](int b) { return (kMask && b >= hole ? b + skipped : b) * kKeys; };

  const char* kbase = uniform_pointer(a.k + row * a.k_st.row + head * a.k_st.head);
  const char* vbase = uniform_pointer(a.v + row * a.v_st.row + head * a.v_st.head);
  const uint32_t k_tok_bytes = (uint32_t)(a.k_st.token * 2);
  const uint32_t v_tok_bytes = (uint32_t)(a.v_st.token * 2);
  const uint32_t mine = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)lds + wave * kWaveLds);    // this wave's part of LDS

  // ---- the queries: B fragments, query 16 qt + lane % 16, dimensions 32 ks + 8 g .. ----
  bf16x8 qf[2][4];
  const uint16_t* q_ptr[2];
  int q_tok[2];
#pragma unroll
  for (int qt = 0; qt < 2; ++qt) {
    q_tok[qt] = q0 + 16 * qt + n16 < a.q_tokens ? q0 + 16 * qt + n16 : a.q_tokens - 1;
    q_ptr[qt] = a.q + row * a.q_st.row + (int64_t)q_tok[qt] * a.q_st.token + head * a.q_st.head + 8 * g;
  }

  if constexpr (kRope) {
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
  } else if constexpr (kEarly) {
    load_rotated(qf, q_ptr[0], q_ptr[1]);
  } else {
#pragma unroll
    for (int qt = 0; qt < 2; ++qt)
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) qf[qt][ks] = *reinterpret_cast<const bf16x8*>(q_ptr[qt] + 32 * ks);
  }

  // ---- streaming: eight transfers a block of K or V, which complete in the order they were issued.  The last block,
  // where it is not whole, is moved down to end with the last valid key: the keys it shares with its predecessor
  // are masked.  With fewer than 32 keys in all the same is done with the block's second half, and the rows of the
  // first half past the last key repeat it.
  const int last_key0 = seq > kKeys ? seq - kKeys : 0;
  auto loaded_from = [&](int key0) { return key0 < last_key0 ? key0 : last_key0; };
  const int second = seq >= kKeys ? 16 : seq > 16 ? seq - 16 : 0;         // where the second 16 keys start
  uint32_t k_off[4], v_off[kVTransfers / 2];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int r = 4 * j + g;
    const uint32_t rr = r < seq ? r : seq - 1, chunk = (uint32_t)((n16 ^ swz16(r)) << 4);
    k_off[j] = rr * k_tok_bytes + chunk;
    if constexpr (kParts == 1) v_off[j] = rr * v_tok_bytes + chunk;
  }
  if constexpr (kParts == 2)
#pragma unroll
    for (int j = 0; j < kVTransfers / 2; ++j) {
      const int r = 8 * j + (lane >> 3);
      v_off[j] = (uint32_t)(r < seq ? r : seq - 1) * v_tok_bytes + (uint32_t)(((lane & 7) ^ swz_half(r)) << 4) + part * kVRow;
    }
  auto fetch = [&](const char* base, uint32_t tok_bytes, const auto& off, int b, uint32_t dst) {
    constexpr int kEach = sizeof(off) / sizeof(uint32_t);        // transfers of 16 keys
    const char* first = base + (int64_t)loaded_from(key0_of(b)) * tok_bytes;
    const char* half = first + (int64_t)second * tok_bytes;
#pragma unroll
    for (int j = 0; j < 2 * kEach; ++j) dma16(j < kEach ? first : half, off[j % kEach], dst + j * 1024);
  };
  auto fetch_k = [&](int b) { fetch(kbase, k_tok_bytes, k_off, b, mine); };
  auto fetch_v = [&](int b) { fetch(vbase, v_tok_bytes, v_off, b, mine + kBlockBytes); };
  if (block0 < nblocks) {
    fetch_k(block0);
    fetch_v(block0);
  }

  const float c2 = a.scale_log2;
  // this lane's fragment addresses, for d-step / d block 0 (see swa_attn_fwd_m16.hip)
  const uint32_t k_at = mine + n16 * 256 + ((g ^ swz16(n16)) << 4);
  const int v_row = 4 * g + (n16 >> 2);
  const uint32_t v_at = mine + kBlockBytes + v_row * kVRow + ((((n16 & 3) >> 1) ^ (kParts == 1 ? swz16(v_row) : swz_half(v_row))) << 4) + (n16 & 1) * 8;
  const bf16x8 ones = __builtin_bit_cast(bf16x8, u32x4{0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u});

  f32x4 oacc[kDb][2], lacc[2];
#pragma unroll
  for (int qt = 0; qt < 2; ++qt) {
#pragma unroll
    for (int db = 0; db < kDb; ++db) oacc[db][qt] = f32x4{0.f, 0.f, 0.f, 0.f};
    lacc[qt] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  float m_run[2] = {-INFINITY, -INFINITY}, neg_ref[2] = {0.f, 0.f};

  for (int b = block0; b < nblocks; b += kWaves) {
    const bool more = b + kWaves < nblocks;
    u32x4 k[2][4];
    land<kVTransfers>(true);                   // (V of this block is the newest)
    read_k_now(k_at, k);
    if (more) fetch_k(b + kWaves);
#pragma unroll
    for (int qt = 0; qt < 2; ++qt) asm volatile("" : "+v"(qf[qt][0]), "+v"(qf[qt][1]), "+v"(qf[qt][2]), "+v"(qf[qt][3]));
    const int key0 = key0_of(b), loaded = loaded_from(key0);
    f32x4 s[2][2];          // [key tile][query tile]: keys 16 kt + 4 g + i
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int qt = 0; qt < 2; ++qt) s[kt][qt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int qt = 0; qt < 2; ++qt)
          s[kt][qt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, k[kt][ks]), qf[qt][ks], s[kt][qt], 0, 0, 0);
    if (key0 + kKeys > seq || (kMask && key0 + kKeys > m_lo_first && key0 < m_hi)) {
      int own = loaded + 4 * g;
      asm volatile("" : "+v"(own));      // (sixteen sums of it are not worth keeping in registers for the rare block that is masked)
#pragma unroll
      for (int kt = 0; kt < 2; ++kt) {
        const int from = kt == 0 || key0 > loaded + 16 ? key0 : loaded + 16;
#pragma unroll
        for (int qt = 0; qt < 2; ++qt)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int key = own + kt * second + i;
            if (key < from || key >= seq || (kMask && key >= m_lo[qt] && key < m_hi)) s[kt][qt][i] = -INFINITY;
          }
      }
    }
    float m_new[2];
#pragma unroll
    for (int qt = 0; qt < 2; ++qt) {
      float top = s[0][qt][0];
#pragma unroll
      for (int i = 0; i < 4; ++i) top = fmaxf(top, fmaxf(s[0][qt][i], s[1][qt][i]));
      m_new[qt] = fmaxf(m_run[qt], col_max(top));
    }
    if (__builtin_amdgcn_ballot_w64(m_new[0] > m_run[0] || m_new[1] > m_run[1])) {
#pragma unroll
      for (int qt = 0; qt < 2; ++qt) {
        // (-inf only while every key so far was hidden from this query: nothing has been summed)
        const float alpha = m_new[qt] == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f((m_run[qt] - m_new[qt]) * c2);
        m_run[qt] = m_new[qt];
        neg_ref[qt] = m_new[qt] == -INFINITY ? 0.f : -m_new[qt] * c2;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          lacc[qt][i] *= alpha;
#pragma unroll
          for (int db = 0; db < kDb; ++db) oacc[db][qt][i] *= alpha;
        }
      }
    }
    u32x4 p[2];
#pragma unroll
    for (int qt = 0; qt < 2; ++qt)
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int i = 0; i < 4; i += 2)
          p[qt][2 * kt + i / 2] = pack_bf16x2(__builtin_amdgcn_exp2f(__builtin_fmaf(s[kt][qt][i], c2, neg_ref[qt])),
                                              __builtin_amdgcn_exp2f(__builtin_fmaf(s[kt][qt][i + 1], c2, neg_ref[qt])));
#pragma unroll
    for (int qt = 0; qt < 2; ++qt)
      lacc[qt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, __builtin_bit_cast(bf16x8, p[qt]), lacc[qt], 0, 0, 0);
    land<8>(more);
    bf16x8 v[kDb / 4][4];
    read_v_now<kParts>(v_at, v[0]);
    if constexpr (kParts == 1) read_v_now<kParts>(v_at ^ 128u, v[1]);
    if (more) fetch_v(b + kWaves);
#pragma unroll
    for (int db = 0; db < kDb; ++db)
#pragma unroll
      for (int qt = 0; qt < 2; ++qt)
        oacc[db][qt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v[db >> 2][db & 3], __builtin_bit_cast(bf16x8, p[qt]), oacc[db][qt], 0, 0, 0);
  }
  // (a wave without a block has yet to see its query land, in registers that are free from here on)
  asm volatile("s_waitcnt vmcnt(0)"
               : "+v"(qf[0][0]), "+v"(qf[0][1]), "+v"(qf[0][2]), "+v"(qf[0][3]), "+v"(qf[1][0]), "+v"(qf[1][1]), "+v"(qf[1][2]),
                 "+v"(qf[1][3])
               :
               : "memory");

  // ---- the waves meet -------------------------------------------------------------
  // Largest score and row sum of every wave first; each scales its own result to the common reference and the
  // total, and the eight scaled results are added up in wave order.
  if (lane < kQBlock) {      // lanes 0-15 the first query tile, 16-31 the second
    const f32x2 x = {lane < 16 ? m_run[0] : m_run[1], lane < 16 ? lacc[0][0] : lacc[1][0]};
    *reinterpret_cast<lds_f32x2*>(lds + kLdsStats + (wave * kQBlock + lane) * 8) = x;
  }
  __syncthreads();
#pragma unroll
  for (int qt = 0; qt < 2; ++qt) {
    f32x2 x[kWaves];
    float top = -INFINITY, total = 0.f;
#pragma unroll
    for (int u = 0; u < kWaves; ++u) {
      x[u] = *reinterpret_cast<lds_f32x2*>(lds + kLdsStats + (u * kQBlock + 16 * qt + n16) * 8);
      top = fmaxf(top, x[u][0]);
    }
    auto to_top = [&](float m) { return m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f((m - top) * c2); };
#pragma unroll
    for (int u = 0; u < kWaves; ++u) total += x[u][1] * to_top(x[u][0]);
    const float f = to_top(m_run[qt]) * (total > 0.f ? 1.0f / total : 0.f);
    const int r = 16 * qt + n16;
#pragma unroll
    for (int db = 0; db < kDb; ++db) {
      f32x4 o = oacc[db][qt];
#pragma unroll
      for (int i = 0; i < 4; ++i) o[i] *= f;
      *reinterpret_cast<lds_f32x4*>(lds + wave * kWaveLds + r * (512 / kParts) + (((4 * db + g) ^ n16) << 4)) = o;
    }
  }
  __syncthreads();
  {
    constexpr int kPieces = 2 / kParts;
    const int r = tid >> 4, c = kPieces * (tid & 15);    // row, first of its 16-byte pieces
#pragma unroll
    for (int e = 0; e < kPieces; ++e) sum[e] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < kWaves; ++u)
#pragma unroll
      for (int e = 0; e < kPieces; ++e) {
        const f32x4 x = *reinterpret_cast<lds_f32x4*>(lds + u * kWaveLds + r * (512 / kParts) + (((c + e) ^ (r & 15)) << 4));
#pragma unroll
        for (int i = 0; i < 4; ++i) sum[e][i] += x[i];
      }
  }
}

// log2 of the sum of the weights of row tid / 16, from what the waves left in LDS
__device__ __forceinline__ float row_lse(lds_char* lds, float c2) {
  float top = -INFINITY, total = 0.f;
  f32x2 x[kWaves];
#pragma unroll
  for (int u = 0; u < kWaves; ++u) {
    x[u] = *reinterpret_cast<lds_f32x2*>(lds + kLdsStats + (u * kQBlock + (threadIdx.x >> 4)) * 8);
    top = fmaxf(top, x[u][0]);
  }
#pragma unroll
  for (int u = 0; u < kWaves; ++u) total += x[u][0] == -INFINITY ? 0.f : x[u][1] * __builtin_amdgcn_exp2f((x[u][0] - top) * c2);
  return total > 0.f ? __builtin_amdgcn_logf(total) + top * c2 : -INFINITY;
}

template <typename Args>
__device__ __forceinline__ void write_row(Args& a, int head, int row, int q0, const f32x4 (&sum)[2]) {
  const int token = q0 + (threadIdx.x >> 4);
  if (token >= a.q_tokens) return;
  u32x4 x;
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    x[2 * e] = pack_bf16x2(sum[e][0], sum[e][1]);
    x[2 * e + 1] = pack_bf16x2(sum[e][2], sum[e][3]);
  }
  *reinterpret_cast<u32x4*>(a.out + row * a.o_st.row + head * a.o_st.head + (int64_t)token * a.o_st.token + 8 * (threadIdx.x & 15)) = x;
}

template <typename Args>
__device__ __forceinline__ void write_half_row(Args& a, int head, int row, int q0, int part, const f32x4& sum) {
  const int token = q0 + (threadIdx.x >> 4);
  if (token >= a.q_tokens) return;
  const u32x2 x = {pack_bf16x2(sum[0], sum[1]), pack_bf16x2(sum[2], sum[3])};
  *reinterpret_cast<u32x2*>(a.out + row * a.o_st.row + head * a.o_st.head + (int64_t)token * a.o_st.token + part * (kD / 2) + 4 * (threadIdx.x & 15)) = x;
}

}  // namespace wave
}  // namespace attn
}  // namespace sdv2

#endif  // SDV2KV_ATTN_WAVE_DEVICE_H
