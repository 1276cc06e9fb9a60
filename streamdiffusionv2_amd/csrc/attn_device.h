// What the bf16 attention kernels share (gfx950 only): the launch arguments,
// the layout of a work list over (row, head, key range, query tile), LDS reads
// and global->LDS transfers with hand-placed waits, packing, and the
// device-coherent accesses that carry partial results between workgroups.
#ifndef SDV2KV_ATTN_DEVICE_H
#define SDV2KV_ATTN_DEVICE_H

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <utility>

#include "sdv2kv.h"
#include "sdv2kv_internal.h"
#include "rope_device.h"
#include "attn_even_plan.h"

namespace sdv2 {
namespace attn {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(2))) float f32x2;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
typedef __attribute__((ext_vector_type(2))) uint32_t u32x2;
typedef __attribute__((ext_vector_type(2))) _Float16 f16x2;
typedef __attribute__((ext_vector_type(8))) _Float16 f16x8;
typedef __attribute__((address_space(3))) char lds_char;
typedef __attribute__((address_space(3))) int lds_int;

constexpr int kD = SDV2_HEAD_DIM;           // 128
constexpr int kQBlock = 32;                 // query rows per wave
constexpr int kKTile = 64;                  // keys per tile
constexpr int kTileBytes = kKTile * kD * 2; // 16 KB per matrix
constexpr int kIssuers = 4;                 // waves that issue the global->LDS transfers
constexpr int kPieces = 16 / kIssuers;      // global->LDS instructions per issuing wave and matrix tile
// The first of them, of eight waves.  Where a query tile has rows for four only, the other four move the tiles, so that
// nothing holds up a wave that has its SIMD to itself: 1 x 2560 x 12 heads against 9360 keys 144.2 -> 131.2 us, 1 x 1560 x
// 12 against themselves 30.4 -> 27.6, 1 x 640 x 40 against 512 15.0 -> 14.4.  (With a wave each for five to seven it is the
// other way round, 64.2 -> 67.8 us for 3120 x 12 against themselves, 83.0 -> 84.9 for 3840 x 12, and two of the spare waves for
// all transfers, 65.8 and 82.9, no better: waves that share a SIMD and do not run in step share it better.)
__host__ __device__ constexpr int first_issuer(int q_tile_rows) { return q_tile_rows <= kIssuers * kQBlock ? kIssuers : 0; }
constexpr int kStageBytes = 16384;          // epilogue staging per wave
constexpr int kMaxDevices = 64;
constexpr int kPartBlockHalves = kQBlock * kD;   // one block's partial output: 32 x 128 fp16 = 8 KB

struct AttnKernelArgs {
  const uint16_t* q;
  const uint16_t* k;
  const uint16_t* v;
  uint16_t* out;
  const int32_t* seq_lens;
  sdv2_stride3 q_st, k_st, v_st, o_st;
  int32_t rows, q_tokens, heads, max_seq_len;
  // Key ranges per (row, head): num_splits, except that of every group_pairs
  // consecutive (row, head) pairs the last more_pairs take num_splits + 1.
  // (Uniform: group_pairs = rows * heads, more_pairs = 0.)
  int32_t num_splits, group_pairs, more_pairs;
  int32_t q_tiles, per_group, total_items;        // query tiles per (row, head); work items per group and in all
  int32_t q_tile_rows;         // rows of a query tile
  FastDiv div_group, div_q_tiles, div_splits, div_splits_more, div_heads;
  float scale_log2;            // softmax_scale * log2(e)
  int32_t mask_block_tokens;   // 0 = no mask inside the chunk
  FastDiv div_mask_block;      // by mask_block_tokens
  // Split calls.  Partial results are kept per 32-row query block in the order
  // the registers hold them (see store_partial), q_blocks = ceil(q_tokens / 32).
  int32_t q_blocks;
  int32_t* tickets;            // [row][head][query tile], zero between calls
  uint16_t* part_o;            // [split][row][head][block][8 KB] fp16: normalised output / row scale
  float* part_lse;             // [split][row][head][block][32]   log2 sum exp
  float* part_scale;           // [split][row][head][block][32]   largest magnitude of the normalised row
  // Rotation of the queries inside the kernel (q is then the chunk's query
  // BEFORE RoPE): the complex128 table, or null when q arrives rotated.
  const double2* freqs;
  int32_t grid_w, frame_tokens, split_t, split_h;
  int64_t start_frame[SDV2_MAX_ROWS];
  // RMSNorm of the queries inside the kernel (q is then the raw projection):
  // the norm weight [heads * 128] and 1 / rms per (row, token), or null
  const uint16_t* q_norm_w;
  const float* q_inv_rms;
  // the same for a query that is not rotated: sums of squares of 32 columns each of (row, token), or null
  const float* q_row_squares;
  float q_norm_eps;
  sdv2::ChunkStarts chunk_starts;   // with the mask inside the chunk
};
template <typename Args>
__device__ __forceinline__ int row_chunk_start(Args& a, int row) {
  return sdv2::row_chunk_start<offsetof(AttnKernelArgs, chunk_starts)>(a.chunk_starts.device, row);
}

// The kernel's arguments, read where they lie each time: what is held from the start of a kernel to its end for the
// few places that need it crowds the scalar registers of the loop between: seventy of them lived in vector registers, and
// some of those in scratch memory.  (With the offsets of issue_tile out of the way too, no register of the m16 kernel is
// spilled: six layers of 1560 x 12 heads against 9360 keys 556 -> 541 us, layer calls and all.)
template <typename Args>
using late_args = const __attribute__((address_space(4))) Args;
template <typename Args>
__device__ __forceinline__ late_args<Args>& read_late() {
  auto* p = (late_args<Args>*)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return *p;
}
__device__ __forceinline__ FastDiv read_div(late_args<FastDiv>& d) { return FastDiv{d.mul, d.shift}; }

// v_max without the NaN-quieting canonicalisation fmaxf() drags in.
__device__ __forceinline__ float vmax(float a, float b) {
  float r;
  asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}

// exchange between the two lanes that share a query column (lane and lane ^ 32)
__device__ __forceinline__ float half_max(float x) {
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return vmax(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float half_sum(float x) {
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) {
  // fptrunc <2 x float> -> <2 x bfloat> selects v_cvt_pk_bf16_f32 (nearest-even)
  const f32x2 x = {lo, hi};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(x, bf16x2));
}

// two floats -> packed fp16 pair (lo in the low half), nearest-even
__device__ __forceinline__ uint32_t pack_f16x2(float lo, float hi) {
  const f32x2 x = {lo, hi};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(x, f16x2));
}

// ---------------------------------------------------------------------------
// LDS reads with hand-placed waits.  The compiler treats every LDS access as
// possibly aliasing an in-flight global->LDS transfer and would drain all
// counters before each dependent MFMA; issuing the reads as asm and tying an
// explicit s_waitcnt to the fragment about to be consumed keeps several reads
// in flight behind the matrix pipe.  LDS returns data in issue order, so
// lgkmcnt(N) means "all but the newest N reads have landed".
// ---------------------------------------------------------------------------
template <int... I, typename F>
__device__ __forceinline__ void static_for_impl(std::integer_sequence<int, I...>, F&& f) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_impl(std::make_integer_sequence<int, N>{}, f);
}

template <int kOffset>
__device__ __forceinline__ u32x4 lds_read_b128(uint32_t addr) {
  u32x4 r;
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(r) : "v"(addr), "n"(kOffset));
  return r;
}
template <int kOffset>
__device__ __forceinline__ u32x2 lds_read_tr16_b64(uint32_t addr) {
  u32x2 r;
  asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(r) : "v"(addr), "n"(kOffset));
  return r;
}
// The same reads for the exact pass, which is not pipelined: the value is
// waited for inside the statement and handed to compiler-generated MFMAs.
// (Absolute per-lane addresses as in the fast pass: taking them relative to
// the LDS base would keep a second copy of all sixteen alive across the
// streaming loop.)
__device__ __forceinline__ bf16x8 lds_read_b128_now(uint32_t addr) {
  u32x4 r;
  asm volatile("ds_read_b128 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=v"(r) : "v"(addr) : "memory");
  return __builtin_bit_cast(bf16x8, r);
}
__device__ __forceinline__ bf16x8 lds_read_tr16_b64x2_now(uint32_t addr_lo, uint32_t addr_hi) {
  u32x2 lo, hi;
  asm volatile("ds_read_b64_tr_b16 %0, %2\n\tds_read_b64_tr_b16 %1, %3\n\ts_waitcnt lgkmcnt(0)"
               : "=&v"(lo), "=&v"(hi) : "v"(addr_lo), "v"(addr_hi) : "memory");
  return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3));
}
// Optimisation passes may sink pure arithmetic down to its first use, which
// here is a whole pipeline slot later.  Passing a value through an empty
// volatile asm fixes the point by which it has to be computed.
__device__ __forceinline__ void pin(float& x) { asm volatile("" : "+v"(x)); }
__device__ __forceinline__ void pin(uint32_t& x) { asm volatile("" : "+v"(x)); }

// 16 bytes per lane from (wave-uniform base + this lane's 32-bit offset) to
// (wave-uniform LDS address + 16 * lane).  Written as asm so that the address
// stays "SGPR pair + one VGPR" instead of a 64-bit pointer per lane.
__device__ __forceinline__ void dma16(const char* uniform_base, uint32_t lane_off, uint32_t lds_dst) {
  asm volatile(
      "s_mov_b32 m0, %2\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %0, %1"
      :
      : "v"(lane_off), "s"(uniform_base), "s"(lds_dst)
      : "memory");
}

// ---------------------------------------------------------------------------
// Partial results travel between workgroups that may sit on different XCDs,
// each behind its own L2.  Fences would make that safe by writing back and
// invalidating a whole L2 per workgroup (measured: 13 us per workgroup, and the
// K / V lines the neighbours are streaming go with it).  Instead every access
// to a partial result is itself device-coherent, as a relaxed atomic access of
// agent scope is (the sc1 scope bit: the store writes through to memory, the
// load does not hit in a stale line), and the ticket orders them: a workgroup
// draws its ticket only after its stores have been acknowledged (vmcnt(0),
// barrier), and the last one reads only after it has drawn.  The 16-byte
// accesses have no atomic spelling in the language, so they are asm (8-byte
// atomics were measured 4 % of the whole kernel slower).
// A store of 16 bytes reads its data up to two cycles after its issue, which the
// compiler does not know of a store inside a statement: two wait states end it, or
// the next instruction might write those registers.
// ---------------------------------------------------------------------------
__device__ __forceinline__ void store_coherent_x4(void* base, const u32x4& w0, const u32x4& w1, const u32x4& w2,
                                                  const u32x4& w3) {
  asm volatile(
      "global_store_dwordx4 %0, %1, off sc1\n\t"
      "global_store_dwordx4 %0, %2, off offset:1024 sc1\n\t"
      "global_store_dwordx4 %0, %3, off offset:2048 sc1\n\t"
      "global_store_dwordx4 %0, %4, off offset:3072 sc1\n\t"
      "s_nop 1"
      :
      : "v"(base), "v"(w0), "v"(w1), "v"(w2), "v"(w3)
      : "memory");
}
// Four 16-byte pieces, 1 KB apart, of each of four blocks' partial outputs in one trip to memory.  Issue and wait
// are ONE asm statement: between a load's issue and its return the compiler believes the destination registers hold
// the value, and is free to copy them elsewhere and reuse them - as an address, say - for the load to overwrite when
// it lands.
__device__ __forceinline__ void load_coherent_4x4(const char* b0, const char* b1, const char* b2, const char* b3,
                                                  u32x4 (&w)[4][4]) {
  asm volatile(
      "global_load_dwordx4 %0, %16, off sc1\n\t"
      "global_load_dwordx4 %1, %16, off offset:1024 sc1\n\t"
      "global_load_dwordx4 %2, %16, off offset:2048 sc1\n\t"
      "global_load_dwordx4 %3, %16, off offset:3072 sc1\n\t"
      "global_load_dwordx4 %4, %17, off sc1\n\t"
      "global_load_dwordx4 %5, %17, off offset:1024 sc1\n\t"
      "global_load_dwordx4 %6, %17, off offset:2048 sc1\n\t"
      "global_load_dwordx4 %7, %17, off offset:3072 sc1\n\t"
      "global_load_dwordx4 %8, %18, off sc1\n\t"
      "global_load_dwordx4 %9, %18, off offset:1024 sc1\n\t"
      "global_load_dwordx4 %10, %18, off offset:2048 sc1\n\t"
      "global_load_dwordx4 %11, %18, off offset:3072 sc1\n\t"
      "global_load_dwordx4 %12, %19, off sc1\n\t"
      "global_load_dwordx4 %13, %19, off offset:1024 sc1\n\t"
      "global_load_dwordx4 %14, %19, off offset:2048 sc1\n\t"
      "global_load_dwordx4 %15, %19, off offset:3072 sc1\n\t"
      "s_waitcnt vmcnt(0)"
      : "=&v"(w[0][0]), "=&v"(w[0][1]), "=&v"(w[0][2]), "=&v"(w[0][3]), "=&v"(w[1][0]), "=&v"(w[1][1]), "=&v"(w[1][2]),
        "=&v"(w[1][3]), "=&v"(w[2][0]), "=&v"(w[2][1]), "=&v"(w[2][2]), "=&v"(w[2][3]), "=&v"(w[3][0]), "=&v"(w[3][1]),
        "=&v"(w[3][2]), "=&v"(w[3][3])
      : "v"(b0), "v"(b1), "v"(b2), "v"(b3)
      : "memory");
}
// the same for 32 contiguous bytes per lane
__device__ __forceinline__ void store_coherent_x2(void* base, const f32x4& w0, const f32x4& w1) {
  asm volatile(
      "global_store_dwordx4 %0, %1, off sc1\n\t"
      "global_store_dwordx4 %0, %2, off offset:16 sc1\n\t"
      "s_nop 1"
      :
      : "v"(base), "v"(w0), "v"(w1)
      : "memory");
}
__device__ __forceinline__ void load_coherent_x2(const void* base, f32x4& w0, f32x4& w1) {
  asm volatile(
      "global_load_dwordx4 %0, %2, off sc1\n\t"
      "global_load_dwordx4 %1, %2, off offset:16 sc1\n\t"
      "s_waitcnt vmcnt(0)"
      : "=&v"(w0), "=&v"(w1)
      : "v"(base)
      : "memory");
}
__device__ __forceinline__ void store_coherent(float* p, float x) {
  __hip_atomic_store(reinterpret_cast<uint32_t*>(p), __float_as_uint(x), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float load_coherent(const float* p) {
  return __uint_as_float(
      __hip_atomic_load(reinterpret_cast<const uint32_t*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}


struct QueryRope {
  const double2* freqs;        // null: the query arrives rotated
  int64_t start_frame;         // of this cache row
  int32_t grid_w, frame_tokens, split_t, split_h;
  // With norm_w (this head's 128 norm weights, offset like qp) the row is the
  // raw q projection: every slice is normalised with the token's 1 / rms as
  // the append kernel's fused norm would have done it (sdv2::normalise: two
  // roundings to bf16), then rotated.
  const uint16_t* norm_w;
  float inv_rms;
};

// the row's first absolute frame (constant indices and selects: indexing the by-value argument block with a
// run-time row would move the whole block, its pointers included, out of scalar registers)
template <typename Args>
__device__ __forceinline__ int64_t row_start_frame(Args& a, int row) {
  int64_t frame = a.start_frame[0];
  static_for<SDV2_MAX_ROWS - 1>([&](auto ic) {
    constexpr int i = decltype(ic)::value + 1;
    frame = row == i ? a.start_frame[i] : frame;
  });
  return frame;
}

// ---- the 16x16x32 kernels ------------------------------------------------------
// Where 16-byte chunk c of LDS row r (a key) is stored: position c ^ swz16(r).  A
// linear map of the four low bits of r with two properties.  Its upper three bits
// differ on any eight consecutive rows: a V read takes 8 keys x 32 bytes per half
// wave.  And swz16(12) = 1: a 16-byte K read is served to lanes 0-3, 12-15 and 20-27
// together (then 4-11, 16-19 and 28-31), that is, to keys 0-3 and 12-15 of one chunk
// and 4-11 of the next, and those two sets of positions must not meet.  Measured: no
// bank conflicts (with a swizzle that has the first property alone, 1.3 cycles per read).
__device__ __forceinline__ int swz16(int r) { return (r & 3) << 1 | ((r >> 2 ^ r >> 3) & 1) << 3 | (r >> 3 & 1); }

// over the four lanes that share a query column (lane, lane ^ 16, lane ^ 32, lane ^ 48)
__device__ __forceinline__ float col_max(float x) {
  x = half_max(x);
  auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return vmax(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float col_sum(float x) {
  x = half_sum(x);
  auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// One query row as the B operand of S^T = K Q^T: d-step ks takes the 8 elements
// 32 ks + 8 g of the row.  The row is the query before rotation and is rotated
// here, in the arithmetic of the append kernel, after the
// RMSNorm of the raw projection when the norm's weight is given.
__device__ __forceinline__ void load_query(const QueryRope& rope, const uint16_t* qp, int token, int g, bf16x8 (&qf)[4]) {
  const int fi = token / rope.frame_tokens;
  const int rem = token - fi * rope.frame_tokens;
  const int hi = rem / rope.grid_w;
  const int wi = rem - hi * rope.grid_w;
  const int64_t frame = rope.start_frame + fi;
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) {
    double2 cs[4];
    sdv2::load_rotation(rope.freqs, kD / 2, rope.split_t, rope.split_h, 4 * ks + g, frame, hi, wi, cs);
    sdv2::Vec8<uint16_t> x = sdv2::Vec8<uint16_t>::load(qp + 32 * ks);
    if (rope.norm_w) x = sdv2::normalise(x, rope.inv_rms, sdv2::Vec8<uint16_t>::load(rope.norm_w + 32 * ks));
    qf[ks] = __builtin_bit_cast(bf16x8, sdv2::rotate(x, cs).raw);
  }
}

// (the transfers take their base addresses from scalar registers: say so to the compiler)
__device__ __forceinline__ const char* uniform_pointer(const void* ptr) {
  const uint64_t x = reinterpret_cast<uint64_t>(ptr);
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)x), hi = __builtin_amdgcn_readfirstlane((uint32_t)(x >> 32));
  return reinterpret_cast<const char*>(((uint64_t)hi << 32) | lo);
}

// Workgroups are dealt to the eight XCDs round robin by id, and each XCD has
// its own L2.  Work items are ordered so that the query tiles of one (row,
// head, key split) are neighbours, and XCD x takes the x-th eighth of that
// list: the workgroups that stream the same K / V run on the same XCD at the
// same time and all but the first fetch of a tile hit in L2.
//
// With a mixed split count a group of (row, head) pairs is one XCD's share:
// its pairs with fewer, longer key ranges come first, so that the workgroups
// the dispatcher hands out last are the short ones (longest first is what
// packs unequal pieces best onto the CUs).
struct WorkItem {
  int qtile, head, row, split, nsplits;
  // false: this workgroup has nothing to do
  __device__ __forceinline__ bool decode(const AttnKernelArgs& a, int block_id) {
    const int xcd = block_id & 7;
    const int first = (int)(((int64_t)xcd * a.total_items) >> 3);
    const int end = (int)(((int64_t)(xcd + 1) * a.total_items) >> 3);
    const int item = first + (block_id >> 3);
    if (item >= end) return false;
    const int group = a.div_group(item);
    const int lo_pairs = a.group_pairs - a.more_pairs;
    int piece = a.div_q_tiles(item - group * a.per_group);          // (pair, split) within the group
    qtile = item - group * a.per_group - piece * a.q_tiles;
    int pair = group * a.group_pairs;
    int in_group;
    if (piece < lo_pairs * a.num_splits) {
      nsplits = a.num_splits;
      in_group = a.div_splits(piece);
    } else {
      nsplits = a.num_splits + 1;
      piece -= lo_pairs * a.num_splits;
      in_group = a.div_splits_more(piece);
      pair += lo_pairs;
    }
    split = piece - in_group * nsplits;
    pair += in_group;
    row = a.div_heads(pair);
    head = pair - row * a.heads;
    return true;
  }
};
// host: everything decode() needs, for query tiles of q_tile_rows rows
inline void set_work_list(AttnKernelArgs* a, int q_tile_rows, int parts = 1) {
  a->q_tile_rows = q_tile_rows;
  a->q_tiles = (a->q_tokens + q_tile_rows - 1) / q_tile_rows * parts;       // (every tile as often as it has parts)
  a->per_group = a->q_tiles * ((a->group_pairs - a->more_pairs) * a->num_splits + a->more_pairs * (a->num_splits + 1));
  a->total_items = a->rows * a->heads / a->group_pairs * a->per_group;
  a->div_group = FastDiv::by((uint32_t)a->per_group);
  a->div_q_tiles = FastDiv::by((uint32_t)a->q_tiles);
  a->div_splits = FastDiv::by((uint32_t)a->num_splits);
  a->div_splits_more = FastDiv::by((uint32_t)a->num_splits + 1);
  a->div_heads = FastDiv::by((uint32_t)a->heads);
}

// what the kernel of equal shares is launched with (swa_attn_fwd_even.hip)
struct EvenArgs {
  AttnKernelArgs call;         // (first: its helpers read fields where the launch's arguments lie)
  EvenPlan plan;
  float* part_o;               // [workgroup][0: rest or middle of an item, 1: start of one][128 KB] fp32: normalised output
  float* part_lse;             // [workgroup][the same][256]   log2 sum exp
};
constexpr int kEvenPartFloats = 256 * kD;
constexpr int kEvenPartRows = 256;

// the kernel on 16x16x32 matrix instructions (swa_attn_fwd_m16.hip), and for query tiles of at most four blocks
int launch_m16(const AttnKernelArgs& a, uint32_t workgroups, hipStream_t stream);
int launch_m16_few(const AttnKernelArgs& a, uint32_t workgroups, hipStream_t stream);
// ... of five or six blocks, the last ones shared by several waves (no mask)
int launch_m16_shared(const AttnKernelArgs& a, uint32_t workgroups, hipStream_t stream);
// the kernel whose waves share the keys of one query block (swa_attn_fwd_wave.hip)
int launch_wave(const AttnKernelArgs& a, uint32_t workgroups, hipStream_t stream);
// ... and two workgroups a block, each with half of V's columns: query tile 2 i + part of the work list (no rotation)
int launch_wave_half(const AttnKernelArgs& a, uint32_t workgroups, hipStream_t stream);

// the same with equal shares of the key tiles for all workgroups (swa_attn_fwd_even.hip)
int launch_even(const EvenArgs& a, hipStream_t stream);

}  // namespace attn
}  // namespace sdv2

#endif  // SDV2KV_ATTN_DEVICE_H
