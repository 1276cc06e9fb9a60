// Layout-changing copy of one layer's cache block, for the hand-off of a
// block between owners.
//
// The reference moves a block by broadcasting kv_cache1[i]["k"], ["v"] and the
// two index tensors from the donor and then shifting the receiver's
// global_end_index (streamv2v/communication/kv_cache_manager.py:66-82).  Its
// tensors are token-major [B, cap, H, 128]; this library keeps a cache
// head-major in HBM.  The wire format stays the reference's, so a block goes
// through this kernel once on either side: head-major -> token-major
// contiguous before it is sent, back after it was received, with the index
// update folded into the second copy (no host round trip for the indices).
//
// HBM-bound: every byte is read once and written once, so what counts is how the
// accesses lie.  A workgroup moves 4 KB, the 16 (bf16) or 8 (fp32) tokens of one head
// that its threads' single 16-byte vectors cover: whole 256 / 512-byte runs on either
// side whatever the two stride sets are, one contiguous piece on the head-major one, and
// no address arithmetic to speak of (the kernel before this one divided four 64-bit
// indices per thread).  Workgroups of neighbouring heads are neighbours, so that the
// token-major side is written or read in long runs at any moment.  K and V of a block
// are one launch.  Loads are streamed (non-temporal): a source is not read again, and
// what the cache holds of the other tensor is the next launch's source.
// Four blocks of 2 x 9360 tokens x 12 heads out to the wire and in again, 115 MB per
// tensor and copy: 481 us as sixteen launches of the kernel before, 307 as eight of this
// one (6.0 TB/s; an element-wise pass over 4 GiB reaches 6.25).  Several vectors a thread
// (2: 314, 4: 325, 12: 335) or cached loads (346) are slower; non-temporal stores too
// where the copies fit the memory-side cache (330), 3 % faster where they do not.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "sdv2kv.h"
#include "sdv2kv_profile.h"
#include "sdv2kv_internal.h"

namespace {

constexpr int kThreads = 256;
constexpr int64_t kMostItems = 1 << 23;      // workgroups of a tensor; past that each takes several (a grid has fewer than 2^32 threads)

typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;

struct Tensor {
  const char* src;
  char* dst;
  int64_t src_row, src_token, src_head;     // byte strides
  int64_t dst_row, dst_token, dst_head;
};
struct RelayoutArgs {
  Tensor first, second;                      // K and V of a block, say
  int64_t tokens, items;                     // items: (16 or 8 tokens, head) of one row
  int32_t heads;
  int32_t vec_shift;                         // log2(16-byte vectors per (token, head)): 4 bf16, 5 fp32
  int32_t both;                              // 1: even workgroups move `first`, odd ones `second`; 0: `first` only
  const int64_t* src_global;
  const int64_t* src_local;
  int64_t* dst_global;
  int64_t* dst_local;
  int64_t global_shift;
};

__global__ __launch_bounds__(kThreads) void cache_relayout_kernel(const RelayoutArgs a) {
  const int row = blockIdx.y;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    if (a.dst_global) a.dst_global[row] = a.src_global[row] + a.global_shift;
    if (a.dst_local) a.dst_local[row] = a.src_local[row];
  }
  const bool second = blockIdx.x & a.both;
  const Tensor t = second ? a.second : a.first;
  const int slot = threadIdx.x >> a.vec_shift, c = threadIdx.x & ((1 << a.vec_shift) - 1);
  const char* src = t.src + row * t.src_row + c * 16;
  char* dst = t.dst + row * t.dst_row + c * 16;
  for (int64_t item = blockIdx.x >> a.both; item < a.items; item += gridDim.x >> a.both) {
    // heads run fastest (a 64-bit division only where the index needs it)
    const int64_t group = item >> 32 ? item / a.heads : (int64_t)((uint32_t)item / (uint32_t)a.heads);
    const int64_t head = item - group * a.heads, token = group * (kThreads >> a.vec_shift) + slot;
    if (token < a.tokens) {
      const u32x4 x = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(src + token * t.src_token + head * t.src_head));
      *reinterpret_cast<u32x4*>(dst + token * t.dst_token + head * t.dst_head) = x;
    }
  }
}

bool stride_ok(const sdv2_stride3& s, int64_t elem) {
  // 16-byte vectors: every stride a multiple of 16 bytes
  return ((s.row * elem) % 16 == 0) && ((s.token * elem) % 16 == 0) && ((s.head * elem) % 16 == 0) && s.row >= 0 &&
         s.token >= 0 && s.head >= 0;
}

// What a call asks for, looked over; *with_data: there are elements to move
int check(const sdv2_relayout_params* p, bool* with_data) {
  if (!p) return SDV2_ERR_INVALID_ARG;
  if (p->head_dim != SDV2_HEAD_DIM) return SDV2_ERR_UNSUPPORTED;
  if (p->dtype != SDV2_BF16 && p->dtype != SDV2_F32) return SDV2_ERR_UNSUPPORTED;
  if (p->rows < 0 || p->tokens < 0 || p->heads < 0 || p->rows > 65535) return SDV2_ERR_INVALID_ARG;
  if ((p->dst_global_end_index && !p->src_global_end_index) || (p->dst_local_end_index && !p->src_local_end_index))
    return SDV2_ERR_INVALID_ARG;
  *with_data = p->rows > 0 && p->tokens > 0 && p->heads > 0;
  if (!*with_data) return SDV2_OK;
  const int64_t elem = p->dtype == SDV2_BF16 ? 2 : 4;
  if (!p->src || !p->dst) return SDV2_ERR_INVALID_ARG;
  if ((reinterpret_cast<uintptr_t>(p->src) | reinterpret_cast<uintptr_t>(p->dst)) & 15) return SDV2_ERR_INVALID_ARG;
  if (!stride_ok(p->src_stride, elem) || !stride_ok(p->dst_stride, elem)) return SDV2_ERR_INVALID_ARG;
  // distinct (token, head) elements of the destination must not overlap
  if (p->dst_stride.token < SDV2_HEAD_DIM && p->tokens > 1) return SDV2_ERR_INVALID_ARG;
  if (p->dst_stride.head < SDV2_HEAD_DIM && p->heads > 1) return SDV2_ERR_INVALID_ARG;
  if (p->dst_stride.row == 0 && p->rows > 1) return SDV2_ERR_INVALID_ARG;
  // (a row of 2^31 times 16 KB and more: no index below overflows)
  if (p->tokens > ((int64_t)0x7fffffff << 10) / ((int64_t)p->heads << (p->dtype == SDV2_BF16 ? 4 : 5))) return SDV2_ERR_INVALID_ARG;
  return SDV2_OK;
}

Tensor tensor_of(const sdv2_relayout_params& p) {
  const int64_t elem = p.dtype == SDV2_BF16 ? 2 : 4;
  return Tensor{static_cast<const char*>(p.src),  static_cast<char*>(p.dst),
                p.src_stride.row * elem, p.src_stride.token * elem, p.src_stride.head * elem,
                p.dst_stride.row * elem, p.dst_stride.token * elem, p.dst_stride.head * elem};
}

bool same_shape(const sdv2_relayout_params& a, const sdv2_relayout_params& b) {
  return a.dtype == b.dtype && a.rows == b.rows && a.heads == b.heads && a.tokens == b.tokens && a.stream == b.stream;
}

// the call p, together with the data of `other` where it is given (same shape, no indices of its own)
int launch(const sdv2_relayout_params& p, const sdv2_relayout_params* other, bool with_data) {
  const bool with_idx = p.dst_global_end_index || p.dst_local_end_index;
  if (p.rows == 0 || (!with_data && !with_idx)) return SDV2_OK;
  RelayoutArgs a{};
  a.first = tensor_of(p);
  if (other) a.second = tensor_of(*other);
  a.both = other ? 1 : 0;
  a.vec_shift = p.dtype == SDV2_BF16 ? 4 : 5;
  a.tokens = with_data ? p.tokens : 0;
  a.heads = p.heads;
  const int64_t per_group = kThreads >> a.vec_shift;
  a.items = with_data ? (p.tokens + per_group - 1) / per_group * p.heads : 0;
  a.src_global = p.src_global_end_index;
  a.src_local = p.src_local_end_index;
  a.dst_global = p.dst_global_end_index;
  a.dst_local = p.dst_local_end_index;
  a.global_shift = p.global_end_shift;
  int64_t blocks = a.items < kMostItems ? a.items : kMostItems;
  if (blocks < 1) blocks = 1;
  sdv2::launch_timed(SDV2_KERNEL_RELAYOUT, cache_relayout_kernel, dim3((unsigned)blocks << a.both, (unsigned)p.rows),
                     dim3(kThreads), 0, static_cast<hipStream_t>(p.stream), a);
  return hipGetLastError() == hipSuccess ? SDV2_OK : SDV2_ERR_LAUNCH;
}

}  // namespace

extern "C" int sdv2_cache_relayout(const sdv2_relayout_params* p) {
  bool with_data;
  const int status = check(p, &with_data);
  return status == SDV2_OK ? launch(*p, nullptr, with_data) : status;
}

extern "C" int sdv2_cache_relayout_pair(const sdv2_relayout_params* first, const sdv2_relayout_params* second) {
  bool first_data, second_data;
  int status = check(first, &first_data);
  if (status == SDV2_OK) status = check(second, &second_data);
  if (status != SDV2_OK) return status;
  if (first_data && second_data && same_shape(*first, *second) && !second->dst_global_end_index && !second->dst_local_end_index)
    return launch(*first, second, true);
  status = launch(*first, nullptr, first_data);
  return status == SDV2_OK ? launch(*second, nullptr, second_data) : status;
}
