// out = x W^T + bias in bf16 for gfx950 (MI355X): the projections around the
// attention (models/wan/causal_model.py:212-218, :389; wan_base/modules/model.py:181,
// :195) at the sizes of a chunk, where the vendor library's kernels leave the chip
// idle.  fp32 accumulation in the order of the contraction, 32 products at a time, one
// rounding after the bias; at every size tried the bits of the vendor library's.
//
// What bounds it: a chunk's projection is one round of workgroups, 24 steps of 64
// along a contraction of 1536.  A workgroup is four waves that multiply, one per
// SIMD, and four that fetch.  A wave's products need its LDS reads and LDS takes
// what the transfers bring, so the split of a tile over the waves decides: 2 x 2 waves
// of 80 x 64 read 9 fragments for 20 products (LDS busy 432 of 320 matrix cycles,
// the transfers' writes included).  Fetching is the work of waves of its own because a
// wave that waits for room in the memory pipe issues no products: with the transfers
// dealt out between the products of four waves 160 x 128 tiles took 15 us for what
// the products alone take 8.8 and the transfers alone 7.6; with waves for each, 10.
//
// In a stream the weights come from memory, a trip longer than the stages in
// flight: as many as LDS holds (seven of 96 x 64 instead of four: 512 x 1536 15.0 ->
// 13.1 us).  (Bringing lines to L2 ahead of that, by the waves that multiply, cost
// what it gave; tiles of 160 x 192, three stages, lost to the vendor's with cold
// weights, 34.5 against 33.4 us for 1560 x 4608.)
//
// The vendor's and this one, weights cold, x just written: 3120 x 1536 by 1536 x 1536
// 28.6 -> 22.8 us, 1560 x 1536 21.8 -> 18.0, 256 x 4608 25.5 -> 16.2; all warm
// 25.2 -> 20.1, 18.0 -> 14.9, 18.1 -> 10.2.
//
// Stages of 64 along the contraction lie in LDS as rows of 128 bytes (x's rows, then
// W's), 16-byte chunk c of row r at c ^ r % 8: 16 rows of one chunk are read without
// a bank conflict.  kStages of them are in use at a time.  Output: W's rows are the A operand, so a
// lane ends up with four neighbouring columns of a row; each wave turns its part
// through LDS and writes whole lines.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>

#include "sdv2kv.h"
#include "sdv2kv_profile.h"
#include "sdv2kv_internal.h"
#include "attn_device.h"

namespace {

using namespace sdv2::attn;

constexpr int kThreads = 512;
constexpr int kDepth = 64;                   // of a stage, along the contraction
constexpr int kRowBytes = kDepth * 2;
constexpr int kGroupTiles = 8;               // row tiles that are gone through together, all columns

struct LinearArgs {
  const uint16_t* x;
  const uint16_t* w;
  const uint16_t* bias;
  uint16_t* out;
  float* squares;                            // [row][n / 32], or null
  int64_t x_st, w_st, out_st;                // elements between rows
  int32_t m, stages;                         // rows; stages of the contraction
  int32_t row_tiles, col_tiles, square_groups;       // square_groups = n / 32
};

// Fragments in flight from LDS are nobody's to move: passing them through here, behind the wait, fixes that.
template <int N>
__device__ __forceinline__ void landed(u32x4 (&x)[N]) {
#pragma unroll
  for (int i = 0; i < N; ++i) asm volatile("" : "+v"(x[i]));
}

// Tile (32 kM) x (32 kN): 2 x 2 waves of (16 kM) x (16 kN).
template <int kM, int kN, int kStages>
__global__ __launch_bounds__(kThreads, 1)
void linear_kernel(const LinearArgs a) {
  constexpr int kTileM = 32 * kM, kTileN = 32 * kN, kRows = kTileM + kTileN, kStageBytes = kRows * kRowBytes;
  constexpr int kPieces = kRows / 32;        // transfers of 8 rows per fetching wave and stage
  static_assert(kStages >= 3 && kStages * kStageBytes <= 160 * 1024, "stages in LDS");
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  lds_char* lds = (lds_char*)smem;
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)lds);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave8 = __builtin_amdgcn_readfirstlane(tid >> 6), wave = wave8 & 3;
  const int n16 = lane & 15, g = lane >> 4;

  // Each XCD takes an eighth of the list of tiles: kGroupTiles row tiles, all columns, the next row tiles.
  const int total = a.row_tiles * a.col_tiles, xcd = blockIdx.x & 7;
  const int item = (int)(((int64_t)xcd * total) >> 3) + (blockIdx.x >> 3);
  if (item >= (int)(((int64_t)(xcd + 1) * total) >> 3)) return;
  const int group = item / (kGroupTiles * a.col_tiles), in_group = item - group * kGroupTiles * a.col_tiles;
  const int left = a.row_tiles - group * kGroupTiles, rows_in = left < kGroupTiles ? left : kGroupTiles;
  const int col = in_group / rows_in, m0 = (group * kGroupTiles + in_group - col * rows_in) * kTileM, n0 = col * kTileN;
  const int stages = a.stages;

  if (wave8 >= 4) {
    // ---- fetching: piece i (wave + 4 j) of a stage is rows 8 i .. 8 i + 7, lane l row l / 8, stored chunk l % 8
    const char* xb = uniform_pointer(a.x + m0 * a.x_st);
    const char* wb = uniform_pointer(a.w + n0 * a.w_st);
    const int r8 = lane >> 3;
    const uint32_t chunk = (uint32_t)(((lane & 7) ^ r8) << 4);
    uint32_t off[kPieces];
#pragma unroll
    for (int j = 0; j < kPieces; ++j) {
      int r = 8 * (wave + 4 * j) + r8;
      if (j < kTileM / 32) {
        r = m0 + r < a.m ? r : a.m - 1 - m0;               // (rows past the last repeat it; nobody writes them)
        off[j] = (uint32_t)r * (uint32_t)(a.x_st * 2) + chunk;
      } else {
        off[j] = (uint32_t)(r - kTileM) * (uint32_t)(a.w_st * 2) + chunk;
      }
    }
    auto fetch = [&](int stage, uint32_t buf) {
#pragma unroll
      for (int j = 0; j < kPieces; ++j)
        dma16((j < kTileM / 32 ? xb : wb) + (int64_t)stage * kRowBytes, off[j], lds0 + buf + (wave + 4 * j) * 1024);
    };
#pragma unroll
    for (int s = 0; s < kStages - 1; ++s)
      if (s < stages) fetch(s, s * kStageBytes);
    // stage 0 is there when at most the kStages - 2 behind it are in flight
    if (stages >= kStages - 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((kStages - 2) * kPieces) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    asm volatile("s_barrier" ::: "memory");
    uint32_t buf = (kStages - 1) * kStageBytes;
    for (int t = 0; t < stages; ++t) {
      // half way through stage t: stage t + 1 has to be there (t + 2 may be on its way), and t - 1's buffer is free
      if (kStages > 3 && t + kStages - 2 < stages) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((kStages - 3) * kPieces) : "memory");
      else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      asm volatile("s_barrier" ::: "memory");
      if (t + kStages - 1 < stages) fetch(t + kStages - 1, buf);
      buf = buf == (kStages - 1) * kStageBytes ? 0 : buf + kStageBytes;
    }
    __syncthreads();
    return;
  }

  // ---- multiplying
  const int wm = wave >> 1, wn = wave & 1;
  const int col0 = n0 + wn * 16 * kN;
  u32x2 bias[kN];
#pragma unroll
  for (int f = 0; f < kN; ++f)
    bias[f] = a.bias ? *reinterpret_cast<const u32x2*>(a.bias + col0 + 16 * f + 4 * g) : u32x2{0u, 0u};
  f32x4 acc[kN][kM];
#pragma unroll
  for (int fn = 0; fn < kN; ++fn)
#pragma unroll
    for (int fm = 0; fm < kM; ++fm) acc[fn][fm] = f32x4{0.f, 0.f, 0.f, 0.f};
  // this lane's 16 bytes of a fragment of 16 rows: row n16, chunk g of the stage's first 32, g + 4 of the second
  const uint32_t at = lds0 + n16 * kRowBytes + ((g ^ (n16 & 7)) << 4);
  const uint32_t xa = at + wm * (16 * kM * kRowBytes), wa = at + (kTileM + wn * 16 * kN) * kRowBytes;
  u32x4 xf[2][kM], wf[2][kN];
  asm volatile("s_barrier" ::: "memory");
  static_for<kM>([&](auto i) { xf[0][decltype(i)::value] = lds_read_b128<decltype(i)::value * 2048>(xa); });
  static_for<kN>([&](auto i) { wf[0][decltype(i)::value] = lds_read_b128<decltype(i)::value * 2048>(wa); });

  // 32 along the contraction: the products of fragments kP, and the next ones' reads dealt out between them
  auto step = [&](auto pc, uint32_t xr, uint32_t wr) {
    constexpr int kP = decltype(pc)::value, kReads = kM + kN, kProducts = kM * kN;
    constexpr int kEvery = kProducts / kReads > 0 ? kProducts / kReads : 1;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    landed(xf[kP]);
    landed(wf[kP]);
    __builtin_amdgcn_sched_barrier(0);
    auto read = [&](auto qc) {
      constexpr int q = decltype(qc)::value;
      if constexpr (q < kM) xf[kP ^ 1][q] = lds_read_b128<q * 2048>(xr);
      else wf[kP ^ 1][q - kM] = lds_read_b128<(q - kM) * 2048>(wr);
    };
    static_for<kProducts>([&](auto ic) {
      constexpr int i = decltype(ic)::value, fn = i / kM, fm = i % kM;
      acc[fn][fm] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wf[kP][fn]), __builtin_bit_cast(bf16x8, xf[kP][fm]),
                                                            acc[fn][fm], 0, 0, 0);
      if constexpr (i % kEvery == 0 && i / kEvery < kReads) read(std::integral_constant<int, i / kEvery < kReads ? i / kEvery : 0>{});
      if constexpr (i == kProducts - 1)
        static_for<kReads>([&](auto qc) {
          if constexpr (decltype(qc)::value * kEvery >= kProducts) read(qc);
        });
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  uint32_t buf = 0;
  for (int t = 0; t < stages; ++t) {
    const uint32_t next = buf == (kStages - 1) * kStageBytes ? 0 : buf + kStageBytes;
    step(std::integral_constant<int, 0>{}, (xa + buf) ^ 64u, (wa + buf) ^ 64u);
    asm volatile("s_barrier" ::: "memory");
    // (behind the last stage this reads what an earlier one left)
    step(std::integral_constant<int, 1>{}, xa + next, wa + next);
    buf = next;
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  landed(xf[0]);
  landed(wf[0]);
  __syncthreads();

  // ---- bias, rounding, whole lines
  constexpr int kOutBytes = 32 * kN + 16;    // of a row of this wave's part (padded against bank conflicts)
  static_assert(4 * 16 * kM * kOutBytes <= kStages * kStageBytes, "the output is turned in the stages' place");
  lds_char* mine = lds + wave * (16 * kM * kOutBytes);
#pragma unroll
  for (int fn = 0; fn < kN; ++fn) {
    const float b[4] = {__uint_as_float(bias[fn][0] << 16), __uint_as_float(bias[fn][0] & 0xffff0000u),
                        __uint_as_float(bias[fn][1] << 16), __uint_as_float(bias[fn][1] & 0xffff0000u)};
#pragma unroll
    for (int fm = 0; fm < kM; ++fm) {
      const f32x4 s = acc[fn][fm];
      const u32x2 y = {pack_bf16x2(s[0] + b[0], s[1] + b[1]), pack_bf16x2(s[2] + b[2], s[3] + b[3])};
      *reinterpret_cast<__attribute__((address_space(3))) u32x2*>(mine + (16 * fm + n16) * kOutBytes + 32 * fn + 8 * g) = y;
    }
  }
  const int row0 = m0 + wm * 16 * kM;
  if (a.squares != nullptr) {
    // what a norm of the rows is to be made of: two fragments are 32 columns, four of each with every lane of a row
    static_assert(kN % 2 == 0, "groups of 32 columns");
#pragma unroll
    for (int fm = 0; fm < kM; ++fm)
#pragma unroll
      for (int half = 0; half < kN / 2; ++half) {
        float sum = 0.f;
#pragma unroll
        for (int fn = 2 * half; fn < 2 * half + 2; ++fn) {
          const u32x2 y = *reinterpret_cast<__attribute__((address_space(3))) const u32x2*>(mine + (16 * fm + n16) * kOutBytes + 32 * fn + 8 * g);
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            const float lo = __uint_as_float(y[i] << 16), hi = __uint_as_float(y[i] & 0xffff0000u);
            sum = __builtin_fmaf(lo, lo, sum);
            sum = __builtin_fmaf(hi, hi, sum);
          }
        }
        sum += __shfl_xor(sum, 16);
        sum += __shfl_xor(sum, 32);
        const int r = row0 + 16 * fm + n16;
        if (g == 0 && r < a.m) a.squares[(int64_t)r * a.square_groups + (col0 >> 5) + half] = sum;
      }
  }
  uint16_t* dst = a.out + row0 * a.out_st + col0;
  constexpr int kChunks = 2 * kN;            // 16-byte chunks of a row
#pragma unroll
  for (int j = 0; j < (16 * kM * kChunks + 63) / 64; ++j) {
    const int i = j * 64 + lane, r = i / kChunks, c = i - r * kChunks;
    if (r < 16 * kM && row0 + r < a.m)
      *reinterpret_cast<u32x4*>(dst + r * a.out_st + c * 8) =
          *reinterpret_cast<__attribute__((address_space(3))) const u32x4*>(mine + r * kOutBytes + c * 16);
  }
}

// The tiles there are.  us_per_stage: what a stage of 64 takes, measured at a contraction of 1536 (24 stages, less 5 us of
// launch, start and end).
struct Tile {
  int m, n;
  float us_per_stage;
};
constexpr Tile kTiles[] = {{64, 64, 0.17f}, {96, 64, 0.19f}, {160, 64, 0.29f}, {96, 128, 0.30f}, {128, 128, 0.34f}, {160, 128, 0.51f}};
constexpr int kTileCount = sizeof(kTiles) / sizeof(kTiles[0]);
constexpr int kCus = 256;

int64_t tiles_of(const Tile& t, int64_t m, int64_t n) { return (m + t.m - 1) / t.m * (n / t.n); }

// The tile that takes least for m x n, or -1 where none divides n; a round is a tile per CU, and a second one costs more
// than its share.
int best_tile(int64_t m, int64_t n) {
  int best = -1;
  double best_us = 0;
  for (int i = 0; i < kTileCount; ++i) {
    if (n % kTiles[i].n != 0) continue;
    const int64_t rounds = (tiles_of(kTiles[i], m, n) + kCus - 1) / kCus;
    const double us = (double)rounds * kTiles[i].us_per_stage * (rounds > 1 ? 1.3 : 1.0);
    if (best < 0 || us < best_us) {
      best = i;
      best_us = us;
    }
  }
  return best;
}

template <int kM, int kN, int kStages>
int launch(const LinearArgs& a, hipStream_t stream) {
  constexpr int kLds = kStages * 32 * (kM + kN) * kRowBytes;
  // the stages exceed the static limit: ask for the dynamic size once per device
  static std::atomic<bool> ready[kMaxDevices];
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= kMaxDevices) return SDV2_ERR_LAUNCH;
  if (!ready[device].load(std::memory_order_acquire)) {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(linear_kernel<kM, kN, kStages>), hipFuncAttributeMaxDynamicSharedMemorySize, kLds) !=
        hipSuccess)
      return SDV2_ERR_LAUNCH;
    ready[device].store(true, std::memory_order_release);
  }
  const uint32_t tiles = (uint32_t)a.row_tiles * (uint32_t)a.col_tiles;
  sdv2::launch_timed(SDV2_KERNEL_LINEAR, linear_kernel<kM, kN, kStages>, dim3(8 * ((tiles + 7) / 8)), dim3(kThreads), kLds, stream, a);
  return hipGetLastError() == hipSuccess ? SDV2_OK : SDV2_ERR_LAUNCH;
}

}  // namespace

extern "C" int sdv2_linear_preferred(int64_t m, int32_t n, int32_t k) {
  if (m <= 0 || n <= 0 || k <= 0 || n % 64 != 0 || k % kDepth != 0) return 0;
  // One round of tiles (9360 x 1536 are three: 44.7 us, the vendor's 37.5), and contractions whose weights, cold, do not
  // outweigh the rest (464 x 3968 by 3968: 41.1, the vendor's 37.4, though 24.6 and 28.5 all warm).
  constexpr int kMostK = 2048;
  const int i = best_tile(m, n);
  return i >= 0 && tiles_of(kTiles[i], m, n) <= kCus && k <= kMostK;
}

extern "C" int sdv2_linear(const sdv2_linear_params* p) {
  if (!p) return SDV2_ERR_INVALID_ARG;
  if (p->dtype != SDV2_BF16 || p->n <= 0 || p->k <= 0 || p->n % 64 != 0 || p->k % kDepth != 0) return SDV2_ERR_UNSUPPORTED;
  if (p->m < 0) return SDV2_ERR_INVALID_ARG;
  if (p->m == 0) return SDV2_OK;
  if (!p->x || !p->weight || !p->out) return SDV2_ERR_INVALID_ARG;
  if ((reinterpret_cast<uintptr_t>(p->x) | reinterpret_cast<uintptr_t>(p->weight) | reinterpret_cast<uintptr_t>(p->out)) & 15)
    return SDV2_ERR_INVALID_ARG;
  if ((reinterpret_cast<uintptr_t>(p->bias) & 7) || (reinterpret_cast<uintptr_t>(p->row_squares) & 3)) return SDV2_ERR_INVALID_ARG;
  // rows of 16-byte vectors that do not overlap; offsets within a tile's rows are 32-bit
  constexpr int64_t kMostStride = 1 << 22;
  for (int64_t st : {p->x_row_stride, p->weight_row_stride})
    if (st < p->k || st % 8 != 0 || st > kMostStride) return SDV2_ERR_INVALID_ARG;
  if (p->out_row_stride < p->n || p->out_row_stride % 8 != 0) return SDV2_ERR_INVALID_ARG;
  const int i = best_tile(p->m, p->n);
  if (p->m > 0x7fffffff - 256 || tiles_of(kTiles[i], p->m, p->n) > (1 << 22)) return SDV2_ERR_UNSUPPORTED;
  LinearArgs a;
  a.x = static_cast<const uint16_t*>(p->x);
  a.w = static_cast<const uint16_t*>(p->weight);
  a.bias = static_cast<const uint16_t*>(p->bias);
  a.out = static_cast<uint16_t*>(p->out);
  a.x_st = p->x_row_stride;
  a.w_st = p->weight_row_stride;
  a.out_st = p->out_row_stride;
  a.m = (int32_t)p->m;
  a.squares = p->row_squares;
  a.square_groups = p->n / 32;
  a.stages = p->k / kDepth;
  a.row_tiles = (int32_t)((p->m + kTiles[i].m - 1) / kTiles[i].m);
  a.col_tiles = p->n / kTiles[i].n;
  hipStream_t stream = static_cast<hipStream_t>(p->stream);
  switch (i) {
    case 0: return launch<2, 2, 9>(a, stream);
    case 1: return launch<3, 2, 7>(a, stream);
    case 2: return launch<5, 2, 5>(a, stream);
    case 3: return launch<3, 4, 5>(a, stream);
    case 4: return launch<4, 4, 5>(a, stream);
    default: return launch<5, 4, 4>(a, stream);
  }
}
