// The kernel of sdv2_linear (linear.hip, which see) and its launch, for the sources that compile it.
#ifndef SDV2KV_LINEAR_KERNEL_H
#define SDV2KV_LINEAR_KERNEL_H

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>

#include "sdv2kv.h"
#include "sdv2kv_profile.h"
#include "sdv2kv_internal.h"
#include "attn_device.h"
#include "linear_args.h"

namespace {

using namespace sdv2::attn;
using namespace sdv2::linear;

constexpr int kThreads = 512;
constexpr int kRowBytes = kDepth * 2;
constexpr int kGroupTiles = 8;               // row tiles that are gone through together, all columns

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
  // Of three stages a buffer is filled again as soon as all of it has been read, half way through its own stage: else one
  // stage at most would be on its way.  (The waves then wait for their last reads before the barrier and not behind
  // it; with more stages that costs more than the stage in flight gives, 3120 x 1536 x 1536 18.6 -> 19.7 us.)
  constexpr bool kWhole = kStages == 3;
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
    if constexpr (!kWhole) {
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
    } else {
#pragma unroll
      for (int s = 0; s < kStages; ++s)
        if (s < stages) fetch(s, s * kStageBytes);
      if (stages >= kStages) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((kStages - 1) * kPieces) : "memory");
      else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      asm volatile("s_barrier" ::: "memory");
      // half way through stage t its own buffer is free, and t + 1 has to be there (what lies behind may be on its way)
      uint32_t buf = 0;
      int t = 0;
      for (; t + kStages - 1 < stages; ++t) {
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((kStages - 2) * kPieces) : "memory");
        asm volatile("s_barrier" ::: "memory");
        if (t + kStages < stages) fetch(t + kStages, buf);
        buf = buf == (kStages - 1) * kStageBytes ? 0 : buf + kStageBytes;
      }
      // the last stages, with nothing left to ask for
      static_for<kStages - 1>([&](auto jc) {
        constexpr int behind = kStages - 2 - decltype(jc)::value;          // stages behind this one
        if (t + behind < stages) {
          asm volatile("s_waitcnt vmcnt(%0)" ::"n"(behind > 1 ? (behind - 1) * kPieces : 0) : "memory");
          asm volatile("s_barrier" ::: "memory");
          ++t;
        }
      });
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
    if constexpr (kWhole) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
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
  if (kN % 2 == 0 && a.squares != nullptr) {
    // what a norm of the rows is to be made of: two fragments are 32 columns, four of each with every lane of a row
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

#endif  // SDV2KV_LINEAR_KERNEL_H
