// Grouped W8A16 on GGUF Q8_0 weights for decode batches and mid-size prefills: the contract
// and arithmetic of gguf_q8.hip (csrc/gguf_q8_packed.cu:161-285),
//
//   out[i, g, j] = bf16_rn(sum_t x[i, g, t] * bf16_rn(codes[g, j, t] * scales[g, j, t / 32]))
//
// with FP32 sums. The 256 x 128 and 128 x 128 tiles of gguf_q8.hip leave most CUs idle
// below about a thousand rows (M = 32, N = K = 4096: 32 workgroups, 38 us, whatever M is),
// and its M <= 16 kernel reads 16 rows x 64 bytes per load. Here a tile is picked per shape
// (tile_plan.h, kGgufTiles) so that the tiles fill the CUs about once.
//
// One workgroup of eight waves per tile, in KG = 8 or 4 K groups. A stage is 32 KG values
// of K in an LDS ring filled by buffer_load ... lds: x rows (BF16), code rows and block
// scales, all as they lie in memory. Each wave takes one 32-value step of the stage, one
// scale block: it reads its x and code fragments (double-buffered in registers),
// dequantizes the codes right before their MFMAs and keeps an FP32 sum of its K group. A
// weight is dequantized once per workgroup, since the waves of a K group split N, not M.
// The groups' sums are added through the ring at the end, in ascending group order.
//
// What bounds it: no one thing. At 128 x 128 a stage takes 2,100-2,350 cycles against 1,024
// of MFMAs; without the copies, the dequantization or the scale reads (timing only) it was
// 10-20% faster each. Tried and dropped: each block's dequantization interleaved with the
// previous block's MFMAs (0-4% slower). The K tail is masked only outside the steady loop,
// soffsets stay scalar and the code words are opaque until their use (the compiler
// otherwise splits each byte conversion in three): 41.0 against 62.8 us at M = 1000.
//
// Measured on MI355X, gguf_q8.hip's kernels in parentheses, us (three rotated weight
// copies): N = K = 8192: M = 1 14.4 (21.2), 16 14.8 (23.1), 32 16.8 (73.5), 128 30.1
// (74.8), 500 73.0 (83.5); N = K = 4096: M = 16 7.6 (8.9), 32 9.1 (38.4), 256 17.6 (40.0),
// 500 25.0 (40.6), 1000 39.4 (43.4); N = 1925, K = 2176: M = 32 6.0 (22.6). Over 162 shapes
// the time fell by 39% in the mean. From about 2000 rows the 256 x 128 tiles are faster
// (M = 2048, N = K = 4096: 66 against 78 us) and stay.
#include <climits>
#include <type_traits>

#include "ci8_device.h"
#include "launch.h"

namespace ci8 {
namespace {

constexpr int kXcds = 8;
constexpr int kLdsLimit = 160 * 1024;

__device__ __forceinline__ f32x4 mfma_bf16(u32x4 a, u32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                 __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// The value itself; the compiler does not move work on it above this point.
__device__ __forceinline__ uint32_t opaque(uint32_t value) {
  asm volatile("" : "+v"(value));
  return value;
}

// The largest divisor of n that is at most `most` (>= 1).
constexpr int largest_divisor(int n, int most) {
  int d = most < n ? most : n;
  while (d > 1 && n % d) --d;
  return d;
}

template <int BM_, int BN_>
struct GgufRingConfig {
  static constexpr int BM = BM_, BN = BN_;
  static constexpr int kWaves = 8, kThreads = 64 * kWaves;
  static_assert(kThreads == kGgufRingThreads, "tile_plan.h");
  static constexpr int WN = BM * BN >= 64 * 64 ? 2 : 1;  // waves of one K group, along n
  static constexpr int KG = kWaves / WN;                 // K groups
  static constexpr int TM = BM / 16, TN = BN / WN / 16;
  static constexpr int BK = 32 * KG;                  // K values per stage: one step a wave
  static constexpr int kXRow = 2 * BK, kWRow = BK, kSRow = BK / 16;  // bytes of a stage's row
  static constexpr int kXChunks = kXRow / 16, kWChunks = kWRow / 16;
  static constexpr int kXCopyRows = 1024 / kXRow, kWCopyRows = 1024 / kWRow;
  static constexpr int kXCopies = BM / kXCopyRows, kWCopies = BN / kWCopyRows;
  static constexpr int kSCopies = (BN * kSRow + 255) / 256;  // 4 bytes a lane
  static constexpr int kCopies = (kXCopies + kWCopies + kWaves - 1) / kWaves;  // per wave
  static constexpr int kWBase = BM * kXRow, kSBase = kWBase + BN * kWRow;
  static constexpr int kStageBytes = kSBase + kSCopies * 256;
  static constexpr int kJunk = 1024 + 256;  // copies past the stage's last
  static constexpr int kFit = (kLdsLimit - kJunk) / kStageBytes;
  static constexpr int kSlots = kFit < 4 ? kFit : 4;
  static constexpr int kRingBytes = kSlots * kStageBytes;
  // K groups' partial sums: m blocks per pass through the ring.
  static constexpr int kPassTM = largest_divisor(TM, kRingBytes / (kWaves * TN * 1024));
  static constexpr int kLdsBytes = kRingBytes + kJunk;
  static_assert(BM % 16 == 0 && BN % (WN * 16) == 0, "16-row MFMA blocks");
  static_assert(kXCopies * kXCopyRows == BM && kWCopies * kWCopyRows == BN, "whole copies");
  static_assert(kSCopies <= kWaves, "one scale copy a wave");
  static_assert(kSlots >= 3 && kWaves * kPassTM * TN * 1024 <= kRingBytes, "LDS");
  static_assert((kSlots - 1) * (kCopies + 1) < 64, "vmcnt");
};

// Waits until at most `after` stages (kAfter at most) of kCopies copies are in flight.
template <int kCopies, int kAfter>
__device__ __forceinline__ void wait_stages(int after) {
  if constexpr (kAfter <= 0) {
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
  } else {
    if (after >= kAfter)
      __builtin_amdgcn_s_waitcnt(vmcnt_imm(kAfter * kCopies));
    else
      wait_stages<kCopies, kAfter - 1>(after);
  }
}

template <class C>
__global__ void __launch_bounds__(C::kThreads, 1) gguf_ring_kernel(
    const uint16_t* __restrict__ x, const int8_t* __restrict__ codes,
    const uint16_t* __restrict__ scales, uint16_t* __restrict__ out, int m, int n, int k,
    int groups, int64_t xs, int64_t xg, int tiles_m, int tiles_n, bool vec_n) {
  extern __shared__ __attribute__((aligned(1024))) char lds_raw[];
  auto* lds = (char __attribute__((address_space(3)))*)(lds_raw);
  using lds_u32x4 = __attribute__((address_space(3))) u32x4;
  using lds_u32x2 = __attribute__((address_space(3))) u32x2;
  using lds_f32x4 = __attribute__((address_space(3))) f32x4;
  using lds_u16 = __attribute__((address_space(3))) uint16_t;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kg = wave / C::WN, wn = wave % C::WN;

  // Workgroup -> tile: each XCD runs a contiguous range of tiles, m fastest, group by
  // group, so the tiles that share weights fetch them into one XCD's L2.
  const int tiles = tiles_m * tiles_n * groups;
  int logical = blockIdx.x;
  {
    const int per = tiles / kXcds, extra = tiles % kXcds;
    const int xcd = logical % kXcds, idx = logical / kXcds;
    logical = (xcd < extra ? xcd * (per + 1) : extra * (per + 1) + (xcd - extra) * per) + idx;
  }
  const int g = logical / (tiles_m * tiles_n), tile = logical % (tiles_m * tiles_n);
  const int m0 = tile % tiles_m * C::BM, n0 = tile / tiles_m * C::BN;
  const int ns = (k + C::BK - 1) / C::BK;
  const uint16_t* gx = x + int64_t(g) * xg;
  const int8_t* gcodes = codes + int64_t(g) * n * k;
  const uint16_t* gscales = scales + int64_t(g) * n * (k / 32);
  // The ranges end with the last row's last value; rows past M or N and chunks past K get
  // out-of-range offsets, so padding and other groups' values are never taken for data.
  const uint32_t x_bytes = uint32_t((int64_t(m - 1) * xs + k) * 2);
  const uint32_t w_bytes = uint32_t(int64_t(n) * k);

  // 16-byte copies b = i * kWaves + wave: x rows, then code rows, then junk; the wave's
  // scale copy last.
  uint32_t c_off[C::kCopies], s_off;
  int c_unit[C::kCopies];  // bytes of a K value: 2 (x) or 1 (codes)
  // LDS rows hold their 16-byte chunks XOR-swizzled by the row, as the fragment reads expect.
  auto x_chunk = [&] __device__(int b) __attribute__((always_inline)) {
    const int row = b * C::kXCopyRows + lane / C::kXChunks;
    return (lane % C::kXChunks) ^ (row & (C::kXChunks < 16 ? C::kXChunks - 1 : 15));
  };
  auto w_chunk = [&] __device__(int b) __attribute__((always_inline)) {
    const int row = (b - C::kXCopies) * C::kWCopyRows + lane / C::kWChunks;
    return (lane % C::kWChunks) ^ (row & (C::kWChunks - 1));
  };
#pragma unroll
  for (int i = 0; i < C::kCopies; ++i) {
    const int b = i * C::kWaves + wave;
    c_off[i] = kOutOfRange;
    c_unit[i] = __builtin_amdgcn_readfirstlane(b < C::kXCopies ? 2 : 1);
    if (b < C::kXCopies) {
      const int row = m0 + b * C::kXCopyRows + lane / C::kXChunks;
      if (row < m) c_off[i] = uint32_t(row * xs * 2) + uint32_t(x_chunk(b) * 16);
    } else if (b < C::kXCopies + C::kWCopies) {
      const int row = n0 + (b - C::kXCopies) * C::kWCopyRows + lane / C::kWChunks;
      if (row < n) c_off[i] = uint32_t(row) * uint32_t(k) + uint32_t(w_chunk(b) * 16);
    }
  }
  constexpr int kSLanes = C::kSRow / 4;  // lanes of a row's scales
  const int s_row = n0 + wave * (64 / kSLanes) + lane / kSLanes;
  s_off = wave < C::kSCopies && s_row < n && wave * (64 / kSLanes) + lane / kSLanes < C::BN
              ? uint32_t(s_row) * uint32_t(k / 16) + uint32_t(lane % kSLanes * 4)
              : kOutOfRange;
  // whole: the stage lies within K (only the last one may not).
  const bool exact_k = k % C::BK == 0;
  auto copy = [&] __device__(int slot, int k0, int i, bool whole) __attribute__((always_inline)) {
    const int b = i * C::kWaves + wave;
    uint32_t off = c_off[i];
    const int at = k0 * c_unit[i];
    const bool is_x = b < C::kXCopies, is_w = !is_x && b < C::kXCopies + C::kWCopies;
    if (!whole && !exact_k && k0 + (is_x ? x_chunk(b) * 8 : w_chunk(b) * 16) >= k) off = kOutOfRange;
    const int to = is_x ? slot * C::kStageBytes + b * 1024
                   : is_w ? slot * C::kStageBytes + C::kWBase + (b - C::kXCopies) * 1024
                          : C::kRingBytes;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        make_rsrc(is_x ? static_cast<const void*>(gx) : gcodes, is_x ? x_bytes : w_bytes),
        reinterpret_cast<lds_void*>(lds + to), 16, off,
        at, 0, 0);
  };
  auto copy_scales = [&] __device__(int slot, int k0, bool whole) __attribute__((always_inline)) {
    uint32_t off = s_off;
    if (!whole && !exact_k && k0 + lane % kSLanes * 64 >= k) off = kOutOfRange;
    const int to = wave < C::kSCopies ? slot * C::kStageBytes + C::kSBase + wave * 256
                                      : C::kRingBytes + 1024;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(make_rsrc(gscales, w_bytes / 16),
                                             reinterpret_cast<lds_void*>(lds + to), 4, off,
                                             k0 / 16, 0, 0);
  };
  auto copy_stage = [&] __device__(int slot, int t) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < C::kCopies; ++i) copy(slot, t * C::BK, i, false);
    copy_scales(slot, t * C::BK, false);
  };

  // Fragments of K group kg: K values 32 kg + 8 (lane / 16) .. + 7 of the stage.
  const int f_row = lane & 15, f_group = lane >> 4;
  const int x_base = f_row * C::kXRow +
                     ((4 * kg + f_group) ^ (f_row & (C::kXChunks < 16 ? C::kXChunks - 1 : 15))) * 16;
  const int w_base = C::kWBase + (wn * C::TN * 16 + f_row) * C::kWRow +
                     ((2 * kg + f_group / 2) ^ (f_row & (C::kWChunks - 1))) * 16 + (f_group & 1) * 8;
  const int s_base = C::kSBase + (wn * C::TN * 16 + f_row) * C::kSRow + 2 * kg;
  u32x4 xf[2][C::TM];
  u32x2 wf[2][C::TN];
  uint32_t sf[2][C::TN];
  auto read = [&] __device__(int buf, int slot) __attribute__((always_inline)) {
    const auto* s = lds + slot * C::kStageBytes;
#pragma unroll
    for (int i = 0; i < C::TN; ++i) {
      wf[buf][i] = *reinterpret_cast<const lds_u32x2*>(s + w_base + i * 16 * C::kWRow);
      sf[buf][i] = *reinterpret_cast<const lds_u16*>(s + s_base + i * 16 * C::kSRow);
    }
#pragma unroll
    for (int j = 0; j < C::TM; ++j)
      xf[buf][j] = *reinterpret_cast<const lds_u32x4*>(s + x_base + j * 16 * C::kXRow);
  };
  auto barrier = [&] __device__() __attribute__((always_inline)) {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };

  f32x4 acc[C::TM][C::TN];
#pragma unroll
  for (int j = 0; j < C::TM; ++j)
#pragma unroll
    for (int i = 0; i < C::TN; ++i) acc[j][i] = f32x4{0, 0, 0, 0};

  for (int t = 0; t < C::kSlots && t < ns; ++t) copy_stage(t, t);
  wait_stages<C::kCopies + 1, C::kSlots - 1>(min(ns, C::kSlots) - 1);
  barrier();
  read(0, 0);
  // Eight codes of one channel and their block's scale -> BF16 weights bf16_rn(code * s).
  auto dequant = [&] __device__(const u32x2& words, uint32_t s16) __attribute__((always_inline)) {
    const float s = float(__builtin_bit_cast(_Float16, uint16_t(s16)));
    u32x4 w;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const uint32_t word = opaque(words[h]);
      w[2 * h] = pack_bf16x2(float(int8_t(word)) * s, float(int8_t(word >> 8)) * s);
      w[2 * h + 1] = pack_bf16x2(float(int8_t(word >> 16)) * s, float(int8_t(word >> 24)) * s);
    }
    return w;
  };

  int slot = 0;  // t % kSlots
  // Stage t, its fragments in register buffer `parity`. kSteady: stages t + 1 and t +
  // kSlots exist, and stage t + kSlots lies within K.
  auto iteration = [&] __device__(int t, auto parity, auto steady) __attribute__((always_inline)) {
    constexpr int buf = decltype(parity)::value;
    constexpr bool kSteady = decltype(steady)::value;
    const int next = slot + 1 == C::kSlots ? 0 : slot + 1;
    __builtin_amdgcn_sched_barrier(0);
    // This wave has read stage t, and its copies of stage t + 1 have landed; past the
    // barrier, every wave's, so stage t + 1 can be read and the slot of stage t refilled.
    __builtin_amdgcn_s_waitcnt(lgkmcnt0_imm());
    wait_stages<C::kCopies + 1, C::kSlots - 2>(
        kSteady ? C::kSlots - 2 : max(0, min(C::kSlots - 2, ns - 2 - t)));
    barrier();
    if (kSteady || t + 1 < ns) read(buf ^ 1, next);
    if (!kSteady && t + C::kSlots < ns) copy_stage(slot, t + C::kSlots);
    const int k0 = (t + C::kSlots) * C::BK;
    // One step per n block: dequantize its fragment, then TM MFMAs, with the copies spread.
    constexpr int kAll = C::kCopies + 1;
#pragma unroll
    for (int i = 0; i < C::TN; ++i) {
      if (kSteady) {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int c = i * kAll / C::TN; c < (i + 1) * kAll / C::TN; ++c) {
          if (c < C::kCopies)
            copy(slot, k0, c, true);
          else
            copy_scales(slot, k0, true);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      const u32x4 w = dequant(wf[buf][i], sf[buf][i]);
#pragma unroll
      for (int j = 0; j < C::TM; ++j) acc[j][i] = mfma_bf16(w, xf[buf][j], acc[j][i]);
    }
    __builtin_amdgcn_sched_barrier(0);
    slot = next;
  };
  using Even = std::integral_constant<int, 0>;
  using Odd = std::integral_constant<int, 1>;
  int t = 0;
  for (; t + 2 + C::kSlots < ns; t += 2) {
    iteration(t, Even{}, std::true_type{});
    iteration(t + 1, Odd{}, std::true_type{});
  }
  for (; t + 1 < ns; t += 2) {
    iteration(t, Even{}, std::false_type{});
    iteration(t + 1, Odd{}, std::false_type{});
  }
  if (t < ns) iteration(t, Even{}, std::false_type{});

  // Partial sums of the K groups, added in ascending group order: m blocks in passes of
  // kPassTM; group kg finishes the blocks (j, i) with (j * TN + i) % KG == kg.
  auto* part = reinterpret_cast<lds_f32x4*>(lds);
#pragma unroll
  for (int p = 0; p < C::TM / C::kPassTM; ++p) {
    __syncthreads();
#pragma unroll
    for (int j = 0; j < C::kPassTM; ++j)
#pragma unroll
      for (int i = 0; i < C::TN; ++i)
        part[((wave * C::kPassTM + j) * C::TN + i) * 64 + lane] = acc[p * C::kPassTM + j][i];
    __syncthreads();
#pragma unroll
    for (int b0 = 0; b0 < C::kPassTM * C::TN; b0 += C::KG) {
      const int b = b0 + kg;
      if (b >= C::kPassTM * C::TN) continue;  // uniform over the wave
      f32x4 sum = part[(wn * C::kPassTM * C::TN + b) * 64 + lane];
#pragma unroll
      for (int q = 1; q < C::KG; ++q)
        sum += part[((q * C::WN + wn) * C::kPassTM * C::TN + b) * 64 + lane];
      const int j = p * C::kPassTM + b / C::TN, i = b % C::TN;
      const int row = m0 + j * 16 + f_row;
      const int col = n0 + (wn * C::TN + i) * 16 + 4 * f_group;
      if (row >= m || col >= n) continue;
      uint16_t* dst = out + (int64_t(row) * groups + g) * n + col;
      if (vec_n) {
        *reinterpret_cast<u32x2*>(dst) =
            u32x2{pack_bf16x2(sum[0], sum[1]), pack_bf16x2(sum[2], sum[3])};
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (col + e < n) dst[e] = uint16_t(f32_to_bf16(sum[e]));
      }
    }
  }
}

template <class C>
hipError_t run_gguf_ring(const void* x, const int8_t* codes, const void* scales, void* out,
                         int m, int n, int k, int groups, int64_t xs, int64_t xg,
                         hipStream_t stream) {
  auto kernel = gguf_ring_kernel<C>;
  if (const hipError_t e = prepare_lds<gguf_ring_kernel<C>>(C::kLdsBytes); e != hipSuccess)
    return e;
  const int tiles_m = (m + C::BM - 1) / C::BM, tiles_n = (n + C::BN - 1) / C::BN;
  const bool vec_n = n % 4 == 0 && reinterpret_cast<uintptr_t>(out) % 8 == 0;
  kernel<<<unsigned(tiles_m * tiles_n * groups), C::kThreads, C::kLdsBytes, stream>>>(
      static_cast<const uint16_t*>(x), codes, static_cast<const uint16_t*>(scales),
      static_cast<uint16_t*>(out), m, n, k, groups, xs, xg, tiles_m, tiles_n, vec_n);
  return hipGetLastError();
}

// The kernel of tile kGgufTiles[I], or of a later one.
template <int I = 0>
hipError_t run_gguf_tile(int tile, const void* x, const int8_t* codes, const void* scales,
                         void* out, int m, int n, int k, int groups, int64_t xs, int64_t xg,
                         hipStream_t stream) {
  if constexpr (I >= kGgufTileCount) {
    return hipErrorInvalidValue;
  } else {
    if (tile != I)
      return run_gguf_tile<I + 1>(tile, x, codes, scales, out, m, n, k, groups, xs, xg, stream);
    return run_gguf_ring<GgufRingConfig<kGgufTiles[I].bm, kGgufTiles[I].bn>>(
        x, codes, scales, out, m, n, k, groups, xs, xg, stream);
  }
}

}  // namespace

hipError_t launch_gguf_ring(int tile, const void* x, const int8_t* codes, const void* scales,
                            void* out, int m, int n, int k, int groups, int64_t xs, int64_t xg,
                            hipStream_t stream) {
  return run_gguf_tile(tile, x, codes, scales, out, m, n, k, groups, xs, xg, stream);
}

}  // namespace ci8
