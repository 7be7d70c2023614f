// Mid-size INT8 GEMM for gfx950: the product and epilogue of gemm.hip, bit for bit,
//
//   out[m, n] = bf16_rn( fl( fl( float_rn(acc[m, n]) * sa[m] ) * float(sw[n]) ) )
//   acc[m, n] = sum_k a[m, k] * w[n, k]            (exact INT32)
//
// for shapes between a decode batch and a large prefill, where 256 x 224 or 128 x 128
// tiles leave many of the 256 CUs idle. What bounds such a shape is the rate at which a CU
// copies operands from the L2 into LDS, (BM + BN) * K bytes per tile: about 80 B/ns while
// the weights sit in the Infinity Cache and 55-60 B/ns when they come from HBM, whatever
// the ring's depth (3 to 8 slots), the number of busy CUs (64 to 256), the cache policy of
// the copies or an L2 prefetch of the panels by a ninth wave (all measured within 3%; the
// nontemporal policy 10-50% slower). So the tile is picked per shape (tile_plan.h) to put
// one tile on every CU with as few operand bytes as possible. (Splitting K over workgroups would
// copy fewer, but the entry points have no buffer for the partial sums and no counter.)
//
// Measured on MI355X against the kernels that took these shapes before (fused_channel_mm
// alone, three rotated weight copies, identical outputs), us: M = 256, N = 7168, K = 5120:
// 18.2 (29.9); M = 333, N = 5120, K = 8704: 25.4 (55.5); M = 1024, N = 5120, K = 17408: 94
// (145); M = 128, N = 17408, K = 5120: 23.7 (43.3); M = 512, N = 2048, K = 8192: 17.3
// (51.3). Over 162 shapes from M = 17 to 3000 the time fell by a quarter in the mean.
//
// One workgroup of eight waves per tile:
//   - K advances in stages of 128 or 256 bytes through an LDS ring filled by buffer_load
//     ... lds (1 KiB per copy: 8 rows x 128 or 4 rows x 256 bytes; 256-byte row pieces ran
//     3-6% faster where three such stages fit). Rows past M or N and bytes past K are
//     zeros from the buffer range check.
//   - The waves form two K groups: group g takes the g-th half of every stage, so a wave's
//     output tile is twice as large as with eight waves side by side and its fragments
//     are read from LDS half as often (128 x 160: 72 KB of LDS reads a stage for 36 KB
//     copied). The groups' INT32 partials are added through the ring at the end.
//   - Fragments are double-buffered in registers: a stage's MFMAs run while the next
//     stage's fragments are read, with this wave's copies spread between the MFMAs (a copy
//     stalls its wave while the address unit's queue is full). One barrier per stage: past
//     it every wave's copies of stage t + 1 have landed and the slot of stage t is free.
#include <type_traits>

#include "ci8_device.h"
#include "launch.h"

namespace ci8 {
namespace {

constexpr int kXcds = 8;
constexpr int kKGroups = 2;
constexpr int kLdsLimit = 160 * 1024;

template <int BM_, int BN_>
struct RingConfig {
  static constexpr int BM = BM_, BN = BN_;
  static constexpr int WM = BN % 32 == 0 ? 2 : 4, WN = 4 / WM;  // waves of one K group
  static constexpr int kWaves = WM * WN * kKGroups, kThreads = 64 * kWaves;
  static constexpr int TM = BM / WM / 16, TN = BN / WN / 16;
  static constexpr int BK = 3 * (BM + BN) * 256 <= kLdsLimit ? 256 : 128;  // stage, bytes of K
  static constexpr int kChunks = BK / 16;            // 16-byte chunks of a stage's row
  static constexpr int kCopyRows = 1024 / BK;        // rows per copy
  static constexpr int kSteps = BK / 64 / kKGroups;  // MFMA K steps of a wave per stage
  static constexpr int kACopies = BM / kCopyRows;
  static constexpr int kStageCopies = (BM + BN) / kCopyRows;
  static constexpr int kCopies = (kStageCopies + kWaves - 1) / kWaves;  // per wave, at most
  static constexpr int kLastWaves = kStageCopies - (kCopies - 1) * kWaves;  // with that many
  static constexpr int kStageBytes = kStageCopies * 1024;
  static constexpr int kSlots = kLdsLimit / kStageBytes < 4 ? kLdsLimit / kStageBytes : 4;
  static constexpr int kMine = (TN + 1) / 2;  // n blocks a K group finishes, at most
  static constexpr int kPartialBytes = kWaves * kMine * TM * 1024;
  static constexpr int kRingBytes = kSlots * kStageBytes;
  static constexpr int kLdsBytes = kRingBytes > kPartialBytes ? kRingBytes : kPartialBytes;
  static_assert(BM % (WM * 16) == 0 && BN % (WN * 16) == 0, "16-row MFMA blocks");
  static_assert(kSlots >= 3 && kLdsBytes <= kLdsLimit, "LDS");
  static_assert((kSlots - 1) * kCopies < 64, "vmcnt");
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

template <class C, WeightCode kCode, bool kWorkspace>
__global__ void __launch_bounds__(C::kThreads, 1) ring_gemm_kernel(
    const int8_t* __restrict__ a, const int8_t* __restrict__ w, const float* __restrict__ sa,
    const uint16_t* __restrict__ sw, uint16_t* __restrict__ out, int32_t* __restrict__ ws,
    int m, int n, int k, bool vec_n) {
  extern __shared__ __attribute__((aligned(1024))) char lds_raw[];
  auto* lds = (char __attribute__((address_space(3)))*)(lds_raw);
  using lds_i32x4 = __attribute__((address_space(3))) i32x4;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int group = wave / (C::WM * C::WN), member = wave % (C::WM * C::WN);
  const int wm = member % C::WM, wn = member / C::WM;

  // Workgroup -> tile. The hardware deals workgroups round-robin over the 8 XCDs; undo
  // that so each XCD runs a contiguous range of tiles, m fastest, and the tiles that share
  // a weight panel fetch it into one XCD's L2.
  const int tiles_m = (m + C::BM - 1) / C::BM;
  const int tiles_n = (n + C::BN - 1) / C::BN;
  const int tiles = tiles_m * tiles_n;
  int logical = blockIdx.x;
  {
    const int per = tiles / kXcds, extra = tiles % kXcds;
    const int xcd = logical % kXcds, idx = logical / kXcds;
    logical = (xcd < extra ? xcd * (per + 1) : extra * (per + 1) + (xcd - extra) * per) + idx;
  }
  const int tile_m = logical % tiles_m, tile_n = logical / tiles_m;
  const int m0 = tile_m * C::BM, n0 = tile_n * C::BN;
  // K order: stages t0, t0 + 1, ..., wrapping round, with a start per tile, so the tiles
  // that share a panel do not all miss on the same lines (INT32 sums are exact in any
  // order; against one start for all 0-5% faster, as gemm_pp_kernel.h describes).
  const int ns = (k + C::BK - 1) / C::BK;
  const int t0 = (tile_m + tile_n) % 8 % ns;
  auto stage_k0 = [&] __device__(int t) __attribute__((always_inline)) {
    return (t + t0 < ns ? t + t0 : t + t0 - ns) * C::BK;
  };

  // Copy b = i * kWaves + wave of a stage (i < kCopies) brings rows b * kCopyRows + lane /
  // kChunks of the stage (A's rows, then W's) into LDS in order; slot lane % kChunks of a
  // row holds logical chunk slot ^ (row % 8 or 16), so that the fragment reads below (16
  // rows at one logical chunk) spread over all banks.
  const int c_row = lane / C::kChunks;
  auto chunk_of = [&] __device__(int b) __attribute__((always_inline)) {
    return (lane % C::kChunks) ^ ((b * C::kCopyRows + c_row) & (C::kChunks - 1));
  };
  uint32_t c_off[C::kCopies];
#pragma unroll
  for (int i = 0; i < C::kCopies; ++i) {
    const int b = i * C::kWaves + wave;
    const bool is_a = b < C::kACopies;
    const int row = is_a ? m0 + b * C::kCopyRows + c_row
                         : n0 + (b - C::kACopies) * C::kCopyRows + c_row;
    c_off[i] = row < (is_a ? m : n) ? uint32_t(row) * uint32_t(k) + uint32_t(chunk_of(b) * 16)
                                    : kOutOfRange;
  }
  const bool all_copies = C::kLastWaves == C::kWaves || wave < C::kLastWaves;  // per wave
  const bool exact_k = k % C::BK == 0;
  auto copy = [&] __device__(int slot, int k0, int i) __attribute__((always_inline)) {
    const int b = i * C::kWaves + wave;
    const bool is_a = b < C::kACopies;  // uniform over the wave
    uint32_t off = c_off[i];
    // A 16-byte chunk lies wholly inside or wholly past K (k % 32 == 0).
    if (!exact_k && k0 + chunk_of(b) * 16 >= k) off = kOutOfRange;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        make_rsrc(is_a ? a : w, uint32_t(is_a ? m : n) * uint32_t(k)),
        reinterpret_cast<lds_void*>(lds + slot * C::kStageBytes + b * 1024), 16, off, k0, 0, 0);
  };
  auto copy_stage = [&] __device__(int slot, int t) __attribute__((always_inline)) {
    const int k0 = stage_k0(t);
#pragma unroll
    for (int i = 0; i < C::kCopies; ++i)
      if (i + 1 < C::kCopies || all_copies) copy(slot, k0, i);
  };

  // Fragments: row lane % 16 of a 16-row block at logical chunk 4 step + lane / 16 of the
  // stage, steps group * kSteps + h (A and W alike, so the sums are those of any K order).
  const int f_row = lane & 15, f_group = lane >> 4;
  int a_base[C::kSteps], w_base[C::kSteps];
#pragma unroll
  for (int h = 0; h < C::kSteps; ++h) {
    const int chunk = 4 * (group * C::kSteps + h) + f_group;
    const int swz = (chunk ^ (f_row & (C::kChunks - 1))) * 16;
    a_base[h] = (wm * C::TM * 16 + f_row) * C::BK + swz;
    w_base[h] = (C::BM + wn * C::TN * 16 + f_row) * C::BK + swz;
  }
  i32x4 af[2][C::kSteps][C::TM], wf[2][C::kSteps][C::TN];
  auto read = [&] __device__(int buf, int slot) __attribute__((always_inline)) {
    const auto* s = lds + slot * C::kStageBytes;
#pragma unroll
    for (int h = 0; h < C::kSteps; ++h) {
#pragma unroll
      for (int j = 0; j < C::TM; ++j)
        af[buf][h][j] = *reinterpret_cast<const lds_i32x4*>(s + a_base[h] + j * 16 * C::BK);
#pragma unroll
      for (int i = 0; i < C::TN; ++i)
        wf[buf][h][i] = *reinterpret_cast<const lds_i32x4*>(s + w_base[h] + i * 16 * C::BK);
    }
  };

  // The wave's copies of all but the latest `after` stages have landed.
  auto wait = [&] __device__(int after) __attribute__((always_inline)) {
    if (all_copies)
      wait_stages<C::kCopies, C::kSlots - 1>(after);
    else
      wait_stages<C::kCopies - 1, C::kSlots - 1>(after);
  };
  auto barrier = [&] __device__() __attribute__((always_inline)) {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };

  // The epilogue's scales, loaded ahead of the K loop (in the epilogue their latency cost
  // 1-2 us). The counted waits hold wherever the compiler issues these loads: one that is
  // younger than a copy only makes a wait longer. K group g finishes the n blocks 2q + g.
  float rs[C::TM];
  u32x2 cs[C::kMine];
#pragma unroll
  for (int j = 0; j < C::TM; ++j) {
    const int row = m0 + (wm * C::TM + j) * 16 + f_row;
    rs[j] = row < m ? sa[row] : 0.f;
  }
#pragma unroll
  for (int q = 0; q < C::kMine; ++q) {
    const int i = 2 * q + group;
    const int col = n0 + (wn * C::TN + i) * 16 + f_group * 4;
    if (vec_n) {
      cs[q] = i < C::TN && col < n ? *reinterpret_cast<const u32x2*>(sw + col) : u32x2{0, 0};
    } else {
      uint32_t s[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) s[e] = i < C::TN && col + e < n ? sw[col + e] : 0;
      cs[q] = u32x2{s[0] | s[1] << 16, s[2] | s[3] << 16};
    }
  }

  i32x4 acc[C::TM][C::TN];
#pragma unroll
  for (int j = 0; j < C::TM; ++j)
#pragma unroll
    for (int i = 0; i < C::TN; ++i) acc[j][i] = i32x4{0, 0, 0, 0};

  for (int t = 0; t < C::kSlots && t < ns; ++t) copy_stage(t, t);
  wait(min(ns, C::kSlots) - 1);
  barrier();
  read(0, 0);

  int slot = 0;  // t % kSlots
  // Stage t, its fragments in register buffer `parity`. kSteady: stages t + 1 and t +
  // kSlots exist.
  auto iteration = [&] __device__(int t, auto parity, auto steady) __attribute__((always_inline)) {
    constexpr int buf = decltype(parity)::value;
    constexpr bool kSteady = decltype(steady)::value;
    const int next = slot + 1 == C::kSlots ? 0 : slot + 1;
    // This wave has read stage t, and its copies of stage t + 1 have landed; past the
    // barrier, every wave's, so stage t + 1 can be read and the slot of stage t refilled.
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(lgkmcnt0_imm());
    wait(kSteady ? C::kSlots - 2 : max(0, min(C::kSlots - 2, ns - 2 - t)));
    barrier();
    if (kSteady || t + 1 < ns) read(buf ^ 1, next);
    if (!kSteady && t + C::kSlots < ns) copy_stage(slot, t + C::kSlots);
    const int k0 = stage_k0(t + C::kSlots);
    if constexpr (kCode == WeightCode::kBiasedU8) {
      // Biased UINT8 codes (code + 128) -> signed INT8 codes: flip each byte's top bit.
#pragma unroll
      for (int h = 0; h < C::kSteps; ++h)
#pragma unroll
        for (int i = 0; i < C::TN; ++i) wf[buf][h][i] ^= int(0x80808080u);
    }
    constexpr int kMfmas = C::kSteps * C::TN * C::TM;
    constexpr int kEvery = kMfmas / C::kCopies > 0 ? kMfmas / C::kCopies : 1;
#pragma unroll
    for (int q = 0; q < (kMfmas > C::kCopies ? kMfmas : C::kCopies); ++q) {
      if (kSteady && q % kEvery == 0 && q / kEvery < C::kCopies) {
        const int i = q / kEvery;
        __builtin_amdgcn_sched_barrier(0);
        if (i + 1 < C::kCopies || all_copies) copy(slot, k0, i);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (q < kMfmas) {
        const int h = q / (C::TN * C::TM), i = q / C::TM % C::TN, j = q % C::TM;
        acc[j][i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wf[buf][h][i], af[buf][h][j],
                                                          acc[j][i], 0, 0, 0);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    slot = next;
  };
  using Even = std::integral_constant<int, 0>;
  using Odd = std::integral_constant<int, 1>;
  int t = 0;
  for (; t + 1 + C::kSlots < ns; t += 2) {
    iteration(t, Even{}, std::true_type{});
    iteration(t + 1, Odd{}, std::true_type{});
  }
  for (; t + 1 < ns; t += 2) {
    iteration(t, Even{}, std::false_type{});
    iteration(t + 1, Odd{}, std::false_type{});
  }
  if (t < ns) iteration(t, Even{}, std::false_type{});

  // The K groups exchange partial sums through the ring (every copy has landed and every
  // fragment has been read): each hands over the n blocks that the other finishes.
  __syncthreads();
  auto* part = reinterpret_cast<lds_i32x4*>(lds);
#pragma unroll
  for (int i = 0; i < C::TN; ++i)
    if (i % 2 != group) {
#pragma unroll
      for (int j = 0; j < C::TM; ++j)
        part[((wave * C::kMine + i / 2) * C::TM + j) * 64 + lane] = acc[j][i];
    }
  __syncthreads();
  const int other = wave ^ (C::WM * C::WN);
#pragma unroll
  for (int i = 0; i < C::TN; ++i) {
    if (i % 2 != group) continue;  // uniform over the wave
    const int col = n0 + (wn * C::TN + i) * 16 + f_group * 4;
#pragma unroll
    for (int j = 0; j < C::TM; ++j) {
      const i32x4 sum = acc[j][i] + part[((other * C::kMine + i / 2) * C::TM + j) * 64 + lane];
      const int row = m0 + (wm * C::TM + j) * 16 + f_row;
      if (row >= m || col >= n) continue;
      const int64_t base = int64_t(row) * n + col;
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t bits = (cs[i / 2][e >> 1] >> (16 * (e & 1))) & 0xFFFFu;
        v[e] = (float(sum[e]) * rs[j]) * bf16_to_f32(bits);
      }
      if (vec_n) {
        *reinterpret_cast<u32x2*>(out + base) =
            u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
        if constexpr (kWorkspace) *reinterpret_cast<i32x4*>(ws + base) = sum;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (col + e < n) {
            out[base + e] = uint16_t(f32_to_bf16(v[e]));
            if constexpr (kWorkspace) ws[base + e] = sum[e];
          }
      }
    }
  }
}

template <class C, WeightCode kCode, bool kWorkspace>
hipError_t run_ring(const int8_t* a, const void* w, const float* sa, const void* sw, void* out,
                    int32_t* ws, int m, int n, int k, hipStream_t stream) {
  auto kernel = ring_gemm_kernel<C, kCode, kWorkspace>;
  if (const hipError_t e = prepare_lds<ring_gemm_kernel<C, kCode, kWorkspace>>(C::kLdsBytes);
      e != hipSuccess)
    return e;
  const int blocks = ((m + C::BM - 1) / C::BM) * ((n + C::BN - 1) / C::BN);
  const bool vec_n = n % 4 == 0 && reinterpret_cast<uintptr_t>(sw) % 8 == 0 &&
                     reinterpret_cast<uintptr_t>(out) % 8 == 0 &&
                     reinterpret_cast<uintptr_t>(ws) % 16 == 0;
  kernel<<<blocks, C::kThreads, C::kLdsBytes, stream>>>(
      a, static_cast<const int8_t*>(w), sa, static_cast<const uint16_t*>(sw),
      static_cast<uint16_t*>(out), ws, m, n, k, vec_n);
  return hipGetLastError();
}

// The kernel of tile kRingTiles[I], or of a later one.
template <WeightCode kCode, bool kWorkspace, int I = 0>
hipError_t run_ring_tile(int tile, const int8_t* a, const void* w, const float* sa,
                         const void* sw, void* out, int32_t* ws, int m, int n, int k,
                         hipStream_t stream) {
  if constexpr (I >= kRingTileCount) {
    return hipErrorInvalidValue;
  } else {
    if (tile != I)
      return run_ring_tile<kCode, kWorkspace, I + 1>(tile, a, w, sa, sw, out, ws, m, n, k, stream);
    using C = RingConfig<kRingTiles[I].bm, kRingTiles[I].bn>;
    return run_ring<C, kCode, kWorkspace>(a, w, sa, sw, out, ws, m, n, k, stream);
  }
}

}  // namespace

hipError_t launch_ring_gemm(int tile, const int8_t* a, const void* w, WeightCode code,
                            const float* sa, const void* sw, void* out, int32_t* ws, int m,
                            int n, int k, hipStream_t stream) {
  if (code == WeightCode::kBiasedU8)
    return run_ring_tile<WeightCode::kBiasedU8, false>(tile, a, w, sa, sw, out, nullptr, m, n, k,
                                                       stream);
  if (ws)
    return run_ring_tile<WeightCode::kSigned, true>(tile, a, w, sa, sw, out, ws, m, n, k, stream);
  return run_ring_tile<WeightCode::kSigned, false>(tile, a, w, sa, sw, out, nullptr, m, n, k,
                                                   stream);
}

}  // namespace ci8
