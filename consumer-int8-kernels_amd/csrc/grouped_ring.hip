// Grouped, summed W8A8 (grouped_summed_mm) for the shapes that gemm_grouped.hip's 256 x 128
// tiles leave short: fewer than 1024 rows, M % 4 != 0, or too few tiles for the CUs. The
// same closed form, bit for bit:
//
//   out[m, n] = bf16_rn( t_0 + t_1 + ... + t_{G-1} )   (FP32 additions, ascending g),
//   t_g = fl( fl( float_rn(acc_g[m, n]) * sa[g, m] ) * float(sw[n]) ),
//   acc_g = A_g[m, :] . W_g[n, :]   (exact INT32), A [G, M, K], W [G, N, K], sa [G, M].
//
// The structure is gemm_ring.hip's (one tile per CU picked per shape, an LDS ring filled by
// buffer_load ... lds, register-double-buffered fragments, one barrier per stage) with the K
// stages of all groups in one stream: stage s is K stage s % ns of group s / ns, so copies
// run across group boundaries. The eight waves split the tile in m and n only, so that a
// group's INT32 sums are whole in their wave's registers and are folded into the FP32 sum
// beside them after the group's last stage (as two K groups ran gemm_ring.hip's 64 x 128 tile
// no faster, the copies bound it either way). The tile's row scales of every group are put
// into LDS once: a vector load inside the loop would make the compiler wait there for every
// copy in flight.
//
// What bounds it is gemm_ring.hip's: the operand copies, at 55-80 B/ns per CU. Measured on
// MI355X, the kernels that took these shapes before in parentheses, us (K = 4096 per group,
// three rotated weight copies, identical outputs): G = 4, N = 4096: M = 17 25.7 (92.7), 128
// 28.6 (104.6), 512 48.8 (105.5), 1135 93.1 (148.4); G = 1, N = 4616: M = 173 11.9 (30.9);
// G = 3, N = 2456: M = 1024 48.2 (71.8). Over 105 shapes the time fell by half in the mean;
// where 256 x 128 tiles fill the CUs (M = 2048, N = 4096: 137 against 165 us) they stay.
#include <type_traits>

#include "ci8_device.h"
#include "launch.h"

namespace ci8 {
namespace {

constexpr int kXcds = 8;
constexpr int kLdsLimit = 160 * 1024;

template <int BM_, int BN_>
struct GroupedRingConfig {
  static constexpr int BM = BM_, BN = BN_;
  static constexpr int WM = BN % 64 == 0 ? 2 : 4, WN = 8 / WM;
  static constexpr int kWaves = 8, kThreads = 64 * kWaves;
  static constexpr int TM = BM / WM / 16, TN = BN / WN / 16;
  static constexpr int BK = 3 * (BM + BN) * 256 <= kLdsLimit - kGroupedScaleBytes ? 256 : 128;
  static constexpr int kChunks = BK / 16, kCopyRows = 1024 / BK, kSteps = BK / 64;
  static constexpr int kACopies = BM / kCopyRows;
  static constexpr int kStageCopies = (BM + BN) / kCopyRows;
  static constexpr int kCopies = (kStageCopies + kWaves - 1) / kWaves;      // per wave, at most
  static constexpr int kLastWaves = kStageCopies - (kCopies - 1) * kWaves;  // with that many
  static constexpr int kStageBytes = kStageCopies * 1024;
  static constexpr int kFit = (kLdsLimit - kGroupedScaleBytes) / kStageBytes;
  static constexpr int kSlots = kFit < 4 ? kFit : 4;
  static constexpr int kRingBytes = kSlots * kStageBytes;
  static_assert(BM % (WM * 16) == 0 && BN % (WN * 16) == 0, "16-row MFMA blocks");
  static_assert(kSlots >= 3, "LDS");
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

template <class C>
__global__ void __launch_bounds__(C::kThreads, 1) grouped_ring_kernel(
    const int8_t* __restrict__ a, const int8_t* __restrict__ w, const float* __restrict__ sa,
    const uint16_t* __restrict__ sw, uint16_t* __restrict__ out, int groups, int m, int n, int k,
    bool vec_n) {
  // Every product and sum below is rounded on its own, as the closed form requires.
#pragma clang fp contract(off)
  extern __shared__ __attribute__((aligned(1024))) char lds_raw[];
  auto* lds = (char __attribute__((address_space(3)))*)(lds_raw);
  using lds_i32x4 = __attribute__((address_space(3))) i32x4;
  using lds_float = __attribute__((address_space(3))) float;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave % C::WM, wn = wave / C::WM;

  // Workgroup -> tile: each XCD runs a contiguous range of tiles, m fastest.
  const int tiles_m = (m + C::BM - 1) / C::BM;
  const int tiles_n = (n + C::BN - 1) / C::BN;
  const int tiles = tiles_m * tiles_n;
  int logical = blockIdx.x;
  {
    const int per = tiles / kXcds, extra = tiles % kXcds;
    const int xcd = logical % kXcds, idx = logical / kXcds;
    logical = (xcd < extra ? xcd * (per + 1) : extra * (per + 1) + (xcd - extra) * per) + idx;
  }
  const int m0 = logical % tiles_m * C::BM, n0 = logical / tiles_m * C::BN;
  const int ns = (k + C::BK - 1) / C::BK;  // stages of a group
  const int total = ns * groups;

  // Copies, as in gemm_ring.hip; the next stage to copy is K stage copy_t of group copy_g.
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
  int copy_t = 0;
  const int8_t* copy_a = a;
  const int8_t* copy_w = w;
  auto copy = [&] __device__(int slot, int i) __attribute__((always_inline)) {
    const int b = i * C::kWaves + wave;
    const bool is_a = b < C::kACopies;  // uniform over the wave
    const int k0 = copy_t * C::BK;
    uint32_t off = c_off[i];
    if (!exact_k && k0 + chunk_of(b) * 16 >= k) off = kOutOfRange;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        make_rsrc(is_a ? copy_a : copy_w, uint32_t(is_a ? m : n) * uint32_t(k)),
        reinterpret_cast<lds_void*>(lds + slot * C::kStageBytes + b * 1024), 16, off, k0, 0, 0);
  };
  auto copied = [&] __device__() __attribute__((always_inline)) {  // one stage on
    if (++copy_t == ns) {
      copy_t = 0;
      copy_a += int64_t(m) * k;
      copy_w += int64_t(n) * k;
    }
  };
  auto copy_stage = [&] __device__(int slot) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < C::kCopies; ++i)
      if (i + 1 < C::kCopies || all_copies) copy(slot, i);
    copied();
  };

  const int f_row = lane & 15, f_group = lane >> 4;
  int a_base[C::kSteps], w_base[C::kSteps];
#pragma unroll
  for (int h = 0; h < C::kSteps; ++h) {
    const int swz = ((4 * h + f_group) ^ (f_row & (C::kChunks - 1))) * 16;
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

  for (int t = 0; t < C::kSlots && t < total; ++t) copy_stage(t);
  // Row scales of every group -> LDS; channels n0 + 16 (wn TN + i) + 4 (lane / 16) + 0..3 in
  // registers. Their loads are waited for here, behind the first copies.
  auto* row_scales = reinterpret_cast<lds_float*>(lds + C::kRingBytes);
  for (int q = threadIdx.x; q < groups * C::BM; q += C::kThreads) {
    const int row = m0 + q % C::BM;
    row_scales[q] = row < m ? sa[int64_t(q / C::BM) * m + row] : 0.f;
  }
  float cs[C::TN][4];
#pragma unroll
  for (int i = 0; i < C::TN; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int col = n0 + (wn * C::TN + i) * 16 + f_group * 4 + e;
      cs[i][e] = col < n ? bf16_to_f32(sw[col]) : 0.f;
    }
  __builtin_amdgcn_s_waitcnt(vm_lgkm_imm(0, 0));
  barrier();
  read(0, 0);

  i32x4 acc[C::TM][C::TN];
  f32x4 sum[C::TM][C::TN];
#pragma unroll
  for (int j = 0; j < C::TM; ++j)
#pragma unroll
    for (int i = 0; i < C::TN; ++i) acc[j][i] = i32x4{0, 0, 0, 0};

  int slot = 0;          // t % kSlots
  int left = ns, g = 0;  // stages left in the group of stage t, that group
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
    wait(kSteady ? C::kSlots - 2 : max(0, min(C::kSlots - 2, total - 2 - t)));
    barrier();
    if (kSteady || t + 1 < total) read(buf ^ 1, next);
    if (!kSteady && t + C::kSlots < total) copy_stage(slot);
    constexpr int kMfmas = C::kSteps * C::TN * C::TM;
    constexpr int kEvery = kMfmas / C::kCopies > 0 ? kMfmas / C::kCopies : 1;
#pragma unroll
    for (int q = 0; q < (kMfmas > C::kCopies ? kMfmas : C::kCopies); ++q) {
      if (kSteady && q % kEvery == 0 && q / kEvery < C::kCopies) {
        const int i = q / kEvery;
        __builtin_amdgcn_sched_barrier(0);
        if (i + 1 < C::kCopies || all_copies) copy(slot, i);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (q < kMfmas) {
        const int h = q / (C::TN * C::TM), i = q / C::TM % C::TN, j = q % C::TM;
        acc[j][i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wf[buf][h][i], af[buf][h][j],
                                                          acc[j][i], 0, 0, 0);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    if (kSteady) copied();
    slot = next;
    if (--left == 0) {  // the group is complete: fold its terms into the sum
      float rs[C::TM];
#pragma unroll
      for (int j = 0; j < C::TM; ++j)
        rs[j] = row_scales[g * C::BM + (wm * C::TM + j) * 16 + f_row];
#pragma unroll
      for (int j = 0; j < C::TM; ++j)
#pragma unroll
        for (int i = 0; i < C::TN; ++i) {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float term = (float(acc[j][i][e]) * rs[j]) * cs[i][e];
            sum[j][i][e] = g == 0 ? term : sum[j][i][e] + term;
          }
          acc[j][i] = i32x4{0, 0, 0, 0};
        }
      left = ns;
      ++g;
    }
  };
  using Even = std::integral_constant<int, 0>;
  using Odd = std::integral_constant<int, 1>;
  int t = 0;
  for (; t + 1 + C::kSlots < total; t += 2) {
    iteration(t, Even{}, std::true_type{});
    iteration(t + 1, Odd{}, std::true_type{});
  }
  for (; t + 1 < total; t += 2) {
    iteration(t, Even{}, std::false_type{});
    iteration(t + 1, Odd{}, std::false_type{});
  }
  if (t < total) iteration(t, Even{}, std::false_type{});

#pragma unroll
  for (int i = 0; i < C::TN; ++i) {
    const int col = n0 + (wn * C::TN + i) * 16 + f_group * 4;
#pragma unroll
    for (int j = 0; j < C::TM; ++j) {
      const int row = m0 + (wm * C::TM + j) * 16 + f_row;
      if (row >= m || col >= n) continue;
      const int64_t base = int64_t(row) * n + col;
      const f32x4& v = sum[j][i];
      if (vec_n) {
        *reinterpret_cast<u32x2*>(out + base) =
            u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (col + e < n) out[base + e] = uint16_t(f32_to_bf16(v[e]));
      }
    }
  }
}

template <class C>
hipError_t run_grouped_ring(const int8_t* a, const int8_t* w, const float* sa, const void* sw,
                            void* out, int groups, int m, int n, int k, hipStream_t stream) {
  auto kernel = grouped_ring_kernel<C>;
  const int lds = C::kRingBytes + groups * C::BM * 4;
  if (const hipError_t e = prepare_lds<grouped_ring_kernel<C>>(lds); e != hipSuccess) return e;
  const int blocks = ((m + C::BM - 1) / C::BM) * ((n + C::BN - 1) / C::BN);
  const bool vec_n = n % 4 == 0 && reinterpret_cast<uintptr_t>(out) % 8 == 0;
  kernel<<<blocks, C::kThreads, lds, stream>>>(a, w, sa, static_cast<const uint16_t*>(sw),
                                               static_cast<uint16_t*>(out), groups, m, n, k,
                                               vec_n);
  return hipGetLastError();
}

// The kernel of tile kGroupedTiles[I], or of a later one.
template <int I = 0>
hipError_t run_grouped_tile(int tile, const int8_t* a, const int8_t* w, const float* sa,
                            const void* sw, void* out, int groups, int m, int n, int k,
                            hipStream_t stream) {
  if constexpr (I >= kGroupedTileCount) {
    return hipErrorInvalidValue;
  } else {
    if (tile != I)
      return run_grouped_tile<I + 1>(tile, a, w, sa, sw, out, groups, m, n, k, stream);
    return run_grouped_ring<GroupedRingConfig<kGroupedTiles[I].bm, kGroupedTiles[I].bn>>(
        a, w, sa, sw, out, groups, m, n, k, stream);
  }
}

}  // namespace

hipError_t launch_grouped_ring_gemm(int tile, const int8_t* a, const int8_t* w, const float* sa,
                                    const void* sw, void* out, int groups, int m, int n, int k,
                                    hipStream_t stream) {
  return run_grouped_tile(tile, a, w, sa, sw, out, groups, m, n, k, stream);
}

}  // namespace ci8
