// W8A16 GEMV for long rows and for few channels per CU (channel_gemv, csrc/gemv.cu:8-59):
//
//   out[m, n] = bf16_rn( sum_k float(x[m, k]) * wq[n, k] ),  FP32 sums,
//   wq[n, k]  = bf16_rn( float(w[n, k]) * float(scale[n]) )
//
// the arithmetic of gemv.hip. Its kernels for K > 8192 hold or copy x per workgroup and give
// N = 5120 channels 320 blocks of 16, 1.25 rounds; its span kernel pads every CU's channels to
// blocks of 16 and reads W in 64-byte row pieces. Here a workgroup takes 8 WC channels, WC
// picked so that the tiles fill the CUs once (N = 5120: 214 tiles of 24), and streams W and x
// together in 128-value stages: each of its 8 (or 4) waves owns every 8th (4th) stage and a
// private LDS ring of 3 or 4 of them, filled by buffer_load ... lds in whole 128-byte lines,
// so the K loop has no workgroup barrier (as gemm_small.hip's). x comes from the L2 once per
// tile, 4 XC rows of it. The waves' FP32 sums are added through LDS at the end, in wave order.
//
// What bounds it is the weight stream at large N * K and one launch's latency chain below a
// few microseconds. Measured on MI355X, gemv.hip's kernels in parentheses, us (three rotated
// weight copies): N = 5120, K = 17408: M = 1 18.9 (23.1), 5 19.6 (29.9), 16 24.4 (30.9); N =
// 9121, K = 13168: M = 1 26.7 (32.0), 8 30.3 (43.5); N = 2560, K = 10240: M = 8 8.5 (17.0); N =
// K = 4096: M = 5 6.2 (7.5), 16 6.6 (8.3). More slots per wave (up to 8) ran 0-5% slower
// (fewer workgroups fit a CU), nontemporal weight copies 3-10% slower up to 89 MB of weights
// and 5-12% faster past that (gemv_stream_nontemporal, tile_plan.h). A barrier-synchronized
// ring with 16-row tiles (gguf_ring.hip's kernel with channel scales) was slower nearly
// everywhere (N = 5120, K = 17408: 22.4), since its stages of a few KiB cost 0.2 us each.
#include "ci8_device.h"
#include "launch.h"

namespace ci8 {
namespace {

constexpr int kLdsLimit = 160 * 1024;

// WC: copies of W per stage (8 channels each); XC: copies of x (4 rows each: 1, 2 or 4); kNt:
// W is copied nontemporally.
template <int WC_, int XC_, bool kNt_>
struct StreamConfig {
  static constexpr int WC = WC_, XC = XC_;
  static constexpr int kWPolicy = kNt_ ? kBufferLoadNontemporal : 0;
  static constexpr int BN = 8 * WC, kRows = 4 * XC;
  static constexpr int TN = (WC + 1) / 2;       // 16-channel MFMA blocks (the last may be half)
  static constexpr int BK = 128;                // K values per stage
  static constexpr int kCopies = WC + XC;
  static constexpr int kStageBytes = kCopies * 1024;
  static constexpr int kWaves = 3 * 8 * kStageBytes <= kLdsLimit ? 8 : 4;
  static constexpr int kThreads = 64 * kWaves;
  static constexpr int kFit = kLdsLimit / (kWaves * kStageBytes);
  static constexpr int kSlots = kFit < 4 ? kFit : 4;
  static constexpr int kWaveBytes = kSlots * kStageBytes;
  static constexpr int kLdsBytes = kWaves * kWaveBytes;
  static_assert(kSlots >= 3 && kWaves * TN * 1024 <= kLdsBytes, "LDS");
  static_assert((kSlots - 1) * kCopies < 64, "vmcnt");
};

template <int kPolicy>
__device__ __forceinline__ void copy_w(__amdgpu_buffer_rsrc_t rsrc, lds_void* to, uint32_t offset,
                                       int k0) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, to, 16, offset, k0, 0, kPolicy);
}

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

// Four INT8 codes -> two packed BF16 pairs bf16_rn(code * s) (exact product, one rounding).
__device__ __forceinline__ u32x2 dequant4(uint32_t word, float s) {
  return u32x2{pack_bf16x2(float(int8_t(word)) * s, float(int8_t(word >> 8)) * s),
               pack_bf16x2(float(int8_t(word >> 16)) * s, float(int8_t(word >> 24)) * s)};
}

template <class C>
__global__ void __launch_bounds__(C::kThreads) channel_gemv_stream_kernel(
    const uint16_t* __restrict__ x, const int8_t* __restrict__ w,
    const uint16_t* __restrict__ scale, uint16_t* __restrict__ out, int m, int n, int k) {
  extern __shared__ __attribute__((aligned(1024))) char lds_raw[];
  auto* lds = (char __attribute__((address_space(3)))*)(lds_raw);
  using lds_u32x4 = __attribute__((address_space(3))) u32x4;
  using lds_f32x4 = __attribute__((address_space(3))) f32x4;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n0 = blockIdx.x * C::BN;
  // Stages wave, wave + kWaves, ... of the ns 128-value stages.
  const int ns = (k + C::BK - 1) / C::BK;
  const int count = (ns - wave + C::kWaves - 1) / C::kWaves;

  // W copy q: channels n0 + 8q + lane / 8, x copy q: rows 4q + lane / 16; LDS slots hold the
  // 16-byte chunks of a row XOR-swizzled by the row, so that the fragment reads spread over
  // all banks. Channels past N and rows past M are zeros from the buffer range check.
  uint32_t w_off[C::WC], x_off[C::XC];
  const int w_chunk = (lane & 7) ^ (lane >> 3);
#pragma unroll
  for (int q = 0; q < C::WC; ++q) {
    const int row = n0 + q * 8 + (lane >> 3);
    w_off[q] = row < n ? uint32_t(row) * uint32_t(k) + uint32_t(w_chunk * 16) : kOutOfRange;
  }
#pragma unroll
  for (int q = 0; q < C::XC; ++q) {
    const int row = q * 4 + (lane >> 4);
    x_off[q] = row < m ? (uint32_t(row) * uint32_t(k) + uint32_t(((lane & 15) ^ row) * 8)) * 2
                       : kOutOfRange;
  }
  auto* ring = lds + wave * C::kWaveBytes;
  auto issue = [&] __device__(int it) __attribute__((always_inline)) {
    auto* slot = ring + (it % C::kSlots) * C::kStageBytes;
    const int k0 = (wave + C::kWaves * it) * C::BK;
    const bool whole = k0 + C::BK <= k;  // uniform; only the last stage may not be
#pragma unroll
    for (int q = 0; q < C::XC; ++q) {
      uint32_t off = x_off[q];
      if (!whole && k0 + ((lane & 15) ^ (q * 4 + (lane >> 4))) * 8 >= k) off = kOutOfRange;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          make_rsrc(x, uint32_t(m) * uint32_t(k) * 2), reinterpret_cast<lds_void*>(slot + q * 1024),
          16, off, k0 * 2, 0, 0);
    }
#pragma unroll
    for (int q = 0; q < C::WC; ++q) {
      uint32_t off = w_off[q];
      if (!whole && k0 + w_chunk * 16 >= k) off = kOutOfRange;
      copy_w<C::kWPolicy>(make_rsrc(w, uint32_t(n) * uint32_t(k)),
                          reinterpret_cast<lds_void*>(slot + (C::XC + q) * 1024), off, k0);
    }
  };

  // Fragments of step (p, h): lane group g takes the K values 16 (4p + g) + 8h .. + 7 of the
  // stage, so one 16-byte read of W serves two steps. Lanes of rows that the stage does not
  // hold (past 4 XC rows of x, past a half last block of W) read others in their place; what
  // they add up is never stored.
  const int f_row = lane & 15, f_group = lane >> 4;
  const int x_row = f_row & (C::kRows - 1);
  int x_base[2][2], w_base[2];
#pragma unroll
  for (int p = 0; p < 2; ++p) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
      x_base[p][h] = x_row * 256 + ((2 * (4 * p + f_group) + h) ^ x_row) * 16;
    w_base[p] = ((4 * p + f_group) ^ (f_row & 7)) * 16;
  }
  float s[C::TN];
  int w_row[C::TN];
#pragma unroll
  for (int i = 0; i < C::TN; ++i) {
    const int r = i * 16 + f_row < C::BN ? i * 16 + f_row : i * 16 + (f_row & 7);
    w_row[i] = C::XC * 1024 + r * 128;
    s[i] = n0 + r < n ? bf16_to_f32(scale[n0 + r]) : 0.f;
  }
  f32x4 acc[C::TN];
#pragma unroll
  for (int i = 0; i < C::TN; ++i) acc[i] = f32x4{0, 0, 0, 0};

  // A slot is refilled an iteration after its fragments were read (the MFMAs consumed them).
  for (int it = 0; it < C::kSlots - 1 && it < count; ++it) issue(it);
  for (int it = 0; it < count; ++it) {
    if (it + C::kSlots - 1 < count) issue(it + C::kSlots - 1);
    wait_stages<C::kCopies, C::kSlots - 1>(min(count - 1 - it, C::kSlots - 1));
    asm volatile("" ::: "memory");
    const auto* slot = ring + (it % C::kSlots) * C::kStageBytes;
    u32x4 xf[2][2], wf[C::TN][2];
#pragma unroll
    for (int p = 0; p < 2; ++p) {
#pragma unroll
      for (int i = 0; i < C::TN; ++i)
        wf[i][p] = *reinterpret_cast<const lds_u32x4*>(slot + w_row[i] + w_base[p]);
#pragma unroll
      for (int h = 0; h < 2; ++h)
        xf[p][h] = *reinterpret_cast<const lds_u32x4*>(slot + x_base[p][h]);
    }
    const int k0 = (wave + C::kWaves * it) * C::BK;
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      // Past K the weights are +0 whatever the scale (0 * infinity would be NaN).
      const bool past_k = k0 + 16 * (4 * p + f_group) >= k;
#pragma unroll
      for (int i = 0; i < C::TN; ++i) {
        const float si = past_k ? 0.f : s[i];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const u32x2 lo = dequant4(wf[i][p][2 * h], si), hi = dequant4(wf[i][p][2 * h + 1], si);
          acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              __builtin_bit_cast(bf16x8, u32x4{lo[0], lo[1], hi[0], hi[1]}),
              __builtin_bit_cast(bf16x8, xf[p][h]), acc[i], 0, 0, 0);
        }
      }
    }
  }

  // Every wave is past its last reads and copies: the rings become the partial sums.
  __builtin_amdgcn_s_waitcnt(lgkmcnt0_imm());
  __syncthreads();
  auto* part = reinterpret_cast<lds_f32x4*>(lds);
#pragma unroll
  for (int i = 0; i < C::TN; ++i) part[(wave * C::TN + i) * 64 + lane] = acc[i];
  __syncthreads();
  for (int i = wave; i < C::TN; i += C::kWaves) {
    f32x4 sum = part[i * 64 + lane];
#pragma unroll
    for (int v = 1; v < C::kWaves; ++v) sum += part[(v * C::TN + i) * 64 + lane];
    const int local = i * 16 + 4 * f_group, col = n0 + local;
    if (f_row >= m || local >= C::BN) continue;
    uint16_t* dst = out + int64_t(f_row) * n + col;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (col + e < n) dst[e] = uint16_t(f32_to_bf16(sum[e]));
  }
}

template <class C>
hipError_t run_stream(const void* x, const int8_t* w, const void* scale, void* out, int m, int n,
                      int k, hipStream_t stream) {
  auto kernel = channel_gemv_stream_kernel<C>;
  if (const hipError_t e = prepare_lds<channel_gemv_stream_kernel<C>>(C::kLdsBytes);
      e != hipSuccess)
    return e;
  kernel<<<(n + C::BN - 1) / C::BN, C::kThreads, C::kLdsBytes, stream>>>(
      static_cast<const uint16_t*>(x), w, static_cast<const uint16_t*>(scale),
      static_cast<uint16_t*>(out), m, n, k);
  return hipGetLastError();
}

// The kernel of 8 WC channels per tile, or of more.
template <bool kNt, int WC = 1>
hipError_t run_stream_width(int wc, const void* x, const int8_t* w, const void* scale, void* out,
                            int m, int n, int k, hipStream_t stream) {
  if constexpr (WC > kStreamMaxCopies) {
    return hipErrorInvalidValue;
  } else {
    if (wc != WC) return run_stream_width<kNt, WC + 1>(wc, x, w, scale, out, m, n, k, stream);
    if (m <= 4) return run_stream<StreamConfig<WC, 1, kNt>>(x, w, scale, out, m, n, k, stream);
    if (m <= 8) return run_stream<StreamConfig<WC, 2, kNt>>(x, w, scale, out, m, n, k, stream);
    return run_stream<StreamConfig<WC, 4, kNt>>(x, w, scale, out, m, n, k, stream);
  }
}

}  // namespace

hipError_t launch_stream_gemv(int copies, const void* x, const int8_t* w, const void* scale,
                              void* out, int m, int n, int k, hipStream_t stream) {
  if (gemv_stream_nontemporal(n, k))
    return run_stream_width<true>(copies, x, w, scale, out, m, n, k, stream);
  return run_stream_width<false>(copies, x, w, scale, out, m, n, k, stream);
}

}  // namespace ci8
