// Row quantizers for gfx950: BF16 [rows, k] -> INT8 codes + FP32 per-row scales.
//
// Numerics follow csrc/kernels.cu:13-35 and :41-86 of the reference exactly:
//   amax  = NaN-ignoring max |x| over the row, starting from 0
//   scale = max(fl(amax / 127), 1e-20f)                       (IEEE division)
//   code  = clamp(rne(fl(x / scale)), -127, 127)              (IEEE division, RNE)
// fl(x/scale) never exceeds 127 in magnitude for finite x, so the clamp only matters
// for non-finite input; rounding uses the 1.5*2^23 add, whose low byte is the
// two's-complement code and which maps NaN to 0 like the reference's
// float->int conversion. The vector path takes the quotient from the row reciprocal and
// divides only near half-integers (codes8 in ci8_device.h), with the same codes.
//
// Layout: one, two or four waves own a row (four past 1024 values, so a lane holds
// at most a few 16-byte packs; eight when few and wide rows leave CUs or loads idle) and keep
// it in registers between the max reduction and the
// store, so HBM sees a single read of x and a single write of the codes, with 16-byte
// loads and 8-byte stores (cache policy: stream_policy.h) fully coalesced across
// the wave.
#include "ci8_device.h"
#include "launch.h"

namespace ci8 {
namespace {

constexpr int kWave = 64;

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int offset = 32; offset >= 1; offset >>= 1) v = fmaxf(v, __shfl_xor(v, offset, kWave));
  return v;
}

// Vector path. Requires k % 8 == 0, x 16-byte aligned, codes 8-byte aligned.
// kWaves waves cooperate on one row when kWaves > 1 (very wide rows).
// Grouped: output row o reads input row (o % m) * groups + o / m ([m,g,k] -> [g,m,k]).
// Workgroups hold four waves (1, 2 or 4 rows), or kWaves waves and one row for kWaves > 4.
template <int kPacks, int kWaves, bool kGrouped, StreamPolicy kPolicy>
__global__ void __launch_bounds__(kWaves > 4 ? 64 * kWaves : 256) quantize_rows_vec_kernel(
    const uint16_t* __restrict__ x, int8_t* __restrict__ codes, float* __restrict__ scales,
    int rows, int k, int m, int groups) {
  constexpr int kRowsPerBlock = kWaves > 4 ? 1 : 4 / kWaves;
  __shared__ float partial[kWaves > 4 ? kWaves : 4];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int out_row = blockIdx.x * kRowsPerBlock + wave / kWaves;
  const int part = wave % kWaves;
  const bool active = out_row < rows;
  const int64_t in_row = kGrouped ? int64_t(out_row % m) * groups + out_row / m : out_row;
  const uint16_t* src = x + in_row * k;

  u32x4 packed[kPacks];
  float amax = 0.f;
#pragma unroll
  for (int i = 0; i < kPacks; ++i) {
    const int col = ((i * kWaves + part) * kWave + lane) * 8;
    packed[i] = u32x4{0, 0, 0, 0};
    if (active && col < k) packed[i] = load16<nt_loads(kPolicy)>(src + col);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t word = packed[i][j];
      amax = fmaxf(amax, fabsf(__uint_as_float(word << 16)));
      amax = fmaxf(amax, fabsf(__uint_as_float(word & 0xFFFF0000u)));
    }
  }
  amax = wave_max(amax);
  if constexpr (kWaves > 1) {
    // Waves (wave / kWaves) * kWaves .. + kWaves - 1 share this row.
    if (lane == 0) partial[wave] = amax;
    __syncthreads();
    const int first = wave - part;
    amax = partial[first];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) amax = fmaxf(amax, partial[first + w]);
  }
  if (!active) return;
  const float scale = fmaxf(amax / 127.f, 1e-20f);
  const float inv = 1.f / scale;
  if (part == 0 && lane == 0) scales[out_row] = scale;
  // Codes are at most INT_MAX bytes.
  const uint32_t bytes = uint32_t(rows) * uint32_t(k), at = uint32_t(out_row) * uint32_t(k);
#pragma unroll
  for (int i = 0; i < kPacks; ++i) {
    const int col = ((i * kWaves + part) * kWave + lane) * 8;
    if (col < k) stream_store<kPolicy>(codes8(packed[i], scale, inv), codes, bytes, at + col);
  }
}

// Fallback for any k and any 2-byte alignment: one wave per row, two passes.
template <bool kGrouped>
__global__ void __launch_bounds__(256) quantize_rows_scalar_kernel(
    const uint16_t* __restrict__ x, int8_t* __restrict__ codes, float* __restrict__ scales,
    int rows, int k, int m, int groups) {
  const int lane = threadIdx.x & 63;
  const int out_row = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (out_row >= rows) return;
  const int64_t in_row = kGrouped ? int64_t(out_row % m) * groups + out_row / m : out_row;
  const uint16_t* src = x + in_row * k;
  float amax = 0.f;
  for (int col = lane; col < k; col += kWave) amax = fmaxf(amax, fabsf(bf16_to_f32(src[col])));
  amax = wave_max(amax);
  const float scale = fmaxf(amax / 127.f, 1e-20f);
  if (lane == 0) scales[out_row] = scale;
  int8_t* dst = codes + int64_t(out_row) * k;
  for (int col = lane; col < k; col += kWave)
    dst[col] = static_cast<int8_t>(code_byte(bf16_to_f32(src[col]) / scale));
}

template <bool kGrouped>
hipError_t dispatch(const void* x, int8_t* codes, float* scales, int rows, int k, int m,
                    int groups, hipStream_t stream) {
  const auto* src = static_cast<const uint16_t*>(x);
  const bool vec = (reinterpret_cast<uintptr_t>(x) % 16 == 0) &&
                   (reinterpret_cast<uintptr_t>(codes) % 8 == 0) && (k % 8 == 0);
  const int packs = (k + 511) / 512;  // 16-byte packs per lane with one wave per row
  const StreamPolicy policy =
      stream_policy(int64_t(rows) * k * 2, int64_t(rows) * k, kQuantizeWriteThrough);
#define CI8_QW(W, P)                                                                       \
  if (packs <= (W) * (P)) {                                                                \
    constexpr int kPerBlock = (W) > 4 ? 1 : 4 / (W);                                       \
    constexpr int kThreads = (W) > 4 ? 64 * (W) : 256;                                     \
    const auto kernel = with_policy(policy, [](auto p) {                                   \
      return quantize_rows_vec_kernel<P, W, kGrouped, decltype(p)::value>;                 \
    });                                                                                    \
    kernel<<<(rows + kPerBlock - 1) / kPerBlock, kThreads, 0, stream>>>(                   \
        src, codes, scales, rows, k, m, groups);                                           \
    return hipGetLastError();                                                              \
  }
  // Waves per row: four once a row has four packs, so each lane holds at most a few
  // 16-byte packs and a workgroup is one row. Measured on MI355X (us, 4 / 2 / 1 waves per
  // row): [128, 4096] 3.04 / 4.05 / 7.33, [16, 5120] 3.76 / 5.20 / 8.12, [256, 5120]
  // 3.37 / 4.31 / 7.11, [4096, 5120] 13.87 / 14.42 / 15.84: more waves keep more loads
  // in flight and let a row's stores start sooner.
  // When the rows do not fill the chip (128 rows on 256 CUs) the op is one
  // memory latency long, and eight waves of one pack per lane shorten it a little
  // (measured on MI355X in a quantize + fused_channel_mm step, 128 x 4096,
  // against four waves of two packs, same box and process: 11.80-11.86 against
  // 12.04-12.18 us on one box, 12.27-12.48 against 12.41-12.57 us on another; identical
  // codes).
  // Eight waves also pay for wider rows, up to 256 of them past 4,096 values and up to 1,024
  // past 8,192 (with the GEMM that follows, four / eight waves: [16, 17408], N = 5120 24.4 /
  // 23.7 us; [64, 8704] 17.0 / 16.8; [256, 17408] 53.2 / 52.3; [600, 17408] 89.6 / 88.3;
  // [1024, 8704] 56.1 / 55.0; [1300, 17408] 130.7 / 133.2).
  const bool eight = packs > 4 && rows <= (packs > 16 ? 1024 : 256);
  if (vec && eight) {
    CI8_QW(8, 1) CI8_QW(8, 2) CI8_QW(8, 3) CI8_QW(8, 5)
  }
  if (vec) {
    CI8_QW(1, 1) CI8_QW(2, 1) CI8_QW(4, 1) CI8_QW(4, 2) CI8_QW(4, 3) CI8_QW(4, 4)
    CI8_QW(4, 5) CI8_QW(4, 6) CI8_QW(4, 7) CI8_QW(4, 8) CI8_QW(4, 9) CI8_QW(4, 10)
    CI8_QW(4, 12) CI8_QW(4, 14) CI8_QW(4, 16) CI8_QW(4, 20) CI8_QW(4, 24) CI8_QW(4, 32)
  }
#undef CI8_QW
  quantize_rows_scalar_kernel<kGrouped><<<(rows + 3) / 4, 256, 0, stream>>>(
      src, codes, scales, rows, k, m, groups);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_quantize_rows(const void* x, int8_t* codes, float* scales, int m, int k,
                                hipStream_t stream) {
  return dispatch<false>(x, codes, scales, m, k, m, 1, stream);
}

hipError_t launch_quantize_grouped(const void* x, int8_t* codes, float* scales, int m,
                                   int groups, int k, hipStream_t stream) {
  if (m == 0) return hipSuccess;
  return dispatch<true>(x, codes, scales, m * groups, k, m, groups, stream);
}

}  // namespace ci8
