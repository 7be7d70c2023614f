// Cache policy of the streaming kernels (quantizers, SwiGLU, unpacking), whose output is the
// next kernel's operand. Plain C++ (no HIP), so a CPU test compiles it with g++.
//
// Measured on MI355X, us, the kernel alone and with the GEMM that follows it (identical
// outputs; nt: nontemporal):
//   Stores. Plain ones leave dirty lines in the L2s, which are written back when the kernel
//   ends. Nontemporal ones do not, but the GEMM then reads the output from HBM. Written through
//   to the 256 MB Infinity Cache (MALL), the output is both, past a fixed cost of about 0.1 us
//   that small outputs feel (plain / nt / written through):
//     quantize_rows [128, 4096] 2.95 / 2.94 / 3.05, + N = 4096 10.8 / 11.8 / 10.9; [512, 5120]
//       3.51 / 3.49 / 3.46, + N = 5120 25.9 / 27.5 / 25.7; [2048, 5120] 7.55 / 6.65 / 6.66, + N =
//       5120 53.4 / 59.8 / 52.8; [4096, 5120] (nt loads) 12.6 / 12.1 / 11.9, + N = 17408 286 / 287
//       / 284; [4096, 8704] (nt loads) 19.4 / 19.1 / 18.9, + N = 5120 163 / 174 / 162;
//     silu_mul [16, 2 x 17408] 2.06 / 2.06 / 1.94; [256, 2 x 8704] 3.44 / 3.16 / 2.90;
//   So outputs are written through from write_through_from bytes on, and stored plainly below.
//   With nontemporal loads (large inputs) the quantizers alone would still be up to 6% faster
//   with nt stores, where their GEMM loses more.
//   unpack_allspark stores plainly (plain / nt / written through: 2048 x 2048 3.42 / 3.40 / 3.65, +
//     M = 256 12.5 / 13.1 / 13.2; 4096 x 4096 7.6 / 6.5 / 6.8, + M = 256 21.7 / 21.9 / 21.0; 7168 x
//     5120 14.7 / 14.2 / 14.6, + M = 256 36.3 / 40.1 / 36.3; 17408 x 5120 39.1 / 34.3 / 38.9, + M =
//     64 62.9 / 63.9 / 63.5, M = 1024 128 / 138 / 127; rows that share lines, 3872 x 7360, + M = 19
//     19.5 / 22.4 / 20.5): a caller who restores a layer without using it at once loses up to 18%.
//   Input and output past the MALL together evict each other whatever the stores: nt loads and
//   stores (quantize_rows [16384, 8704] 75.7 -> 67.4 alone, + N = 5120 599 -> 592; silu_mul
//   [4096, 2 x 17408] 71.2 -> 64.5; unpack_allspark 17408 x 8704 56.0 -> 52.8, + M = 32 94.9 ->
//   88.0, M = 256 127 -> 117, M = 1024 198 -> 203).
//   Loads. Inputs past the eight 4 MB L2s, which the kernel reads once, are loaded
//   nontemporally, so that they do not push the outputs out: [1300, 17408] + N = 5120 133.2 ->
//   126.8; [16384, 5120] 374.9 -> 367.9; silu_mul_quantize [700, 2 x 17408] + N = 5120 90.8 -> 83.3.
#pragma once
#include <stdint.h>

namespace ci8 {

constexpr int64_t kL2Bytes = int64_t(32) << 20, kMallBytes = int64_t(256) << 20;
// From which output size on write-through stores pay.
constexpr int64_t kQuantizeWriteThrough = int64_t(2) << 20, kSiluWriteThrough = 0;

// Plain loads and stores; written-through stores; those with nontemporal loads; both
// nontemporal.
enum StreamPolicy { kCached, kWriteThrough, kNtLoads, kNtLoadsAndStores };
inline StreamPolicy stream_policy(int64_t in_bytes, int64_t out_bytes, int64_t write_through_from) {
  if (in_bytes + out_bytes > kMallBytes) return kNtLoadsAndStores;
  if (in_bytes > kL2Bytes) return kNtLoads;
  return out_bytes >= write_through_from ? kWriteThrough : kCached;
}

// f with the policy as a std::integral_constant-like argument.
template <StreamPolicy kPolicy>
struct PolicyConstant {
  static constexpr StreamPolicy value = kPolicy;
};
template <class F>
auto with_policy(StreamPolicy policy, F f) {
  switch (policy) {
    case kWriteThrough: return f(PolicyConstant<kWriteThrough>{});
    case kNtLoads: return f(PolicyConstant<kNtLoads>{});
    case kNtLoadsAndStores: return f(PolicyConstant<kNtLoadsAndStores>{});
    default: return f(PolicyConstant<kCached>{});
  }
}

}  // namespace ci8
