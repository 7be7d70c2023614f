// Host-side tile plans of the large-M GEMMs: how many rounds of one tile per CU a launch
// takes, and the column split of the persistent kernel. Plain C++ (no HIP), so a CPU test
// compiles it with g++ and checks the plans the dispatcher picks.
#pragma once
#include <stdint.h>

namespace ci8 {

// Tile sizes these rules price (the persistent kernel's 256 x 224 and 256 x 160 tiles,
// gemm_pp_kernel.h, and the one-wave-per-SIMD kernel's 256 x 256 tiles, gemm.hip).
constexpr int kPlanBM = 256, kPlanBN = 224, kPlanNarrowBN = 160, kPlanWideBN = 256;

// Time of a round of 160-wide tiles, in units where a round of 224-wide tiles takes 224
// (measured on MI355X, M = 16384, K = 17408: 5 rounds of 224-wide tiles
// over N = 4480 took 966-978 us, and the split launch over N = 5120 1114-1129 us, so the
// 160-wide round and the second launch took ~0.8 of a 224-wide round).
//
// The split gains less than its rounds suggest: the chip runs at its power limit, so a
// partly filled last round runs faster per tile than a full one. There the single
// launch's sixth round (192 of 256 CUs busy, 672 columns for 640) took ~161 us against
// ~195 us for a full round, and the split launch measured 1114-1129 against 1131-1145 us
// (same process, alternating, identical outputs; at K = 5120, 326.5-327.7 against
// 328.4-329.8 us): about 1%, mostly the 32 padded columns that the 160-wide tiles do not
// compute.
constexpr int64_t kNarrowRoundCost = 180;

// Column plan of the two-waves-per-SIMD GEMM (gemm_pp.hip) at m x n on `cus` CUs where
// pp_width (below) picks its 224-wide tiles: 224-wide
// tiles over the first n_head columns and 160-wide tiles over the rest (n_head = 0: one
// launch of 224-wide tiles over all n). `cost` is the planned rounds' time in units where a
// round of 224-wide tiles takes 224.
struct PPPlan {
  int n_head;
  int64_t cost;
};

inline PPPlan pp_plan(int m, int n, int cus) {
  const int64_t tiles_m = (m + kPlanBM - 1) / kPlanBM;
  const int64_t tiles = tiles_m * ((n + kPlanBN - 1) / kPlanBN);
  PPPlan plan{0, 0};
  if (cus <= 0) return plan;
  plan.cost = (tiles + cus - 1) / cus * kPlanBN;
  // A last round that keeps under half the CUs busy runs faster per tile than the split's
  // round of 160-wide tiles (same process, identical outputs: M = 2048, N = 17408, whose
  // third round holds 112 tiles, 155.4-155.7 us in one launch against 156.7-157.4 us
  // split; M = 1100, N = 15516, 94 tiles, 106.4-106.9 us either way).
  const int64_t last = tiles % cus;
  if (last == 0 || 2 * last < cus) return plan;
  // Split: 224-wide tiles over the columns that the launch's whole rounds cover, then
  // 160-wide tiles over the rest.
  const int64_t head_tiles_n = tiles / cus * cus / tiles_m;
  const int64_t n_head = head_tiles_n * kPlanBN;
  if (head_tiles_n == 0 || n_head >= n) return plan;
  const int64_t head_rounds = (head_tiles_n * tiles_m + cus - 1) / cus;
  const int64_t tail_tiles = tiles_m * ((n - n_head + kPlanNarrowBN - 1) / kPlanNarrowBN);
  const int64_t cost = head_rounds * kPlanBN + (tail_tiles + cus - 1) / cus * kNarrowRoundCost;
  if (cost < plan.cost) plan = PPPlan{int(n_head), cost};
  return plan;
}

// Whether 256-wide large tiles finish an m x n GEMM sooner than 224-wide ones. A launch
// runs its tiles in rounds of one per CU, and a round takes time in proportion to the
// tile width, so the cost of a width is rounds x width. 224 suits N = 17408 at M = 4096
// (1,248 tiles, 4.9 rounds on 256 CUs, where 256-wide tiles need 4.25 rounds, i.e. 5);
// 256 suits N = 5120 at M = 16384 (5 full rounds against 5.75).
inline bool wide_tiles_pay(int m, int n, int cus) {
  if (cus <= 0) return false;
  const int64_t tiles_m = (m + kPlanBM - 1) / kPlanBM;
  const int64_t rounds224 = (tiles_m * ((n + kPlanBN - 1) / kPlanBN) + cus - 1) / cus;
  const int64_t rounds256 = (tiles_m * ((n + kPlanWideBN - 1) / kPlanWideBN) + cus - 1) / cus;
  return rounds256 * kPlanWideBN < rounds224 * kPlanBN;
}

// Whether the persistent kernel (one tile per CU per round, about 1.2x the MFMA rate of
// the 256-wide kernel) finishes sooner than 256-wide tiles: the cost of its column plan
// (rounds x width) against rounds x 256, weighted by that rate.
inline bool pp_beats_wide_tiles(int m, int n, int cus) {
  if (cus <= 0) return false;
  const int64_t tiles_m = (m + kPlanBM - 1) / kPlanBM;
  const int64_t rounds256 = (tiles_m * ((n + kPlanWideBN - 1) / kPlanWideBN) + cus - 1) / cus;
  return pp_plan(m, n, cus).cost * 6 <= rounds256 * kPlanWideBN * 7;
}

// Tile shapes of the small-M kernel (gemm_small.hip), as (BM, BN). A launch runs its tiles
// in rounds of one per CU, and a round lasts about as long as one tile takes to stream its
// (BM + BN) x K operand bytes, so the cost of a shape is rounds x (BM + BN); ties go to the
// larger tile (the earlier entry).
struct SmallShape {
  int bm, bn;
};
constexpr SmallShape kSmallShapes[] = {{64, 32}, {32, 64}, {16, 64}, {32, 32},
                                       {32, 16}, {16, 32}, {16, 16}};

inline int64_t small_shape_cost(SmallShape s, int m, int n, int cus) {
  const int64_t tiles = int64_t((m + s.bm - 1) / s.bm) * ((n + s.bn - 1) / s.bn);
  return (tiles + cus - 1) / cus * (s.bm + s.bn);
}

inline SmallShape small_best_shape(int m, int n, int cus) {
  SmallShape best = kSmallShapes[0];
  for (const SmallShape s : kSmallShapes)
    if (small_shape_cost(s, m, n, cus) < small_shape_cost(best, m, n, cus)) best = s;
  return best;
}

// Largest M the small-M kernel takes under schedule 0, and the M up to which only the ring
// kernel competes with it (gemm_choice).
constexpr int kSmallMaxM = 256, kSmallOnlyMaxM = 128;

// Tiles of the ring kernel (gemm_ring.hip), each with the time of a round of them (one tile
// on every CU): `fixed` + `per_k` * K / 1024 us. Fitted to 162 shapes measured on MI355X
// (M = 17..3000 with (N, K) = 4096 x 4096, 17408 x 5120, 5120 x 17408, 7168 x 5120, 5120 x
// 8704, 2048 x 8192, 1000 x 1024, 3000 x 2048 and 12000 x 3072; three rotated weight
// copies): rms error 5%, and the kernel that the times below pick took 1.2% longer than the
// best of all kernels in the mean. (64 x 80: 2.10 for a fitted 2.20; it is the faster one of
// its size when the weights come from HBM, M = 256, N = 5120, K = 17408: 43.7 against 47.0 us.)
struct RingTile {
  int bm, bn;
  double fixed, per_k;
};
constexpr RingTile kRingTiles[] = {
    {32, 64, 2.2, 1.29},  {32, 96, 2.4, 1.71},  {64, 48, 2.6, 1.55},  {64, 64, 2.6, 1.72},
    {64, 80, 3.2, 2.10},  {64, 96, 3.2, 2.23},  {64, 128, 3.5, 2.72}, {96, 96, 3.9, 2.71},
    {128, 80, 4.2, 3.23}, {96, 128, 4.1, 3.42}, {128, 128, 4.9, 4.13}, {128, 160, 5.5, 4.93},
    {192, 128, 6.2, 5.24}, {160, 160, 6.5, 5.42}, {192, 160, 6.9, 6.36}};
constexpr int kRingTileCount = sizeof(kRingTiles) / sizeof(kRingTiles[0]);

// Time (us) of one launch of a tiled GEMM that runs its tiles in rounds of one per CU: a
// round of the other kernels' tiles by the same measurements (the persistent kernel's tiles;
// 256-wide tiles of the one-wave-per-SIMD kernel; the small-M kernel below). A
// last round that is not full takes three quarters of a round plus its share of the rest
// (fewer CUs share the caches and the power; the best single share over all tiles).
constexpr double kLaunchTime = 1.5;
inline double tile_rounds(int64_t tiles, int cus) {
  const int64_t rest = tiles % cus;
  return double(tiles / cus) + (rest ? 0.75 + 0.25 * double(rest) / cus : 0.0);
}
inline double tiled_time(int64_t tiles, int cus, double fixed, double per_k, int k) {
  return kLaunchTime + tile_rounds(tiles, cus) * (fixed + per_k * k / 1024);
}
inline int64_t tile_count(int m, int n, int bm, int bn) {
  return int64_t((m + bm - 1) / bm) * ((n + bn - 1) / bn);
}
// The ring GEMM's launch; rounds past the first cost it 2% each on all (M = 2696, N = 17148, K =
// 3232, 6.3 rounds of 192 x 160: 228 us, 200 without). Below K = 1024 a round's fixed part shrinks,
// down to 70% (M = 10, N = 24936, K = 96 by 64 x 128 tiles: 3.96 us, 5.0 without).
inline double ring_time(const RingTile& t, int m, int n, int k, int cus) {
  const int64_t tiles = tile_count(m, n, t.bm, t.bn);
  const double rounds = tile_rounds(tiles, cus);
  const double fixed = t.fixed * (k < 1024 ? 0.7 + 0.3 * k / 1024 : 1.0);
  return tiled_time(tiles, cus, fixed, t.per_k, k) * (rounds > 1 ? 1 + 0.02 * (rounds - 1) : 1);
}
// Widths of the persistent kernel's tiles (256 rows each) with the time of a round, fitted to
// 122 shapes measured on MI355X (M = 320..16384; (N, K) = 17408 x 5120, 5120 x 17408, 7168 x
// 5120, 5120 x 8704, 4096 x 4096, 12000 x 3072, 8192 x 8192, 2560 x 10240, 8448 x 128, 4096 x
// 256, 12000 x 512, 8192 x 1024, 5120 x 2048, 20000 x 1024, 6144 x 8192; rms error 6-7%). A
// narrower tile costs more per column (more operand bytes per MFMA) and pays where it fills
// the rounds better: M = 2048, N = 5120, K = 17408 is 184 tiles of 224 or 256 of 160, one
// round each, 157.8 against 151.8 us; M = 2560, N = 12000, K = 3072 is 540 of 224 (95.0 us;
// 101.7 split) or 760 of 160, 85.8. With these times the choice of kernel and width is 0.5%
// off the best in the mean; with 224-wide tiles alone it was 3.7%.
struct PPWidth {
  int bn;
  double fixed, per_k;
};
constexpr PPWidth kPPWidths[] = {
    {kPlanBN, 9.1, 8.71}, {192, 6.9, 7.90}, {kPlanNarrowBN, 6.3, 7.23}, {128, 4.5, 6.77}};
inline double persistent_time(const PPWidth& w, int m, int n, int k, int cus) {
  return tiled_time(tile_count(m, n, kPlanBM, w.bn), cus, w.fixed, w.per_k, k);
}
// The width of a whole launch. 224 (which pp_plan may still split) unless another one is
// expected to save 1%; launch_pp_gemm runs it. cus <= 0: 224.
inline const PPWidth& pp_width(int m, int n, int k, int cus) {
  const PPWidth* best = kPPWidths;
  if (cus <= 0) return *best;
  double time = 0.99 * persistent_time(*best, m, n, k, cus);
  for (const PPWidth& w : kPPWidths) {
    const double t = persistent_time(w, m, n, k, cus);
    if (t < time) time = t, best = &w;
  }
  return *best;
}
inline double persistent_time(int m, int n, int k, int cus) {
  return persistent_time(pp_width(m, n, k, cus), m, n, k, cus);
}
inline double wide_time(int m, int n, int bn, int k, int cus) {
  return tiled_time(tile_count(m, n, kPlanBM, bn), cus, 9.7, 13.8 * bn / kPlanWideBN, k);
}
// The small-M kernel's launch: its rounds' fixed part grows with the tile as well, fitted to 638
// shapes (M <= 512, K = 32..16384; rms error 9%): M = 43, N = 928, K = 288 (174 tiles of 16 x 16)
// 2.4 us, the ring's best tile 3.6.
inline double small_time(int m, int n, int k, int cus) {
  const SmallShape s = small_best_shape(m, n, cus);
  const double rounds = double((tile_count(m, n, s.bm, s.bn) + cus - 1) / cus);
  return kLaunchTime + rounds * (s.bm + s.bn) * (0.019 + 0.012 * k / 1024);
}

// Schedule 0's kernel, by the times above: the ring kernel with tile kRingTiles[ring] where that
// is expected to beat the small-M kernel (up to kSmallMaxM), the persistent kernel (persistent_ok:
// it can run this call; above kSmallOnlyMaxM) and the one-wave-per-SIMD kernel with 256- or
// 224-wide tiles (from M = 1024 on; 256 where the persistent kernel can run). cus > 0.
// workspace: the INT32 products are stored too. out16: the output starts on 16 bytes.
//
// The times above are of BF16 outputs whose rows start on 16 bytes. What else costs time, fitted
// to 1600 shapes, half with N % 8 == 4 and a third with products, in us:
//   - the persistent kernel's narrower stores where rows do not start on 16 bytes: 1.0 per
//     million outputs and 6.5 a round (M = 1018, N = 7340, K = 1088: 26.7, which a 128 x 128 ring
//     tile does in 18.9);
//   - the products, per million: 0.85 + 0.03 per 1024 outputs of a ring tile (a round of large
//     tiles stores them all at its end), 1.3 for the one-wave-per-SIMD kernel, which the ring has
//     to be expected 5% below there (M = 2870, N = 3716, K = 5088: ring 120, that kernel 94);
//   - a K tail (K % 128) in 256-wide tiles of that kernel: it spills 174 registers a lane and
//     takes 2.8 times as long, so they are left out (M = 1335, N = 10392, K = 9568 with products
//     403, ring 210; M = 851, N = 6812, K = 1600 71.6 against 31.5 with 224-wide ones).
// The choice is 0.8-1.1% off the best kernel in the mean from K = 1024 on, and below 0.4% up to M
// = 256 and 2-4% beyond.
enum class GemmKernel { kSmall, kRing, kPersistent, kWide256, kWide224 };
struct GemmChoice {
  GemmKernel kernel;
  int ring;
};
inline GemmChoice gemm_choice(int m, int n, int k, int cus, bool persistent_ok, bool workspace,
                              bool out16 = true) {
  const double outputs = double(m) * n / 1e6;
  const bool whole_stages = k % 128 == 0;
  GemmChoice ring{GemmKernel::kRing, 0};
  double best = 0.0;
  for (int i = 0; i < kRingTileCount; ++i) {
    const RingTile& tile = kRingTiles[i];
    double t = ring_time(tile, m, n, k, cus);
    if (workspace) t += outputs * (0.85 + 0.03 * tile.bm * tile.bn / 1024);
    if (i == 0 || t < best) best = t, ring.ring = i;
  }
  // The ring has to be expected 3% below the small-M kernel: level by the times, it was 4% or more
  // slower at 13 of 293 shapes below K = 1024, and is at 6.
  if (m <= kSmallMaxM &&
      0.97 * (small_time(m, n, k, cus) + (workspace ? 0.85 * outputs : 0.0)) <= best)
    return {GemmKernel::kSmall, -1};
  if (m <= kSmallOnlyMaxM) return ring;
  if (persistent_ok) {
    // Where 224-wide persistent tiles lose to 256-wide ones on rounds, another width or the
    // ring kernel has to be expected 5% below those: M = 4096, N = K = 8192 (two full rounds
    // of 256, 2.69 of 192) 237.8 -> 216.8 us; M = 2048, N = K = 8192 (one round of 256, two of
    // 128, 2% below by the model) measured 118.8 against 124.9, M = 3072, N = 5120, K = 8192
    // (240 of 256, ring 2% below) 112.6 against 119.1.
    double time = persistent_time(m, n, k, cus);
    if (n % 8 != 0 || !out16) {  // the ring has to be expected 5% below, about the fit's error
      const int64_t tiles = tile_count(m, n, kPlanBM, pp_width(m, n, k, cus).bn);
      time = 0.95 * (time + outputs + 6.5 * tile_rounds(tiles, cus));
    }
    const double wide = 0.95 * wide_time(m, n, kPlanWideBN, k, cus);
    if (whole_stages && m >= 1024 && !pp_beats_wide_tiles(m, n, cus) && wide <= time)
      return wide <= best ? GemmChoice{GemmKernel::kWide256, -1} : ring;
    return time <= best ? GemmChoice{GemmKernel::kPersistent, -1} : ring;
  }
  const bool wide256 = whole_stages && wide_tiles_pay(m, n, cus);
  double wide = wide_time(m, n, wide256 ? kPlanWideBN : kPlanBN, k, cus);
  if (workspace) wide = 0.95 * (wide + 1.3 * outputs);
  if (m < 1024 || wide > best) return ring;
  return {wide256 ? GemmKernel::kWide256 : GemmKernel::kWide224, -1};
}

// Tiles of the GGUF ring kernel (gguf_ring.hip) with the time of a round, as kRingTiles:
// fitted to 162 shapes measured on MI355X (M = 1..3000; (N, K, groups) = (4096, 4096, 1),
// (1925, 2176, 1), (2808, 1792, 1), (1085, 1664, 4), (8192, 8192, 1), (3555, 3584, 1), (1024,
// 1024, 1), (5120, 2048, 2), (6000, 6016, 1)), rms error 5-8%.
constexpr RingTile kGgufTiles[] = {
    {16, 16, 1.9, 1.02}, {16, 32, 3.0, 1.25}, {32, 32, 3.5, 1.48},
    {64, 32, 4.9, 1.79}, {64, 64, 4.9, 3.15}, {96, 64, 6.1, 3.84},
    {128, 64, 6.6, 4.76}, {128, 96, 8.1, 6.50}, {128, 128, 10.0, 7.99}};
constexpr int kGgufTileCount = sizeof(kGgufTiles) / sizeof(kGgufTiles[0]);

// The most workgroups of `threads` that one launch can hold along x: HIP counts a launch's
// work-items in 32 bits and refuses more.
constexpr int64_t max_blocks(int threads) { return int64_t(UINT32_MAX) / threads; }
constexpr int kGgufRingThreads = 512;

// Time (us) of the span kernel (gguf_q8.hip, M <= 16) for `channels` of all groups per CU,
// which it pads to blocks of 16, and K, which its 16 waves' ranges pad to 2, 4, 5 or 8 blocks
// of 64 each: fitted to 685 shapes measured on MI355X (M = 1..16, N = 1024..8192, K =
// 1024..8192, one to four groups; rms error 4%). Rows of whole 128-byte lines take longer. Past
// 128 channels a CU the partial sums of K's chunks of 8192 do not fit and the tile kernel takes
// twice as long (N = 11877, K = 8704, four groups, M = 3: 136 us, the ring 80). Past 64 channels a
// CU with ranges past 4 blocks the fit is 18% short up to M = 8 (N = 8078, K = 7168, four groups,
// M = 2: 51.5 us for 44.2, the ring 45.5); beyond, the ring is the one that is short (M = 12, N =
// 7257, K = 7488: 51.1, the ring 55.8).
inline double gguf_span_time(int m, int64_t channels, int k) {
  const int range = (k + 1023) / 1024, blocks = int((channels + 15) / 16);
  const int held = range <= 2 ? 2 : range <= 4 ? 4 : range <= 5 ? 5 : (range + 7) / 8 * 8;
  const double time =
      2.05 + k / 1024.0 * ((k % 128 ? 0.425 : 0.58) + 0.37 * double(channels) / 16) +
      held * (0.0275 * m + 0.192 * blocks + (blocks > 5 ? 0.2 * (blocks - 5) : 0.0));
  if (k > 8192) return blocks > 8 ? 2 * time : time;
  return blocks > 4 && range > 4 && m <= 8 ? 1.18 * time : time;
}

// The ring tile for gguf_q8_packed_mm, or -1 where gguf_q8.hip's kernels are expected to be
// faster: its span kernel up to M = 16, its 256- or 128-row tiles beyond (large_rows, of which
// it takes the one with fewer rounds; a 128-row tile of at most 64 rows takes 8% less). The ring
// has to be expected 3% below the span kernel: of 304 shapes none is then more than 2.5% slower
// than by the span kernel, and the choice is 0.4% off the best kernel in the mean (N = 7022, K =
// 1344, M = 12: 4.8 us by the span kernel, 5.7 by the ring; N = 8038, K = 2112, two groups, M = 16
// 9.6 and 10.4; N = K = 8192, M = 1 21.2 and 14.4); past M = 16 it is 0.3% off over 392. At M <=
// 16, K <= 1024 and up to 16 channels a CU, where launch and latency are most of both, the ring's
// 16 x 16 tiles are faster up to K = 256, one stage, and the span kernel beyond, at each of 170
// shapes (N = 520, M = 2, K = 256 3.01 us and 3.23; N = 502, M = 14, K = 320 3.68 and 3.35). A tile
// whose workgroups a launch cannot hold (M = 2097120, N = 3, K = 2048, 512 groups: 8,388,608 of
// 128 x 64) is left out.
inline int gguf_large_rows(int m, int n, int groups, int cus) {
  const int64_t tiles256 = tile_count(m, n, 256, 128) * groups;
  const int64_t tiles128 = tile_count(m, n, 128, 128) * groups;
  return (tiles256 + cus - 1) / cus * 29 <= (tiles128 + cus - 1) / cus * 20 ? 256 : 128;
}
inline int gguf_ring_tile(int m, int n, int k, int groups, int cus) {
  if (cus <= 0) return -1;
  double best;
  if (m <= 16) {
    const int64_t channels = (int64_t(n) * groups + cus - 1) / cus;
    if (k <= 1024 && channels <= 16) return k <= 256 ? 0 : -1;
    best = 0.97 * gguf_span_time(m, channels, k);
  } else {
    const int rows = gguf_large_rows(m, n, groups, cus);
    best = tiled_time(tile_count(m, n, rows, 128) * groups, cus, rows == 256 ? 8.6 : 4.4,
                      rows == 256 ? 14.2 : 10.7, k);
    if (m <= 64) best *= 0.92;
  }
  int tile = -1;
  for (int i = 0; i < kGgufTileCount; ++i) {
    const RingTile& t = kGgufTiles[i];
    const int64_t tiles = tile_count(m, n, t.bm, t.bn) * groups;
    if (tiles > max_blocks(kGgufRingThreads)) continue;
    const double time = tiled_time(tiles, cus, t.fixed, t.per_k, k);
    if (time < best) best = time, tile = i;
  }
  return tile;
}

// Tiles of the grouped ring kernel (grouped_ring.hip) with the time of a round, `per_k` per
// 1024 of the K of all groups: fitted to 105 shapes measured on MI355X (M = 17..4096; (N,
// groups, K) = (4096, 4, 4096), (4616, 1, 4096), (2456, 3, 4096), (1496, 2, 4096), (8192, 2,
// 4096), (1024, 1, 4096), (3000, 3, 1056)), rms error 5-7%.
constexpr RingTile kGroupedTiles[] = {
    {32, 64, 3.1, 1.47},  {64, 64, 4.2, 1.89},   {96, 64, 4.6, 2.43},  {64, 96, 5.3, 2.44},
    {64, 128, 5.8, 2.74}, {96, 128, 6.4, 3.87},  {128, 96, 6.7, 3.89}, {128, 128, 7.1, 4.47},
    {160, 128, 8.4, 5.34}, {192, 128, 8.3, 6.01}};
constexpr int kGroupedTileCount = sizeof(kGroupedTiles) / sizeof(kGroupedTiles[0]);
// LDS kept for a tile's row scales of all groups, four bytes a row and group.
constexpr int kGroupedScaleBytes = 16 * 1024;

// The grouped ring tile, or -1 where the two-waves-per-SIMD kernel's 256 x 128 tiles
// (persistent_ok: it can run this call; 6.6 us per 1024 of K and round, past 7.8) are
// expected to be faster or the row scales of a tile do not fit. It always beats the 32 x
// 32-MFMA kernel (by 1.3 to 4 times at all 105 shapes). The choice is within 1% of the best
// kernel in the mean.
inline int grouped_ring_tile(int m, int n, int k, int groups, int cus, bool persistent_ok) {
  if (cus <= 0) return -1;
  auto time = [&](int bm, int bn, double fixed, double per_k) {
    return tiled_time(tile_count(m, n, bm, bn), cus, fixed, per_k * groups, k);
  };
  int tile = -1;
  double best = persistent_ok ? time(256, 128, 7.8, 6.6) : 0.0;
  for (int i = 0; i < kGroupedTileCount; ++i) {
    const RingTile& t = kGroupedTiles[i];
    if (int64_t(groups) * t.bm * 4 > kGroupedScaleBytes) continue;
    const double us = time(t.bm, t.bn, t.fixed, t.per_k);
    if ((tile < 0 && !persistent_ok) || us < best) best = us, tile = i;
  }
  return tile;
}

// channel_gemv: 8-channel copies per stage of the stream kernel (gemv_stream.hip) that fill
// the CUs in as few rounds of one tile each as its widest tile allows, or 0 where gemv.hip's
// kernels are faster. Measured on MI355X at 2563 drawn shapes, M = 1..16 (stream against those,
// us; "lines": rows of whole 128-byte lines, K % 128 == 0, of which the stream kernel reads no
// line twice):
//   K > 8192: M >= 3 everywhere (5120 x 17408, M = 5: 19.6 against 29.9; 2560 x 10240, M = 8: 8.5
//     against 17.0). M <= 2: with lines (5120 x 17408, M = 1: 18.9 against 23.1), but not where the
//     resident kernel's 16-channel workgroups, one or two a CU, fill the chip (3755 x 8832, M = 1:
//     8.8 against 8.2; 7846 x 9984, M = 2: 16.2 against 15.2; two a CU past K = 12000 the stream
//     again: 6352 x 17408, M = 2, with its first half 64.0 against 70.7). Without lines, M = 2 up
//     to 79 channels a CU (beyond 4% slower) and M = 1 from 17 to 48 (9121 x 13168: 26.7 against
//     32.0; 2128 x 14688: 10.0 against 9.6, 26801 x 9280: 55.1 against 47.2).
//   M >= 5, up to 16 channels a CU: with lines everywhere (4096 x 4096: 6.2-6.6 against 7.5-8.3).
//     Without, from K = 2048 on, at M <= 7 up to K = 7168 (2481 x 7824, M = 5: 8.7 against 8.2),
//     at M <= 6 and four channels a CU up to 5120 (586 x 5776, M = 6: 5.4 against 4.6); below K =
//     2048 where rows are whole half lines (1866 x 1984, M = 8: 3.5 against 3.7; otherwise 31
//     of 71 shapes ran 2-8% slower: 1684 x 1040, M = 10 3.4 against 3.1) and below K = 1024 (3622 x
//     80, M = 16: 2.7 against 3.0; 366 x 944: 2.9 against 3.1), there up to 20 channels a CU (4373
//     x 16, M = 10: 2.9 against 3.3).
//   17 to 20 channels a CU (24 computed): with lines up to 19, or from K = 5120 on (5120 x 5120:
//     8.2-9.4 against 8.5-10.9; 5036 x 3456, M = 9: 7.8 against 7.5); without, M >= 13 from 18
//     channels and K = 5120 on (5047 x 5568, M = 14: 10.4 against 11.7; 4839 x 1808, M = 14: 5.6
//     against 4.9).
//   Up to 40 channels a CU, K >= 5120: M >= 9 with lines (7168 x 5120 9.8-9.9 against 9.8-11.4,
//     8192 x 8192 15.8-16.7 against 17.4-19.3), M >= 13 without (8630 x 7056, M = 11: 15.8
//     against 15.3). Beyond, the span kernel is level or faster (12000 x 6000, M = 9: 15.9
//     against 16.3; 28672 x 8192: 48.5 against 51.0), and so are the row and quad kernels at M <=
//     4 (17408 x 5120, M = 2: 15.6 against 18.7).
//   Past 96 MB of weights with lines, with nontemporal copies (below): M >= 9, K >= 4096 (14336 x
//     8192 24.0-24.1 against 28.7-31.2; 28672 x 8192 45.1-46.2 against 47.7-50.1; 28672 x 4096
//     26.6-27.2 against 27.9-28.7) and M >= 5, K = 4224..5120 (34816 x 5120 35.1-37.7 against
//     37.8-40.2; 24576 x 5120 25.0-28.1 against 26.9-29.1). At M = 5..8 the quad kernel is faster
//     past K = 5120 (28672 x 8192, M = 5: 41.4 against 45.9) and the span kernel at K = 4096
//     (28672 x 4096: 27.1 against 27.8).
// Of 363 shapes drawn from the operator's range 5 are more than 2.5% slower than by gemv.hip's
// kernels (45 with every K > 8192, M >= 5 up to 20 channels, and M >= 9, K >= 5120 up to 40).
constexpr int kStreamMaxCopies = 9;
// Whether the stream kernel copies W nontemporally: past 96 MB, in whole lines. Plain / nt:
// 14336 x 8192, M = 9 27.0 / 24.0, 20480 x 10240, M = 1 43.2 / 39.9; 89 MB: 17408 x 5120, M =
// 16 19.2 / 19.7; rows that start inside a line: 9121 x 13168, M = 1 27.1 / 29.5.
inline bool gemv_stream_nontemporal(int n, int k) {
  return k % 128 == 0 && int64_t(n) * k > int64_t(96) << 20;
}
inline bool gemv_stream_pays(int m, int64_t channels, int n, int k) {
  const bool lines = k % 128 == 0;
  if (gemv_stream_nontemporal(n, k) && ((m >= 9 && k >= 4096) || (m >= 5 && k > 4096 && k <= 5120)))
    return true;
  if (k > 8192) {
    if (m >= 3) return true;
    if (!lines) return m == 2 ? channels < 80 : channels > 16 && channels <= 48;
    return !(m == 1 && channels > 8 && channels <= 16) &&
           !(channels > 24 && channels <= 32 && k < 12000);
  }
  if (m < 5) return false;
  if (channels <= 16 || (channels <= 20 && k < 1024)) {
    if (lines) return true;
    if (k < 2048) return k < 1024 || k % 64 == 0;
    return m >= 8 || k < (m <= 6 && channels <= 4 ? 5120 : 7168);
  }
  if (lines && (channels <= 19 || (channels <= 20 && k >= 5120))) return true;
  return channels <= 40 && k >= 5120 && (lines ? m >= 9 : m >= 13 && channels >= 18);
}
inline int gemv_stream_copies(int m, int n, int k, int cus) {
  if (cus <= 0) return 0;
  const int64_t channels = (int64_t(n) + cus - 1) / cus;
  if (!gemv_stream_pays(m, channels, n, k)) return 0;
  const int64_t rounds = (channels + 8 * kStreamMaxCopies - 1) / (8 * kStreamMaxCopies);
  return int(((int64_t(n) + cus * rounds - 1) / (cus * rounds) + 7) / 8);
}

}  // namespace ci8
