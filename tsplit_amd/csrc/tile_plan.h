// Which tile of the tile kernel (gemm_tile.h) a product runs on and into how many ranges its depth is cut: a small model of
// the chip, with figures measured on it.
//
// A CU takes its blocks in rounds of as many as are resident at once.  A 32-deep step of a round takes what it takes with that many
// blocks on the CU: one block alone waits for its barriers and loads, several fill each other's gaps (a 64 x 64 tile: 0.52 us alone,
// 2.5 for five; the matrix pipes need 0.43 for each).  Every round costs its first loads and its stores on top, and the ranges cost
// a second launch, which folds them, and its traffic.
//
// The figures come from the times of 617 launches (products and convolutions of ResNet-50, Inception-v4, VGG, a Transformer and drawn
// shapes, on each of the four tiles with up to 30 counts of ranges): a least-squares fit without negative figures, then moved by up to
// a quarter where that makes the choices better.  What a choice costs over the best of the four tiles and all counts, averaged: products
// and layers of one tap 0.9 %, gathered 0.9, pairs of phases 0.5, filter gradients 1.1 (x in words) and 0.7.  A model whose step took
// the same time however many blocks shared the CU, fitted to one count of ranges and with five 64 x 64 blocks resident everywhere, cost
// 1.9, 2.9, 4.0, 2.2 and 3.3 %, at worst 40 (18 x 25088 x 4096 with the second operand transposed: 153 us on 64 x 128, 109 on 64 x 64;
// 3x3 of 512 -> 512 at 7 x 7, data gradient: 181 us in 5 ranges, 156 in 6).
#pragma once
#include <algorithm>
#include <cstdint>

namespace tsplit {

struct TileKind {
  int bm, bn;
};
constexpr TileKind kTiles[] = {{128, 128}, {64, 128}, {128, 64}, {64, 64}};
struct TileCost {
  int resident[4];       // blocks a CU holds of each tile
  double step[4][5];     // us of a step with 1, 2, ... of them on the CU
  double round[4];       // us
  double fold, fold_tb;  // us; TB/s
};
// products
constexpr TileCost kProductCost = {{2, 3, 3, 5},
                                   {{2.59, 3.73}, {1.35, 1.93, 2.82}, {1.21, 2.19, 2.85}, {0.52, 0.96, 1.37, 2.03, 2.47}},
                                   {2.0, 1.3, 2.0, 1.2}, 2.2, 7.2};
// convolutions of one tap
constexpr TileCost kOneTapCost = {{2, 3, 3, 5},
                                  {{1.88, 3.76}, {1.41, 2.28, 2.84}, {0.89, 1.77, 2.84}, {0.48, 0.90, 1.25, 1.74, 2.46}},
                                  {4.2, 2.5, 2.6, 2.3}, 0.5, 11.8};
// one operand gathered by tap: a load and a row of LDS for every 64 values instead of every 256
constexpr TileCost kGatheredCost = {{2, 3, 3, 5},
                                    {{2.44, 4.63}, {1.34, 2.34, 3.57}, {1.44, 2.68, 3.27}, {0.82, 1.25, 1.77, 2.36, 3.07}},
                                    {1.9, 1.7, 0.7, 0.9}, 2.5, 8.1};
// the same in pairs of phases (data gradients of stride 2)
constexpr TileCost kPairsCost = {{2, 3, 3, 5},
                                 {{4.10, 6.99}, {1.87, 3.79, 4.41}, {1.62, 2.98, 4.18}, {0.82, 1.34, 1.92, 3.02, 4.00}},
                                 {3.6, 2.9, 0.8, 1.3}, 1.1, 4.9};
// filter gradients, x in words and by tap: rows of LDS are padded (34 KB for 64 x 64: four blocks, not five).  With several taps
// the ranges are folded even if there is one.
constexpr TileCost kFilterWordsCost = {{2, 3, 3, 4},
                                       {{2.50, 4.25}, {1.22, 2.00, 3.00}, {1.30, 2.40, 3.20}, {0.65, 1.14, 1.67, 2.19}},
                                       {1.5, 1.5, 1.0, 0.3}, 2.0, 7.5};
constexpr TileCost kFilterTapsCost = {{2, 3, 3, 4},
                                      {{3.38, 4.57}, {1.44, 3.07, 3.68}, {1.35, 2.40, 3.34}, {0.85, 1.36, 2.04, 2.49}},
                                      {0.6, 0.5, 0, 0}, 2.0, 6.2};
struct TilePlan {
  int tile, S;
  double us = 0;   // what the model takes it to cost
};

// A launch of `parts` products of M rows each (the phases of a strided data gradient; 1 otherwise), every one `batch` times:
// part i has cols[i] columns and a depth of steps[i] x 32.  max_split 1: the depth stays whole.
inline TilePlan plan_tiles(int64_t M, const int64_t *cols, const int *steps, int parts, int64_t batch, int max_split, double out_values,
                           const TileCost &cost) {
  TilePlan best{0, 1, 1e300};
  int deepest = 1;
  for (int i = 0; i < parts; ++i) deepest = std::max(deepest, steps[i]);
  for (int t = 0; t < 4; ++t) {
    const TileKind &k = kTiles[t];
    const int resident = cost.resident[t];
    int64_t tiles = 0;
    double work = 0;   // steps of all tiles
    for (int i = 0; i < parts; ++i) {
      const int64_t n = ((M + k.bm - 1) / k.bm) * ((cols[i] + k.bn - 1) / k.bn) * batch;
      tiles += n;
      work += static_cast<double>(n) * steps[i];
    }
    auto consider = [&](int S) {
      const int per = (deepest + S - 1) / S;
      S = (deepest + per - 1) / per;
      const int64_t n = (tiles * S + 255) / 256, whole = n / resident, rest = n - whole * resident;   // blocks of the busiest CU
      const double mean = parts == 1 ? per : std::max(1.0, work / (static_cast<double>(tiles) * S));
      double us = whole * (mean * cost.step[t][resident - 1] + cost.round[t]);
      if (rest) us += mean * cost.step[t][rest - 1] + cost.round[t];
      if (S > 1) us += cost.fold + (2 * S + 1) * out_values * 4 / (cost.fold_tb * 1e6);
      if (us < best.us) best = {t, S, us};
    };
    const int most = tiles > 1024 ? 1 : std::min(max_split, deepest);
    for (int S = 1, by = 1; S <= most; S += by) {   // 1 to 8, then four to every doubling
      if (S == 8 * by) by *= 2;
      consider(S);
    }
    // as many ranges as give every CU the same number of blocks
    for (int n = 1; n <= 10; ++n)
      if (const int64_t S = tiles > 0 ? 256 * n / tiles : 0; S > 1 && S <= most) consider(static_cast<int>(S));
  }
  return best;
}

// Small products go to the kernel whose blocks share the depth of one small tile among their waves (gemm_waves.h), where that takes less.
//
// The depth is cut into the tile kernel's own ranges, so that a result has the bits that the tile kernel and the fold give it.  Four waves that
// dealt a whole depth among them 32 values at a time were as fast, but their chains of K / 4 roundings where the tile kernel has K / 16 were
// 1.6 times further from float64 at 128 x 256 over 784 and 1.9 times at 64 x 1000 over 2048.  Up to four ranges where the tile kernel has one to
// three take 0.75-0.9 of the time at depths of 64 to 160 (784 x 256 over 128 4.7-5.0 us, 5.2-5.8 on the tile kernel), but give other bits.
// `whole`: batches, whose depth that kernel cannot cut; they are cut into up to four, whose chains are shorter.
//
// A launch here costs what any launch does, and for every block of the busiest CU a part of its own and one for each value of the depth that
// the busiest wave takes; beyond 2048 of them 8 % more, where loads bound it.  The figures are from 217 shapes, rows 1 to 2048, columns 10 to
// 5003, depth 10 to 65536, batches among them, in the four forms on the four tiles with the depth in four ranges and more: 9 % rms off, the tile
// kernel's model (launches included) 15 %.  Over 260 other shapes, replayed from a graph, with this rule 1.26 times faster than the tile kernel
// alone, none slower by more than 6 %.  In the four forms, tile kernel -> here: 128 x 256 over 784 7.1-7.3 -> 5.0-5.3 us, over 256 6.4-6.6 ->
// 3.7-4.1, 256 x 256 over 128 5.2-5.7 -> 3.7-3.9, 385 x 256 over 1024 9.3-9.8 -> 7.1-8.8, 32 x 4096 over 1024 11.1-12.1 -> 7.1-8.9, 64 x 1000
// over 2048 10.4-10.8 -> 7.7-10.1, 1 x 1908 over 308 6.3-6.8 -> 3.7-4.1, 16 of 64 x 64 over 2048 41-49 -> 8-10; where the tile kernel stays:
// 250 x 5003 over 256 12.2-12.8, 512 x 512 over 64 4.1-4.3 (4.9-5.1 on 32 x 32 here), over 4096 26-28 (27-28).  Beyond 16384 values operands
// come from memory in parts of lines: 1 x 3000 over 16384 53-56 -> 39-59, over 32768 101-107 -> 110-134, so those stay too.
constexpr TileKind kWaveTiles[] = {{16, 16}, {16, 32}, {32, 16}, {32, 32}};
struct WavesPlan {
  int tile, waves;   // waves 0: the tile kernel
  int S, kchunk;     // the ranges that the waves take in turn
};
inline WavesPlan plan_waves(int64_t M, int64_t N, int64_t K, int64_t batch, const TilePlan &tile_kernel, bool whole) {
  constexpr double kLaunch = 3.56, kBlock[] = {0, 0.186, 0.363, 0.951}, kDepth[] = {0.00245, 0.00345, 0.00337, 0.00513};
  WavesPlan best{0, 0, 1, 0};
  if (K <= 0 || (!whole && K > 16384)) return best;
  const int64_t ranges = whole ? 4 : tile_kernel.S, steps = (K + 31) / 32, per = (steps + ranges - 1) / ranges, S = (steps + per - 1) / per;
  const int64_t waves = std::min<int64_t>(4, S), deep = (S + waves - 1) / waves * std::min(4 * K, per * 128);   // 4 x what the busiest wave takes
  double least = 2.3 + 1.15 * tile_kernel.us;
  for (int t = 0; t < 4; ++t) {
    const int64_t blocks = ((M + kWaveTiles[t].bm - 1) / kWaveTiles[t].bm) * ((N + kWaveTiles[t].bn - 1) / kWaveTiles[t].bn) * batch;
    // (the ranges' results lie in LDS: two blocks a CU)
    if (blocks > 1024 || S * (kWaveTiles[t].bm + 1) * kWaveTiles[t].bn * 4 > 81920) continue;
    const int64_t n = (blocks + 255) / 256;
    const double us = (kLaunch + n * (kBlock[t] + kDepth[t] * deep)) * (deep > 2048 ? 1.08 : 1);
    if (us < least) {
      least = us;
      // A wave without a range still adds and stores: with a CU of their own four waves are 3 % faster than two at one or two ranges, where blocks
      // share one up to 8 % slower.  Eight or sixteen gain nothing (over the shapes 0.2 %).
      best = {t, n == 1 ? 4 : std::max(2, static_cast<int>(waves)), static_cast<int>(S), static_cast<int>(per * 32)};
    }
  }
  return best;
}

}  // namespace tsplit
