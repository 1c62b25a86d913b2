// Launches of the tile kernel for convolutions (conv_tile.h).
#include "conv_tile.h"

#include <algorithm>

#include "common.h"
#include "conv_reach.h"
#include "tile_plan.h"

namespace tsplit {
namespace {

using namespace ct;

template <int TM, int TN, bool BWD, int GATHER, bool ACROSS>
void launch_one(const Params &P, unsigned grid, int total, hipStream_t st) {
  if constexpr (!BWD)
    if (P.stats) {
      hipLaunchKernelGGL((conv_tile_kernel<TM, TN, BWD, GATHER, ACROSS, true, false>), dim3(grid), dim3(gt::kThreads), 0, st, P, total);
      return;
    }
  if constexpr (ACROSS)
    if (P.add) {
      hipLaunchKernelGGL((conv_tile_kernel<TM, TN, BWD, GATHER, ACROSS, false, true>), dim3(grid), dim3(gt::kThreads), 0, st, P, total);
      return;
    }
  hipLaunchKernelGGL((conv_tile_kernel<TM, TN, BWD, GATHER, ACROSS, false, false>), dim3(grid), dim3(gt::kThreads), 0, st, P, total);
}

template <bool BWD, int GATHER, bool ACROSS>
void launch_tile(const Params &P, int tile, unsigned grid, int total, hipStream_t st) {
  switch (tile) {
    case 0: return launch_one<4, 4, BWD, GATHER, ACROSS>(P, grid, total, st);
    case 1: return launch_one<2, 4, BWD, GATHER, ACROSS>(P, grid, total, st);
    case 2: return launch_one<4, 2, BWD, GATHER, ACROSS>(P, grid, total, st);
    default: return launch_one<2, 2, BWD, GATHER, ACROSS>(P, grid, total, st);
  }
}

void launch_pair(const Params &P, int tile, unsigned grid, int total, hipStream_t st) {
  switch (tile) {
    case 0: hipLaunchKernelGGL((conv_tile_pair_kernel<4, 4>), dim3(grid), dim3(gt::kThreads), 0, st, P, total); break;
    case 1: hipLaunchKernelGGL((conv_tile_pair_kernel<2, 4>), dim3(grid), dim3(gt::kThreads), 0, st, P, total); break;
    case 2: hipLaunchKernelGGL((conv_tile_pair_kernel<4, 2>), dim3(grid), dim3(gt::kThreads), 0, st, P, total); break;
    default: hipLaunchKernelGGL((conv_tile_pair_kernel<2, 2>), dim3(grid), dim3(gt::kThreads), 0, st, P, total); break;
  }
}

// Runs the phases of P; tiles and ranges are filled in here.  out_values: elements of the output, negative if this launch does
// not write all of them (the fold of ranges adds whole tensors).  add: what the output is added to (`across` alone); null: nothing.
int run_phases(Params &P, bool bwd, int gather, bool across, bool pairs, float *out, int64_t out_values, hipStream_t st, StatsSink *sink,
               const float *add = nullptr) {
  int64_t cols[kMaxPhases];
  int steps[kMaxPhases];
  const int step = pairs ? 2 : 1;
  int parts = 0;
  for (int i = 0; i < P.phases; i += step, ++parts) {
    cols[parts] = P.phase[i].N;
    steps[parts] = (P.phase[i].K + BK - 1) / BK + (pairs ? (P.phase[i + 1].K + BK - 1) / BK : 0);
  }
  const TileCost &cost = gather == kWords || gather == kOneTap ? kOneTapCost : pairs ? kPairsCost : kGatheredCost;
  const TilePlan plan = plan_tiles(P.M, cols, steps, parts, 1, out_values < 0 ? 1 : 32, static_cast<double>(out_values), cost);
  const TileKind &k = kTiles[plan.tile];
  int S = 1;
  const int tm = (P.M + k.bm - 1) / k.bm;
  int tiles = 0;
  for (int i = 0; i < P.phases; ++i) {
    Phase &F = P.phase[i];
    F.first_tile = tiles;
    if (i % step == 0) tiles += tm * ((F.N + k.bn - 1) / k.bn);
    const int ksteps = (F.K + BK - 1) / BK;
    F.kchunk = std::max(1, (ksteps + plan.S - 1) / plan.S) * BK;
    S = std::max(S, (F.K + F.kchunk - 1) / F.kchunk);
  }
  P.tm = FastDiv(tm);
  P.tiles = FastDiv(tiles);
  TS_REQUIRE(static_cast<int64_t>(tiles) * S < (1ll << 31) - 8, "conv: too many tiles");
  P.stats = nullptr;
  if (sink && S > 1) {   // the output has the same bits with and without the sums
    sink->missing = true;
  } else if (sink) {
    const int groups = (P.phase[0].N + k.bn / 2 - 1) / (k.bn / 2);   // a wave's columns
    TS_REQUIRE(sink->used + groups <= sink->capacity, "conv: statistics buffer too small");
    P.stats = sink->part + static_cast<int64_t>(sink->used) * P.M * 2;
    sink->used += groups;
  }
  P.out = out;
  P.add = S > 1 ? nullptr : add;
  P.z_stride = 0;
  if (S > 1) {
    P.out = static_cast<float *>(scratch_get(st, 2, static_cast<size_t>(S) * out_values * sizeof(float)));
    TS_REQUIRE(P.out, "conv: no scratch memory for the ranges' results");
    P.z_stride = out_values;
  }
  const unsigned grid = mg::grid_blocks(tiles, 1, S);
  const int total = tiles * S;
  if (pairs) {
    launch_pair(P, plan.tile, grid, total, st);
  } else if (!bwd) {
    switch (gather) {
      case kWords: launch_tile<false, kWords, false>(P, plan.tile, grid, total, st); break;
      case kOneTap: launch_tile<false, kOneTap, false>(P, plan.tile, grid, total, st); break;
      case kBlocks32: launch_tile<false, kBlocks32, false>(P, plan.tile, grid, total, st); break;
      case kBlocks64: launch_tile<false, kBlocks64, false>(P, plan.tile, grid, total, st); break;
      default: launch_tile<false, kTaps64, false>(P, plan.tile, grid, total, st); break;
    }
  } else if (across) {
    if (gather == kWords)
      launch_tile<true, kWords, true>(P, plan.tile, grid, total, st);
    else
      launch_tile<true, kOneTap, true>(P, plan.tile, grid, total, st);
  } else {
    switch (gather) {
      case kBlocks32: launch_tile<true, kBlocks32, false>(P, plan.tile, grid, total, st); break;
      case kBlocks64: launch_tile<true, kBlocks64, false>(P, plan.tile, grid, total, st); break;
      default: launch_tile<true, kTaps64, false>(P, plan.tile, grid, total, st); break;
    }
  }
  if (S > 1) gt::launch_fold(P.out, out, out_values, S, st, add);
  return 0;
}

inline int padded(int chans) { return (chans + 7) / 8 * 8; }
// blocks of 8 channels, unless padding the last one adds more depth than the filter's own order costs
inline bool in_blocks(int chans) { return padded(chans) * 3 <= chans * 4; }

// filters re-laid in tiles (below that a launch of either takes what any launch takes: 590 K values 5.7 us by single values, the call 2 us
// longer in tiles)
constexpr int kRelayTilesFrom = 1 << 20;
// the re-laid filter of P's phases (their K and w_at are set), in scratch
int relay(Params &P, const float *w, int rows, int chans, int w_row, int w_chan, int f_w, int s, const int (*first_tap)[2], bool plain,
          hipStream_t st) {
  Relay R;
  R.w = w;
  R.rows = rows;
  R.chans = chans;
  R.w_row = w_row;
  R.w_chan = w_chan;
  R.f_w = f_w;
  R.s = s;
  R.phases = P.phases;
  R.plain = plain;
  R.total = 0;
  for (int i = 0; i < P.phases; ++i) {
    Phase &F = P.phase[i];
    F.w_at = R.total;
    R.phase[i] = RelayPhase{F.w_at, F.K, first_tap[i][0], first_tap[i][1], F.taps, F.kw, FastDiv(std::max(1, F.K))};
    R.total += rows * F.K;
  }
  R.out = static_cast<float *>(scratch_get(st, 3, static_cast<size_t>(std::max(4, R.total)) * sizeof(float)));
  TS_REQUIRE(R.out, "conv: no scratch memory for the re-laid filter");
  const int taps = static_cast<int>(P.phase[0].taps.d);
  if (P.phases == 1 && s == 1 && !plain && static_cast<int>(P.phase[0].kw.d) == f_w && taps <= 25 && R.total >= kRelayTilesFrom) {
    const int all = (chans + 7) / 8 * 8, tiles = (all + kRelayChans - 1) / kRelayChans;
    hipLaunchKernelGGL(conv_relay_tiles_kernel, dim3((rows + kRelayRows - 1) / kRelayRows * tiles), dim3(256),
                       kRelayRows * (kRelayChans + 1) * taps * sizeof(float), st, w, R.out, rows, chans, all, P.phase[0].taps, w_row, w_chan,
                       FastDiv(tiles));
  } else if (R.total > 0) {
    hipLaunchKernelGGL(conv_relay_kernel, dim3((R.total + 255) / 256), dim3(256), 0, st, R);
  }
  P.w = R.out;
  return 0;
}

}  // namespace

// The kernels' bit masks hold 64 taps, a data gradient's launch plan 64 phases; 32-bit byte offsets reach the filter as it is
// re-laid and, from the first image a tile touches, the images of its 128 columns.
bool conv_tile_takes(const ConvTileGeo &g, bool bwd) {
  const int64_t in = padded(g.C), out = padded(g.O);
  const int64_t img = bwd ? static_cast<int64_t>(g.C) * g.H * g.W : static_cast<int64_t>(g.O) * g.oH * g.oW;
  const int64_t cols = std::max<int64_t>(1, bwd ? static_cast<int64_t>(g.H / g.s) * (g.W / g.s) : static_cast<int64_t>(g.oH) * g.oW);
  return g.kH * g.kW <= 64 && (!bwd || g.s <= 8) && in * out * g.kH * g.kW < (1ll << 29) && img * (128 / cols + 2) < (1ll << 29);
}

int conv_tile_forward(const float *x, const float *w, float *y, const ConvTileGeo &g, hipStream_t st, StatsSink *sink) {
  const int taps = g.kH * g.kW;
  Params P;
  P.src = x;
  P.w = w;
  P.src_bytes = static_cast<unsigned>(static_cast<int64_t>(g.imgs) * g.C * g.H * g.W * 4);
  P.img_stride = g.C * g.H * g.W;
  P.chan_stride = g.H * g.W;
  P.chans = g.C;
  P.src_h = g.H;
  P.src_w = g.W;
  P.s = g.s;
  P.M = g.O;
  P.out_plane = g.oH * g.oW;
  P.out_img_stride = static_cast<int64_t>(g.O) * P.out_plane;
  P.out_h = g.oH;
  P.out_w = g.oW;
  P.out_s = 1;
  P.phases = 1;
  const bool inside = taps == 1 && g.ph == 0 && g.pw == 0, blocks = !inside && in_blocks(g.C);
  P.phase[0] = Phase{FastDiv(P.out_plane), FastDiv(g.oW), FastDiv(taps), FastDiv(g.kW), g.imgs * P.out_plane,
                     (blocks ? padded(g.C) : g.C) * taps, g.ph, g.pw, g.ph * g.W + g.pw, 0, 0, 0, 0, 0};
  if (blocks) {
    const int none[1][2] = {{0, 0}};
    if (relay(P, w, g.O, g.C, g.C * taps, taps, g.kW, 1, none, false, st)) return -1;
  }
  const int gather = inside ? (g.s == 1 && P.out_plane % 4 == 0 ? kWords : kOneTap) : !blocks ? kTaps64 : taps <= 32 ? kBlocks32 : kBlocks64;
  return run_phases(P, false, gather, false, false, y, static_cast<int64_t>(g.imgs) * P.out_img_stride, st, sink);
}

bool conv_tile_bwd_data_adds(const ConvTileGeo &g) { return g.kH * g.kW == 1 && g.ph == 0 && g.pw == 0 && g.s <= 2; }

int conv_tile_bwd_data(const float *dy, const float *w, const float *add, float *dx, const ConvTileGeo &g, hipStream_t st) {
  const int taps = g.kH * g.kW, s = g.s;
  Params P;
  P.src = dy;
  P.w = w;
  P.src_bytes = static_cast<unsigned>(static_cast<int64_t>(g.imgs) * g.O * g.oH * g.oW * 4);
  P.img_stride = g.O * g.oH * g.oW;
  P.chan_stride = g.oH * g.oW;
  P.chans = g.O;
  P.src_h = g.oH;
  P.src_w = g.oW;
  P.s = 1;
  P.M = g.C;
  P.out_plane = g.H * g.W;
  P.out_img_stride = static_cast<int64_t>(g.C) * P.out_plane;
  P.out_h = g.H;
  P.out_w = g.W;
  P.out_s = s;
  const int64_t values = static_cast<int64_t>(g.imgs) * P.out_img_stride;
  if (s == 1) {
    const bool inside = taps == 1 && g.ph == 0 && g.pw == 0, blocks = !inside && in_blocks(g.O);
    P.phases = 1;
    P.phase[0] = Phase{FastDiv(P.out_plane), FastDiv(g.W), FastDiv(taps), FastDiv(g.kW), g.imgs * P.out_plane,
                       (blocks ? padded(g.O) : g.O) * taps, g.ph, g.pw, (g.kH - 1) * g.oW + g.kW - 1, 0, 0, 0, 0, 0};
    if (inside) return run_phases(P, true, P.out_plane % 4 == 0 ? kWords : kOneTap, true, false, dx, values, st, nullptr, add);
    const int none[1][2] = {{0, 0}};
    if (relay(P, w, g.C, g.O, taps, g.C * taps, g.kW, 1, none, !blocks, st)) return -1;
    return run_phases(P, true, !blocks ? kTaps64 : taps <= 32 ? kBlocks32 : kBlocks64, false, false, dx, values, st, nullptr);
  }
  if (s == 2 && taps == 1 && g.ph == 0 && g.pw == 0) {   // the product over dy's positions, spread over dx
    P.phases = 1;
    P.phase[0] = Phase{FastDiv(P.chan_stride), FastDiv(g.oW), FastDiv(1), FastDiv(1), g.imgs * P.chan_stride, g.O, 0, 0, 0, 0, 0, 0, 0, 0};
    return run_phases(P, true, P.chan_stride % 4 == 0 ? kWords : kOneTap, true, false, dx, values, st, nullptr, add);
  }
  // phases (a, b): input positions a0 + s i, b0 + s j, reached by the filter taps a + s u, b + s v; by rows of positions, in
  // ascending order of b0
  const bool pairs = s == 2;
  Phase all[64];
  int first_tap[64][2], count = 0;
  for (int a0 = 0; a0 < s && a0 < g.H; ++a0)
    for (int b0 = 0; b0 < s && (pairs || b0 < g.W); ++b0) {
      const int a = (a0 + g.ph) % s, b = (b0 + g.pw) % s;
      const int hp = (g.H - a0 + s - 1) / s, wp = pairs ? (g.W + 1) / 2 : (g.W - b0 + s - 1) / s;
      const int nu = a < g.kH ? (g.kH - a + s - 1) / s : 0, nv = b < g.kW ? (g.kW - b + s - 1) / s : 0;
      first_tap[count][0] = a;
      first_tap[count][1] = b;
      all[count++] = Phase{FastDiv(hp * wp), FastDiv(wp), FastDiv(std::max(1, nu * nv)), FastDiv(std::max(1, nv)), g.imgs * hp * wp,
                           padded(g.O) * nu * nv, (a0 + g.ph - a) / s, (b0 + g.pw - b) / s, std::max(0, (nu - 1) * g.oW + nv - 1), a0, b0, 0, 0, 0};
    }
  for (int first = 0; first < count; first += kMaxPhases) {
    P.phases = std::min(kMaxPhases, count - first);
    for (int i = 0; i < P.phases; ++i) P.phase[i] = all[first + i];
    if (relay(P, w, g.C, g.O, taps, g.C * taps, g.kW, s, first_tap + first, false, st)) return -1;
    const int rc = run_phases(P, true, kBlocks32, false, pairs, dx, count <= kMaxPhases ? values : -1, st, nullptr);
    if (rc) return rc;
  }
  return 0;
}

}  // namespace tsplit
