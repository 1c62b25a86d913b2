// Launches of the filter gradient's tile kernel (conv_wgrad_tile.h) and the fold of its depth ranges.
#include "conv_wgrad_tile.h"

#include <algorithm>

#include "common.h"
#include "conv_reach.h"
#include "tile_plan.h"

namespace tsplit {
namespace {

using namespace wt;

// split-K fold for the tap-major bwd-filter: part[z][o][tap][c] summed over z (ascending, so the
// result does not depend on scheduling) and written as dw[o][c][tap]
// A block folds 64 outputs with 4 slice-lanes each (lane l adds slices l, l + 4, ...), combined
// through LDS in a fixed order.
__global__ __launch_bounds__(256) void fold_tap_major_kernel(const float *__restrict__ part, float *__restrict__ dw,
                                                             int O, int C, int kHW, int64_t stride, int S) {
  __shared__ float sm[3][64];
  const int cx = threadIdx.x & 63, ry = threadIdx.x >> 6;
  const int idx = blockIdx.x * 64 + cx;                // index into one partial: (o*kHW + tap)*C + c
  const bool live = idx < O * C * kHW;
  float acc = 0.f;
  if (live) {
#pragma unroll 4
    for (int z = ry; z < S; z += 4) acc += part[z * stride + idx];
  }
  if (ry > 0) sm[ry - 1][cx] = acc;
  __syncthreads();
  if (ry == 0 && live) {
    acc = ((acc + sm[0][cx]) + sm[1][cx]) + sm[2][cx];
    const int c = idx % C;
    const int t = idx / C;
    const int tap = t % kHW, o = t / kHW;
    dw[(o * C + c) * kHW + tap] = acc;
  }
}

// The same sums of few ranges, kFoldChans channels of one output channel a block: the taps of a channel come together in LDS, so that dw is
// written in whole lines: filter gradients of 512 -> 512, 64 images of 4 x 4 72 -> 66 us, of 2 x 2 40 -> 32; from a million values on (590 K: 61.1
// and 61.6, 173 K 17.5 and 22.1).
constexpr int kFoldChans = 64;
__global__ __launch_bounds__(256) void fold_tap_major_tiles_kernel(const float *__restrict__ part, float *__restrict__ dw, int C, FastDiv tiles, int kHW,
                                                                   int64_t stride, int S) {
  extern __shared__ float lds[];   // [channel][tap]
  const uint32_t o = tiles.div(blockIdx.x);
  const int c0 = (blockIdx.x - o * tiles.d) * kFoldChans, here = min(kFoldChans, C - c0);
  const float *from = part + static_cast<int64_t>(o) * kHW * C + c0;
  const int c = threadIdx.x & (kFoldChans - 1);
  for (int tap = threadIdx.x / kFoldChans; tap < kHW; tap += 256 / kFoldChans) {
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    if (c < here)
      for (int z = 0; z < S; z += 4)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (z + i < S) acc[i] += from[(z + i) * stride + static_cast<int64_t>(tap) * C + c];
    lds[c * kHW + tap] = ((acc[0] + acc[1]) + acc[2]) + acc[3];
  }
  __syncthreads();
  float *to = dw + (static_cast<int64_t>(o) * C + c0) * kHW;
  for (int e = threadIdx.x; e < here * kHW; e += 256) to[e] = lds[e];
}
constexpr int64_t kFoldTilesFrom = 1 << 20;

template <int G>
void launch_tile(const Params &P, int tile, const mg::TileGrid &tg, unsigned grid, hipStream_t st) {
  switch (tile) {
    case 0: hipLaunchKernelGGL((conv_wgrad_tile_kernel<4, 4, G>), dim3(grid), dim3(gt::kThreads), 0, st, P, tg); break;
    case 1: hipLaunchKernelGGL((conv_wgrad_tile_kernel<2, 4, G>), dim3(grid), dim3(gt::kThreads), 0, st, P, tg); break;
    case 2: hipLaunchKernelGGL((conv_wgrad_tile_kernel<4, 2, G>), dim3(grid), dim3(gt::kThreads), 0, st, P, tg); break;
    default: hipLaunchKernelGGL((conv_wgrad_tile_kernel<2, 2, G>), dim3(grid), dim3(gt::kThreads), 0, st, P, tg); break;
  }
}

// Channels of a group: a smaller group where it leaves a tenth of the columns out.  32 images, 7x7 filters, stride 1, 112 x 112, 353
// filters, in groups of 16 / 4 / 2: 3 channels 2039 / 737 / - us, 6 channels 2038 / 1182 / 891.  Where it leaves out less: 29 channels,
// 5x5, stride 2, 361 filters at 98 x 98 299 us in 16 and 327 in twos; 33 channels, 200 filters of 7x7 at 56 x 56 227 in fours and 257 in twos.
int group_size(int chans) {
  const int in16 = (chans + 15) / 16 * 16, in4 = (chans + 3) / 4 * 4, in2 = (chans + 1) / 2 * 2;
  if (in2 * 10 <= in4 * 9) return 2;
  return in4 * 10 <= in16 * 9 ? 4 : 16;
}

}  // namespace

void conv_fold_tap_major(const float *part, float *dw, int O, int C, int taps, int S, hipStream_t st) {
  const int64_t mn = static_cast<int64_t>(O) * C * taps, tiles = (C + kFoldChans - 1) / kFoldChans;
  // (a range's result written as a lane's four accumulators from zero adds up to the same bits)
  if (mn >= kFoldTilesFrom && C >= 32 && S <= 16 && taps <= 64 && tiles * O < (1ll << 31)) {
    hipLaunchKernelGGL(fold_tap_major_tiles_kernel, dim3(static_cast<unsigned>(tiles * O)), dim3(256), kFoldChans * taps * sizeof(float), st, part, dw, C,
                       FastDiv(static_cast<uint32_t>(tiles)), taps, mn, S);
    return;
  }
  hipLaunchKernelGGL(fold_tap_major_kernel, dim3(static_cast<unsigned>((mn + 63) / 64)), dim3(256), 0, st, part, dw, O, C, taps, mn, S);
}

bool conv_tile_bwd_filter_takes(const ConvTileGeo &g, int64_t reach) { return filter_gradient_in_reach(g, reach); }

int conv_tile_bwd_filter(const float *x, const float *dy, float *dw, const ConvTileGeo &g, int64_t reach, hipStream_t st, int64_t *ws_elems) {
  const int taps = g.kH * g.kW;
  Params P;
  P.dy = dy;
  P.x = x;
  P.dy_bytes = static_cast<int64_t>(g.imgs) * g.O * g.oH * g.oW * 4;
  P.x_bytes = static_cast<int64_t>(g.imgs) * g.C * g.H * g.W * 4;
  P.M = g.O;
  P.C = g.C;
  P.cols = taps * g.C;
  P.plane = g.oH * g.oW;
  P.dy_img = g.O * P.plane;
  P.K = static_cast<int>(padded_depth(g));
  P.image = FastDiv(depth_per_image(g));
  P.width = FastDiv(g.oW);
  P.kw = FastDiv(g.kW);
  P.x_plane = g.H * g.W;
  P.x_img = g.C * P.x_plane;
  P.x_h = g.H;
  P.x_w = g.W;
  P.ph = g.ph;
  P.pw = g.pw;
  P.s = g.s;
  const bool point = taps == 1 && g.s == 1 && g.ph == 0 && g.pw == 0;
  const int group = point ? 16 : group_size(g.C);
  P.groups = FastDiv((g.C + group - 1) / group);
  P.n_groups = taps * static_cast<int>(P.groups.d);
  const int64_t cols = static_cast<int64_t>(group) * P.n_groups, values = static_cast<int64_t>(g.O) * P.cols;
  const int steps = (P.K + BK - 1) / BK;
  const TilePlan plan = plan_tiles(g.O, &cols, &steps, 1, 1, 1024, static_cast<double>(values), point ? kFilterWordsCost : kFilterTapsCost);
  const TileKind &k = kTiles[plan.tile];
  P.kchunk = range_depth(g, reach, plan.S);
  const int S = std::max(1, (P.K + P.kchunk - 1) / P.kchunk);
  const int tm = (g.O + k.bm - 1) / k.bm, tn = static_cast<int>((cols + k.bn - 1) / k.bn);
  TS_REQUIRE(static_cast<int64_t>(tm) * tn * S < (1ll << 31) - 8, "conv: too many tiles");
  const bool direct = S == 1 && taps == 1;
  P.out = dw;
  P.z_stride = values;
  if (!direct) {
    P.out = static_cast<float *>(scratch_get(st, 2, static_cast<size_t>(S) * values * sizeof(float)));
    TS_REQUIRE(P.out, "conv bwd-filter: no scratch memory for the ranges' results");
    *ws_elems = S * values;
  }
  const mg::TileGrid tg{tm, tn, tm * tn * S};
  const unsigned grid = mg::grid_blocks(tm, tn, S);
  if (point)
    launch_tile<0>(P, plan.tile, tg, grid, st);
  else if (group == 16)
    launch_tile<16>(P, plan.tile, tg, grid, st);
  else if (group == 4)
    launch_tile<4>(P, plan.tile, tg, grid, st);
  else
    launch_tile<2>(P, plan.tile, tg, grid, st);
  if (taps == 1 && S > 1 && S < 8)   // (four lanes share an output's ranges in the other)
    gt::launch_fold(P.out, dw, values, S, st);
  else if (!direct)
    conv_fold_tap_major(P.out, dw, g.O, g.C, taps, S, st);
  return 0;
}

}  // namespace tsplit
