// Convolution filter gradient as a product on the tile kernel of gemm_tile.h: dw[o, (tap, c)] = sum over positions of
// dy[o, position] x[c, position shifted by the tap].
//
//   M = O, N = taps x C (a tap's channels in whole groups of 16, 4 or 2), depth = images x positions, an image's positions padded to
//   a multiple of 4.  Both operands have the depth contiguous.
//
// Groups of 16 test a position against the image's edge once for eight loads, groups of 4 or 2 once for two loads or each one; but
// 3 channels padded to 16 are five times the products and loads (64 x 3 x 224 x 224, 64 filters of 7x7, stride 2: 770 us in groups of
// 16, 259 in groups of 4).
//
// A step's position is worked out once a lane (from the step's before it; by division only where an image begins, which as much
// as doubles what a 64 x 64 tile spends on it) and serves every row the lane loads: rows are
// a wave-uniform distance apart, which travels in the scalar offset.  That needs an LDS layout in which a lane's place along the
// depth is the same in all of them, so rows are kept apart by padding (and, 16 bytes a lane, by an exchange of words inside the
// 8 rows of a load) instead of the exchange by row number of gt::KContig.
//
// dy is loaded in 16-byte words; where an image's positions are not a multiple of 4 its last word ends with the next row's first
// values, which are cleared in LDS.  x is loaded the same way for filters of one tap at stride 1 without padding, else value
// by value, positions outside the image as zeros.  Rows past the last channel hold values of the next image: they belong to
// rows or columns of dw that do not exist.
//
// What bounds it is the matrix pipe where the tiles fill the chip (1x1 layers: 64 x 512 x 28 x 28 -> 128 in 62 us, 106 TFLOP/s) and
// the gathered loads, 4 bytes a lane, elsewhere.  Against 16-deep steps whose operands went through vector registers: 1x1 layers of
// ResNet-50 66, 62, 76, 76 us (were 90, 87, 90, 90), its first layer 259 (411), 1x7 of 256 -> 256 at 17x17 93 (96), 3x3 of 512 -> 512 at
// 4x4 71 (79), 3x3 stride 2 of 96 -> 200 channels 17 (32); 3x3 of 512 -> 512 at 28x28, 18 images, 570 (549), where the loads count
// most.  With the gathered loads between the products (gt::Core) the last two take 14 and 525.
#pragma once
#include <hip/hip_runtime.h>

#include "fastdiv.h"
#include "gemm_tile.h"

namespace tsplit {
namespace wt {

using gt::BK;
using gt::f32x4;
using gt::i32x4;
using mg::kOobOffset;

struct Params {
  const float *dy, *x;
  float *out;
  int64_t z_stride;
  int64_t dy_bytes, x_bytes;
  int M, C, cols;                // O; channels of x; columns of one row of the output, taps * C
  int K, kchunk;                 // depth; one range of it (a multiple of 32)
  FastDiv image, width, groups;  // padded positions of an image; positions in a row; groups of channels of a tap
  FastDiv kw;
  int n_groups;                  // of N
  int plane, dy_img;             // positions of an image; values of an image of dy
  int x_plane, x_img, x_h, x_w;
  int ph, pw, s;
};

// a tensor from image `img` on
__device__ __forceinline__ i32x4 from_image(const float *p, int64_t bytes, int img, int img_values) {
  const int64_t at = static_cast<int64_t>(img) * img_values;
  return gt::raw_buffer(p + at, bytes - 4 * at);
}

// MN rows of `plane` values, 16 bytes a lane.  LDS: 8 rows of a load in 256 floats and 16 to spare, word q of row r at
// q ^ (r / 2 % 4): a product tile's 16 rows then start on 16 different bank groups.
template <int MN, int T>
struct Words {
  static constexpr bool kDense = false, kDealt = false;
  static constexpr int kParts = 1;
  static constexpr int kGroup = 272, kLoads = MN / 32, kFloats = MN / 8 * kGroup;
  i32x4 rsrc;
  FastDiv image;
  int wave, img0, img_values, row_bytes, group_at, plane;
  unsigned lane_at, at;
  int pos;   // this lane's position in its image, `at` its byte offset
  __device__ __forceinline__ void init(const float *p, int64_t bytes, const FastDiv &padded, int positions, int values, int row0, int first_image,
                                       int kbegin) {
    const int lane = threadIdx.x & 63;
    wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    rsrc = from_image(p, bytes, first_image, values);
    image = padded;
    img0 = first_image;
    img_values = values;
    plane = positions;
    row_bytes = positions * 4;
    group_at = (row0 + wave * kLoads * 8) * row_bytes;
    lane_at = static_cast<unsigned>(lane >> 3) * row_bytes;
    place(kbegin + 4 * word());
  }
  __device__ __forceinline__ void place(int k) {
    const int img = image.div(k);
    pos = k - img * image.d;
    at = lane_at + static_cast<unsigned>((img - img0) * img_values + pos) * 4u;
  }
  static __device__ __forceinline__ int word() { return (threadIdx.x & 7) ^ (threadIdx.x >> 4 & 3); }
  // steps come in order
  __device__ __forceinline__ void load(int k0, int kend, unsigned lds) {
    const unsigned from = k0 + 4 * word() < kend ? at : kOobOffset;
    lds += wave * kLoads * kGroup * 4;
#pragma unroll
    for (int s = 0; s < kLoads; ++s) gt::load_to_lds(rsrc, from, group_at + 8 * s * row_bytes, lds + s * kGroup * 4);
    pos += BK;
    at += 4 * BK;
    if (pos >= static_cast<int>(image.d)) place(k0 + BK + 4 * word());
  }
  // the step holds an image's last word, and that word runs past the image
  __device__ __forceinline__ bool cut(int k0, int) const {
    return (plane & 3) != 0 && k0 - static_cast<int>(image.div(k0) * image.d) + BK >= static_cast<int>(image.d);
  }
  __device__ __forceinline__ void clear_tail(int k0, int, float *lds) const {
    const int k = k0 + 4 * word(), p = k - static_cast<int>(image.div(k) * image.d), keep = plane - p;
    if (keep < 4) {
      float *at = lds + wave * kLoads * kGroup + 4 * (threadIdx.x & 63);
#pragma unroll
      for (int s = 0; s < kLoads; ++s)
        for (int i = keep; i < 4; ++i) at[s * kGroup + i] = 0.f;
    }
  }
  static __device__ __forceinline__ void frag(const float *lds, int mn0, int h, int lane, float (&v)[T][4]) {
#pragma unroll
    for (int t = 0; t < T; ++t) {
      const int row = mn0 + 16 * t + (lane & 15);
      const f32x4 q = *reinterpret_cast<const f32x4 *>(lds + (row >> 3) * kGroup + (row & 7) * 32 + 4 * ((4 * h + (lane >> 4)) ^ (row >> 1 & 3)));
#pragma unroll
      for (int i = 0; i < 4; ++i) v[t][i] = q[i];
    }
  }
};

// BN columns of x, in groups of G channels of one tap, 4 bytes a lane.  LDS: two rows of a load in 64 floats and 4 to spare.
template <int BN, int T, int G>
struct Taps {
  static constexpr bool kDense = false;
  static constexpr int kParts = 4;
  static constexpr int kPair = 68, kGroups = BN / 4 / G, kFloats = BN / 2 * kPair;   // a wave's groups
  i32x4 rsrc;
  FastDiv image, width;
  int wave, img0, img_values, plane, x_plane, x_h, x_w, s;
  int down[kGroups], right[kGroups], shift[kGroups], chan_at[kGroups];
  // this lane's position in its image; the input row and column its tap (0, 0) reads before padding, their byte offset
  int pos, row, col;
  unsigned at;
  int row_step, col_step, at_step, col_end, at_wrap;   // what 32 positions on change; the end of a row of positions
  __device__ __forceinline__ void init(const Params &p, int n0, int first_image, int kbegin) {
    wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    rsrc = from_image(p.x, p.x_bytes, first_image, p.x_img);
    image = p.image;
    width = p.width;
    img0 = first_image;
    img_values = p.x_img;
    plane = p.plane;
    x_plane = p.x_plane;
    x_h = p.x_h;
    x_w = p.x_w;
    s = p.s;
#pragma unroll
    for (int g = 0; g < kGroups; ++g) {
      const int ng = min(n0 / G + wave * kGroups + g, p.n_groups - 1);   // groups past the last: its values once more, never stored
      const int tap = p.groups.div(ng), cg = ng - tap * p.groups.d, u = p.kw.div(tap), v = tap - u * p.kw.d;
      down[g] = __builtin_amdgcn_readfirstlane(u - p.ph);
      right[g] = __builtin_amdgcn_readfirstlane(v - p.pw);
      shift[g] = (down[g] * x_w + right[g]) * 4;
      chan_at[g] = __builtin_amdgcn_readfirstlane(G * cg * p.x_plane * 4);
    }
    const int rows = width.div(BK), cols = BK - rows * width.d;
    row_step = rows * s;
    col_step = cols * s;
    at_step = (row_step * x_w + col_step) * 4;
    col_end = width.d * s;
    at_wrap = (s * x_w - col_end) * 4;
    place(kbegin + (threadIdx.x & 31));
  }
  __device__ __forceinline__ void place(int k) {
    const int img = image.div(k);
    pos = k - img * image.d;
    const int r = width.div(pos);
    row = r * s;
    col = (pos - r * static_cast<int>(width.d)) * s;
    at = static_cast<unsigned>((img - img0) * img_values + static_cast<int>(threadIdx.x >> 5 & 1) * x_plane + row * x_w + col) * 4u;
  }
  // steps come in order
  unsigned from[kGroups], to;
  __device__ __forceinline__ void prepare(int k0, int kend, unsigned lds) {
    const bool ok = k0 + static_cast<int>(threadIdx.x & 31) < kend && pos < plane;
    to = lds + wave * kGroups * (G / 2) * kPair * 4;
#pragma unroll
    for (int g = 0; g < kGroups; ++g) {
      const bool in = ok && static_cast<unsigned>(row + down[g]) < static_cast<unsigned>(x_h) &&
                      static_cast<unsigned>(col + right[g]) < static_cast<unsigned>(x_w);
      from[g] = in ? at + shift[g] : kOobOffset;
    }
    pos += BK;
    row += row_step;
    col += col_step;
    at += at_step;
    if (col >= col_end) {
      col -= col_end;
      row += s;
      at += at_wrap;
    }
    if (pos >= static_cast<int>(image.d)) place(k0 + BK + (threadIdx.x & 31));
  }
  __device__ __forceinline__ void part(int i) const {
    constexpr int kLoads = kGroups * (G / 2);
#pragma unroll
    for (int l = kLoads / 4 * i; l < kLoads / 4 * (i + 1); ++l)
      gt::load_word_to_lds(rsrc, from[l / (G / 2)], chan_at[l / (G / 2)] + 2 * (l % (G / 2)) * x_plane * 4, to + l * kPair * 4);
  }
  __device__ __forceinline__ void load(int k0, int kend, unsigned lds) {
    prepare(k0, kend, lds);
#pragma unroll
    for (int i = 0; i < 4; ++i) part(i);
  }
  __device__ __forceinline__ bool cut(int, int) const { return false; }
  __device__ __forceinline__ void clear_tail(int, int, float *) const {}
  static __device__ __forceinline__ void frag(const float *lds, int mn0, int h, int lane, float (&v)[T][4]) {
#pragma unroll
    for (int t = 0; t < T; ++t) {
      const int row = mn0 + 16 * t + (lane & 15);
      const f32x4 q = *reinterpret_cast<const f32x4 *>(lds + (row >> 1) * kPair + (row & 1) * 32 + 4 * (4 * h + (lane >> 4)));
#pragma unroll
      for (int i = 0; i < 4; ++i) v[t][i] = q[i];
    }
  }
};

// G: channels of a group, the columns of one tap; 0: one tap, stride 1, no padding (the columns are the channels themselves)
template <int TM, int TN, int G>
__global__ __launch_bounds__(gt::kThreads, 2) void conv_wgrad_tile_kernel(Params P, mg::TileGrid tg) {
  constexpr int BM = 32 * TM, BN = 32 * TN, kGroup = G ? G : 16;
  using AL = Words<BM, TM>;
  using BL = typename std::conditional<G == 0, Words<BN, TN>, Taps<BN, TN, kGroup>>::type;
  using C = gt::Core<TM, TN, 2, 2, AL, BL>;
  __shared__ __attribute__((aligned(1024))) float lds[C::kLdsFloats];
  int z, tile_m, tile_n;
  if (!mg::block_tile(tg, z, tile_m, tile_n)) return;
  const int m0 = tile_m * BM, n0 = tile_n * BN, kbegin = z * P.kchunk, kend = min(P.K, kbegin + P.kchunk);
  const int first_image = P.image.div(kbegin);
  AL la;
  BL lb;
  la.init(P.dy, P.dy_bytes, P.image, P.plane, P.dy_img, m0, first_image, kbegin);
  if constexpr (G == 0)
    lb.init(P.x, P.x_bytes, P.image, P.plane, P.x_img, n0, first_image, kbegin);
  else
    lb.init(P, n0, first_image, kbegin);
  f32x4 acc[TM][TN];
  C::run(la, lb, kbegin, kend, lds, acc);

  float *out = P.out + z * P.z_stride;
  const int lane = threadIdx.x & 63, m = m0 + C::wave_m0() + C::lane_row();
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int n = n0 + C::wave_n0() + 16 * j + (lane & 15), ng = n / kGroup, tap = P.groups.div(ng), c = (ng - tap * P.groups.d) * kGroup + n % kGroup;
    if (ng >= P.n_groups || c >= P.C) continue;
    float *to = out + static_cast<int64_t>(m) * P.cols + tap * P.C + c;
#pragma unroll
    for (int tm = 0; tm < TM; ++tm)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (m + C::step_row(tm, e) < P.M) to[static_cast<int64_t>(C::step_row(tm, e)) * P.cols] = acc[tm][j][e];
  }
}

}  // namespace wt
}  // namespace tsplit
