// Convolution forward and data gradient as implicit products on the tile kernel of gemm_tile.h.
//
//   forward        y[img,o,p]  : M = O, N = imgs * oH * oW, depth (c, tap)   A = filter [O][depth]
//   data gradient  dx[img,c,q] : M = C, N = imgs * H * W,   depth (o, tap)   A = filter re-laid [C][depth]
//
// B is gathered: row k of the operand is one tap of one channel at the tile's columns, 64 columns a load of 4 bytes a lane
// into LDS.  A lane's offset is fixed for the tile, what changes with k is wave-uniform and travels in the scalar offset; a
// tap in the padding is an out-of-range offset, which LDS receives as zero.  The depth is ordered in blocks of 8 channels of
// one tap, k = ((ch / 8) * taps + tap) * 8 + ch % 8 with channels padded to whole blocks: a wave's 8 rows of a 32-deep step
// are then one block, and the choice between a lane's offset and the padding's is made once for all of them.  In the
// filter's own order (ch, tap) it is made for every row, which costs vector instructions the products pay for (17x17 images,
// 1x7 filters, 256 -> 256: 128 us against 87 in blocks): only layers of few channels, where the padding would cost more, use
// that order.  Where a layer has one tap, no padding and planes of whole 16-byte words, B is loaded in 16-byte words like a
// dense operand.
//
// A strided data gradient splits into s * s phases of input positions, each a stride-1 problem over the taps that reach it
// (those without any are zeros).  For stride 2 a block computes the two phases that share a row of positions and writes them
// together: written one phase at a time every line of dx is written in parts (1x1 filters, 256 -> 512 at 56x56: 825 us).
#pragma once
#include <hip/hip_runtime.h>

#include "fastdiv.h"
#include "gemm_tile.h"

namespace tsplit {
namespace ct {

using gt::BK;
using gt::f32x4;
using gt::i32x4;
using mg::kOobOffset;

constexpr int kMaxPhases = 4;

// One stride phase (forward and stride-1 data gradients have one).
struct Phase {
  FastDiv plane, width;   // columns per image / per row
  FastDiv taps, kw;       // filter taps of the phase, and its taps per row
  int N, K;               // columns; depth
  int ph, pw;             // forward: padding.  Data gradient: the phase's own (see conv.hip)
  int bias;               // elements by which the gathered tensor's base is moved back so that no offset is negative
  int out_a0, out_b0;     // first output row / column of the phase
  int w_at;               // where the phase's filter begins in w
  int first_tile;         // tiles of the phases before it
  int kchunk;             // k range of one split (a multiple of 32)
};

struct Params {
  const float *src, *w;
  float *out;
  int64_t out_img_stride, z_stride;
  unsigned src_bytes;
  int img_stride, chan_stride, chans;   // elements per image / channel plane of src; its channels
  int src_h, src_w, s;
  int M, out_plane, out_h, out_w;
  int out_s;                     // an output position's step in the output plane (data gradient: the stride)
  FastDiv tm, tiles;             // M tiles; tiles of all phases (of all pairs)
  int phases;
  float *stats;
  const float *add;              // laid out as out, which it may be (a lane reads a value before it writes it)
  Phase phase[kMaxPhases];
};

// B, gathered.  BWD: element (k = (ch, u, v), position (r, c)) at [ch][r + ph - u][c + pw - v], else at
// [ch][r s - ph + u][c s - pw + v].  TAPS: a lane's taps as a bit mask of 32 or 64, 0: one tap, always inside.  BLOCKS: the
// depth in blocks of 8 channels of one tap, else (ch, tap).
template <int BN, int T, bool BWD, int TAPS, bool BLOCKS>
struct Gathered {
  static constexpr bool kDense = false;
  static constexpr int kFloats = BK * BN, H = BN / 64;
  static constexpr int kParts = TAPS && BLOCKS ? 4 : 1;   // in which a step's loads may be asked for: prepare() and part(0) to part(3), or load()
  using Mask = typename std::conditional<(TAPS > 32), uint64_t, uint32_t>::type;
  unsigned voff[H];
  Mask inside[H];
  i32x4 rsrc;
  // of the parameters, held in scalar registers: read from the argument buffer they cost a scalar load and its wait a step
  FastDiv taps, kw;
  int plane, chans, src_w, bias, wave, nowhere;
  __device__ __forceinline__ void init(const Params &p, const Phase &f, int n0) {
    taps = f.taps;
    kw = f.kw;
    plane = p.chan_stride * 4;
    chans = p.chans;
    src_w = p.src_w;
    bias = f.bias;
    wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    nowhere = static_cast<int>(p.src_bytes + 4u * f.bias);   // a scalar offset behind the end
    rsrc = gt::raw_buffer(p.src - f.bias, nowhere);
#pragma unroll
    for (int h = 0; h < H; ++h) {
      const int n = n0 + 64 * h + (threadIdx.x & 63);
      const bool ok = n < f.N;
      const uint32_t nn = ok ? n : 0, img = f.plane.div(nn), p0 = nn - img * f.plane.d, row = f.width.div(p0), col = p0 - row * f.width.d;
      const int r0 = BWD ? static_cast<int>(row) + f.ph : static_cast<int>(row) * p.s - f.ph;
      const int c0 = BWD ? static_cast<int>(col) + f.pw : static_cast<int>(col) * p.s - f.pw;
      const int at = BWD ? r0 * p.src_w + c0 : r0 * p.src_w + c0 + f.bias;
      voff[h] = ok ? static_cast<unsigned>(static_cast<int>(img) * p.img_stride + at) * 4u : kOobOffset;
      Mask m = 0;
      if (TAPS)
        for (int t = 0; t < static_cast<int>(f.taps.d); ++t) {
          const int u = f.kw.div(t), v = t - u * f.kw.d;
          const int rr = BWD ? r0 - u : r0 + u, cc = BWD ? c0 - v : c0 + v;
          if (ok && static_cast<unsigned>(rr) < static_cast<unsigned>(p.src_h) && static_cast<unsigned>(cc) < static_cast<unsigned>(p.src_w))
            m |= static_cast<Mask>(1) << t;
        }
      inside[h] = m;
    }
  }
  // displacement of a tap, in elements
  __device__ __forceinline__ int shift(int tap) const {
    const int u = kw.div(tap), v = tap - u * kw.d, at = u * src_w + v;
    return BWD ? bias - at : at;
  }
  unsigned at[H], to;
  int soff, have;
  __device__ __forceinline__ void prepare(int k0, int kend, unsigned lds) {
    to = lds + 8 * wave * BN * 4;
    {
      const int k = k0 + 8 * wave;
      int ch = k;
      if (TAPS) {
        const int block = k >> 3, cb = taps.div(block), tap = block - cb * taps.d;
        ch = 8 * cb;
        soff = ch * plane + shift(tap) * 4;
#pragma unroll
        for (int h = 0; h < H; ++h) at[h] = inside[h] >> tap & 1 ? voff[h] : kOobOffset;
      } else {
        soff = k * plane;
#pragma unroll
        for (int h = 0; h < H; ++h) at[h] = voff[h];
      }
      have = k < kend ? chans - ch : 0;   // channels of this block
    }
  }
  __device__ __forceinline__ void part(int i) const {
#pragma unroll
    for (int r = 2 * i; r < 2 * i + 2; ++r)
#pragma unroll
      for (int h = 0; h < H; ++h) gt::load_word_to_lds(rsrc, at[h], r < have ? soff + r * plane : nowhere, to + (r * BN + 64 * h) * 4);
  }
  __device__ __forceinline__ void load(int k0, int kend, unsigned lds) {
    if constexpr (BLOCKS || !TAPS) {
      prepare(k0, kend, lds);
#pragma unroll
      for (int i = 0; i < 4; ++i) part(i);
    } else {
      lds += 8 * wave * BN * 4;
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        const int k = k0 + 8 * wave + r, ch = taps.div(k), tap = k - ch * taps.d;
        const int soff = k < kend ? ch * plane + shift(tap) * 4 : nowhere;
#pragma unroll
        for (int h = 0; h < H; ++h)
          gt::load_word_to_lds(rsrc, inside[h] >> tap & 1 ? voff[h] : kOobOffset, soff, lds + (r * BN + 64 * h) * 4);
      }
    }
  }
  __device__ __forceinline__ bool cut(int, int) const { return false; }
  __device__ __forceinline__ void clear_tail(int, int, float *) const {}
  static __device__ __forceinline__ void frag(const float *lds, int mn0, int h, int lane, float (&v)[T][4]) {
    gt::MnContig<BN, T>::frag(lds, mn0, h, lane, v);
  }
};

// B of a layer with one tap, no padding, stride 1 and planes of whole 16-byte words: four columns of one image are one word.
template <int BN, int T>
struct Pointwise {
  static constexpr bool kDense = false;
  static constexpr int kParts = 1;
  static constexpr int kFloats = BK * BN;
  static constexpr int kLoads = BN / 32, kWords = BN / 4, kRows = 64 / kWords;
  unsigned voff;
  i32x4 rsrc;
  int wave, row_bytes, row;
  __device__ __forceinline__ void init(const Params &p, const Phase &f, int n0) {
    const int lane = threadIdx.x & 63;
    wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    rsrc = gt::raw_buffer(p.src, p.src_bytes);
    row_bytes = p.chan_stride * 4;
    row = lane / kWords;
    const int n = n0 + 4 * (lane % kWords);
    const uint32_t nn = n < f.N ? n : 0, img = f.plane.div(nn);
    voff = n < f.N ? (img * p.img_stride + row * p.chan_stride + nn - img * f.plane.d) * 4u : kOobOffset;
  }
  __device__ __forceinline__ void load(int k0, int kend, unsigned lds) const {
    lds += wave * kLoads * 1024;
    const int k1 = k0 + wave * kLoads * kRows;
    if (k0 + BK <= kend) {
#pragma unroll
      for (int s = 0; s < kLoads; ++s) gt::load_to_lds(rsrc, voff, (k1 + s * kRows) * row_bytes, lds + s * 1024);
    } else {   // channels past the last one are the next image's, and of large planes beyond 32-bit offsets
#pragma unroll
      for (int s = 0; s < kLoads; ++s) {
        const int k = k1 + s * kRows;
        gt::load_to_lds(rsrc, k + row < kend ? voff : kOobOffset, k < kend ? k * row_bytes : 0, lds + s * 1024);
      }
    }
  }
  __device__ __forceinline__ bool cut(int, int) const { return false; }
  __device__ __forceinline__ void clear_tail(int, int, float *) const {}
  static __device__ __forceinline__ void frag(const float *lds, int mn0, int h, int lane, float (&v)[T][4]) {
    gt::MnContig<BN, T>::frag(lds, mn0, h, lane, v);
  }
};

// How a pass reads B: words of a dense operand, one tap, up to 32 / 64 taps in blocks of 8 channels, up to 64 in the filter's order
enum Gather { kWords, kOneTap, kBlocks32, kBlocks64, kTaps64 };

// ACROSS: A is the filter in memory, [depth][M] (data gradient of one tap); else [M][depth]
template <int TM, int TN, bool BWD, int GATHER, bool ACROSS, bool PAIR = false>
struct Pass {
  static constexpr int BM = 32 * TM, BN = 32 * TN;
  using BL = typename std::conditional<GATHER == kWords, Pointwise<BN, TN>,
                                       Gathered<BN, TN, BWD, GATHER == kOneTap ? 0 : GATHER == kBlocks32 ? 32 : 64, GATHER != kTaps64>>::type;
  using AL = typename std::conditional<ACROSS, gt::MnContig<BM, TM>, gt::KContig<BM, TM, false>>::type;
  // (a pair's 128 x 128 tiles have no registers left for loads between products)
  using C = gt::Core<TM, TN, 2, 2, AL, BL, (BL::kParts > 1 && !(PAIR && TM * TN == 16))>;

  static __device__ __forceinline__ void run(const Params &P, const Phase &F, int m0, int n0, int z, float *lds, f32x4 (&acc)[TM][TN]) {
    AL la;
    BL lb;
    la.init(mg::DenseParams{P.w + F.w_at, ACROSS ? P.M : F.K, P.M, F.K}, m0);
    lb.init(P, F, n0);
    const int kbegin = z * F.kchunk;
    C::run(la, lb, kbegin, min(F.K, kbegin + F.kchunk), lds, acc);
  }
};

// the block's split, phase (or pair of phases) and tile; false for the blocks that only pad the grid
__device__ __forceinline__ bool place(const Params &P, int total, int step, int &z, int &ip, int &tile_m, int &tile_n) {
  const int logical = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  if (logical >= total) return false;
  z = P.tiles.div(logical);
  int tile = logical - z * P.tiles.d;
  ip = 0;
  while (ip + step < P.phases && tile >= P.phase[ip + step].first_tile) ip += step;
  tile -= P.phase[ip].first_tile;
  tile_n = P.tm.div(tile);
  tile_m = tile - tile_n * P.tm.d;
  return true;
}

// Sums over groups of 16 lanes: lane bit BIT decides which half of N registers a lane keeps (both add what the partner held
// of that half); with one register left the partners hold the same sum.
template <int N, int BIT = 8>
__device__ __forceinline__ void halve(float *sum, float *sq, int lane) {
  constexpr int H = N > 1 ? N / 2 : 1;
  const bool up = N > 1 && (lane & BIT);
#pragma unroll
  for (int i = 0; i < H; ++i) {
    const float keep = up ? sum[i + N - H] : sum[i], send = up ? sum[i] : sum[i + N - H];
    const float keep2 = up ? sq[i + N - H] : sq[i], send2 = up ? sq[i] : sq[i + N - H];
    sum[i] = keep + __shfl_xor(send, BIT, 64);
    sq[i] = keep2 + __shfl_xor(send2, BIT, 64);
  }
  if constexpr (BIT > 1) halve<H, BIT / 2>(sum, sq, lane);
}

// Stores a tile of a one-tap data gradient of stride 2: position (r, c) of a column covers the 2 x 2 input positions from (2 r, 2 c)
// on; the value belongs to the first of them, no tap reaches the others.  Both rows of positions leave from here, in words of two
// columns, so that dx is written once and in whole rows (a phase at a time, 64 x 512 x 28 x 28 into 64 x 256 x 56 x 56: 300 us).
// ADD: `from` holds what is added, at every position.
template <int TM, int TN, bool ADD, class StepRow>
__device__ __forceinline__ void spread(const Params &P, const Phase &F, const f32x4 (&acc)[TM][TN], __amdgpu_buffer_rsrc_t to,
                                       __amdgpu_buffer_rsrc_t from, int m, int n, int img0, int lane_row, StepRow step_row) {
  const int plane_bytes = P.out_plane * 4, out_h = P.out_h;
  const unsigned at = static_cast<unsigned>(lane_row) * plane_bytes, down = static_cast<unsigned>(P.out_w) * 4u;
  unsigned off[TN];
  bool below[TN], beside[TN], together = n + TN <= F.N;
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const uint32_t nn = n + j < F.N ? n + j : 0, img = F.plane.div(nn), p = nn - img * F.plane.d, r = F.width.div(p), c = p - r * F.width.d;
    off[j] = n + j < F.N ? at + ((static_cast<int>(img) - img0) * static_cast<unsigned>(P.out_img_stride) + 2 * r * P.out_w + 2 * c) * 4u : kOobOffset;
    below[j] = 2 * static_cast<int>(r) + 1 < out_h;
    beside[j] = 2 * static_cast<int>(c) + 1 < P.out_w;
    if (j == 0) together = together && 2 * (static_cast<int>(c) + TN) <= P.out_w;
  }
  const bool words = __all(together || n >= F.N), ragged = m + 16 * TM > P.M;
  if (words) {
#pragma unroll
    for (int tm = 0; tm < TM; ++tm) {
      float v[4][TN / 2][2][4];   // of four rows at a time: a pair of columns' words, this row of positions' and the next one's
      auto place = [&](int e, int j, int below_it, unsigned &o, int &soff) {
        const int row = step_row(tm, e);
        const bool past = ragged && m + row + lane_row >= P.M;
        soff = past ? 0 : row * plane_bytes;   // (past M the product may leave 32 bits)
        o = past || (below_it && !below[j]) ? kOobOffset : off[j] + (below_it ? down : 0u);
      };
      unsigned o;
      int soff;
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int j = 0; j < TN; j += 2)
#pragma unroll
          for (int u = 0; u < 2; ++u) {
            float(&w)[4] = v[e][j / 2][u];
            place(e, j, u, o, soff);
            if constexpr (ADD) gt::load_words<4>(from, o, soff, w);
          }
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int j = 0; j < TN; j += 2)
#pragma unroll
          for (int u = 0; u < 2; ++u) {
            float(&w)[4] = v[e][j / 2][u];
            const float made[4] = {u == 0 ? acc[tm][j][e] : 0.f, 0.f, u == 0 ? acc[tm][j + 1][e] : 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < 4; ++i) w[i] = ADD ? w[i] + made[i] : made[i];   // (zeros too: -0 + 0 is 0)
            place(e, j, u, o, soff);
            gt::store_words<4>(to, o, soff, w);
          }
    }
    return;
  }
#pragma unroll
  for (int tm = 0; tm < TM; ++tm)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int row = step_row(tm, e);
      const bool past = ragged && m + row + lane_row >= P.M;
      const int soff = past ? 0 : row * plane_bytes;   // (past M the product may leave 32 bits)
      unsigned o[TN][4];
      float v[TN][4];
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const bool none = past || off[j] == kOobOffset;
        o[j][0] = none ? kOobOffset : off[j];
        o[j][1] = none || !beside[j] ? kOobOffset : off[j] + 4u;
        o[j][2] = none || !below[j] ? kOobOffset : off[j] + down;
        o[j][3] = none || !below[j] || !beside[j] ? kOobOffset : off[j] + down + 4u;
        if constexpr (ADD) {
#pragma unroll
          for (int i = 0; i < 4; ++i) v[j][i] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(from, o[j][i] + soff, 0, 0));
        }
      }
#pragma unroll
      for (int j = 0; j < TN; ++j) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float made = i == 0 ? acc[tm][j][e] : 0.f;
          __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(ADD ? v[j][i] + made : made), to, o[j][i] + soff, 0, 0);
        }
      }
    }
}

// STATS: each wave leaves the sums and sums of squares of its rows over its 16 TN columns, for column group
// (first column) / (16 TN) at stats[(group * M + row) * 2].
// ADD: the result and what P.add holds in one store.  A gradient with several terms was a pass of its own that read two arrays
// and wrote a third (64 x 256 x 56 x 56: 95 us); here the other term is read once, between the products and the store.
template <int TM, int TN, bool BWD, int GATHER, bool ACROSS, bool STATS, bool ADD>
__global__ __launch_bounds__(gt::kThreads, 2) void conv_tile_kernel(Params P, int total) {
  using X = Pass<TM, TN, BWD, GATHER, ACROSS>;
  using C = typename X::C;
  __shared__ __attribute__((aligned(1024))) float lds[C::kLdsFloats];
  int z, ip, tile_m, tile_n;
  if (!place(P, total, 1, z, ip, tile_m, tile_n)) return;
  const Phase &F = P.phase[ip];
  const int m0 = tile_m * X::BM, n0 = tile_n * X::BN;
  f32x4 acc[TM][TN];
  X::run(P, F, m0, n0, z, lds, acc);

  // the wave's first row; offsets count from the image its tile begins in (a tile's images lie within 2 GiB)
  const int lane = threadIdx.x & 63, m = m0 + C::wave_m0(), n = n0 + C::wave_n0() + TN * (lane & 15);
  const int img0 = F.plane.div(n0), plane_bytes = P.out_plane * 4;
  const int64_t tile_at = img0 * P.out_img_stride + static_cast<int64_t>(m) * P.out_plane;
  const __amdgpu_buffer_rsrc_t to = gt::output_buffer(P.out + z * P.z_stride + tile_at, 0x7fffffffll);
  const __amdgpu_buffer_rsrc_t from = ADD ? gt::output_buffer(const_cast<float *>(P.add) + tile_at, 0x7fffffffll) : to;
  if constexpr (BWD && ACROSS)
    if (P.out_s == 2)
      return spread<TM, TN, ADD>(P, F, acc, to, from, m, n, img0, C::lane_row(), [](int tm, int e) { return C::step_row(tm, e); });
  // where the lane's TN columns go: together if they lie in one image of a plane without gaps
  const unsigned at = static_cast<unsigned>(C::lane_row()) * plane_bytes;
  unsigned off[TN];
  bool together = P.out_s == 1 && n + TN <= F.N;
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const uint32_t nn = n + j < F.N ? n + j : 0, img = F.plane.div(nn), p = nn - img * F.plane.d;
    unsigned o = (static_cast<int>(img) - img0) * static_cast<unsigned>(P.out_img_stride) + p;
    if (P.out_s != 1) {
      const uint32_t r = F.width.div(p), c = p - r * F.width.d;
      o += (F.out_a0 + P.out_s * r) * P.out_w + F.out_b0 + P.out_s * c - p;
    }
    off[j] = n + j < F.N ? at + o * 4u : kOobOffset;
    if (j == 0) together = together && p + TN <= F.plane.d;
  }
  const bool words = __all(together || n >= F.N);
  auto store = [&](auto ragged, auto in_words) {   // ragged: the wave's rows run past M
    constexpr bool kRagged = decltype(ragged)::value;
    // ADD: all of it is asked for before the first store, which the compiler would keep behind the loads above it alone
    // (1024 channels of 17 x 17: one at a time 50-63 us, without ADD 29)
    if constexpr (ADD) {
      float more[TM][4][TN];
#pragma unroll
      for (int tm = 0; tm < TM; ++tm)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int row = C::step_row(tm, e);
          const bool past = kRagged && m + row + C::lane_row() >= P.M;
          const int soff = past ? 0 : row * plane_bytes;
          if constexpr (decltype(in_words)::value) {
            gt::load_words<TN>(from, past ? kOobOffset : off[0], soff, more[tm][e]);
          } else {
#pragma unroll
            for (int j = 0; j < TN; ++j) more[tm][e][j] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(from, (past ? kOobOffset : off[j]) + soff, 0, 0));
          }
        }
#pragma unroll
      for (int tm = 0; tm < TM; ++tm)
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int j = 0; j < TN; ++j) acc[tm][j][e] = more[tm][e][j] + acc[tm][j][e];
    }
#pragma unroll
    for (int tm = 0; tm < TM; ++tm)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int row = C::step_row(tm, e);
        const bool past = kRagged && m + row + C::lane_row() >= P.M;
        const int soff = past ? 0 : row * plane_bytes;   // (past M the product may leave 32 bits)
        if constexpr (decltype(in_words)::value) {
          float v[TN];
#pragma unroll
          for (int j = 0; j < TN; ++j) v[j] = acc[tm][j][e];
          gt::store_words<TN>(to, past ? kOobOffset : off[0], soff, v);
        } else {
#pragma unroll
          for (int j = 0; j < TN; ++j)
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(acc[tm][j][e]), to, (past ? kOobOffset : off[j]) + (kRagged ? soff : 0),
                                                  kRagged ? 0 : soff, 0);
        }
      }
  };
  if (m + 16 * TM > P.M)
    store(std::true_type{}, std::false_type{});
  else if (words)
    store(std::false_type{}, std::true_type{});
  else
    store(std::false_type{}, std::false_type{});
  if constexpr (STATS) {
    static_assert(!ACROSS, "rows in order");
    // lane c of 16 (TM = 2: the pair c / 2) ends with row register c (tm = c / 4, e = c % 4) summed over the 16 lanes
    constexpr int R = 4 * TM;
    float sum[R], sq[R];
#pragma unroll
    for (int tm = 0; tm < TM; ++tm)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float a = 0.f, b = 0.f;
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          a += acc[tm][j][e];
          b += acc[tm][j][e] * acc[tm][j][e];
        }
        sum[4 * tm + e] = a;
        sq[4 * tm + e] = b;
      }
    halve<R>(sum, sq, lane);
    const int reg = TM == 4 ? lane & 15 : lane >> 1 & 7;   // the register this lane ended with
    const int row = m + C::lane_row() + 16 * (reg >> 2) + (reg & 3), col0 = n0 + C::wave_n0();
    if ((TM == 4 || !(lane & 1)) && row < P.M && col0 < F.N) {
      float *dst = P.stats + (static_cast<int64_t>(col0 / (16 * TN)) * P.M + row) * 2;
      dst[0] = sum[0];
      dst[1] = sq[0];
    }
  }
}

// Data gradient of stride 2: phases 2 q and 2 q + 1 are the even and the odd columns of the same rows of positions.
template <int TM, int TN>
__global__ __launch_bounds__(gt::kThreads, 2) void conv_tile_pair_kernel(Params P, int total) {
  using X = Pass<TM, TN, true, kBlocks32, false, true>;
  using C = typename X::C;
  __shared__ __attribute__((aligned(1024))) float lds[C::kLdsFloats];
  int z, ip, tile_m, tile_n;
  if (!place(P, total, 2, z, ip, tile_m, tile_n)) return;
  const Phase &F = P.phase[ip];
  const int m0 = tile_m * X::BM, n0 = tile_n * X::BN;
  f32x4 even[TM][TN], odd[TM][TN];
  X::run(P, F, m0, n0, z, lds, even);
  __syncthreads();   // the second product's first step is loaded over the first one's last
  X::run(P, P.phase[ip + 1], m0, n0, z, lds, odd);

  const int lane = threadIdx.x & 63, m = m0 + C::wave_m0(), n = n0 + C::wave_n0() + TN * (lane & 15);
  const int img0 = F.plane.div(n0), plane_bytes = P.out_plane * 4;
  const __amdgpu_buffer_rsrc_t to =
      gt::output_buffer(P.out + z * P.z_stride + img0 * P.out_img_stride + static_cast<int64_t>(m) * P.out_plane, 0x7fffffffll);
  const unsigned lane_at = static_cast<unsigned>(C::lane_row()) * plane_bytes;
  unsigned off[TN], off_odd[TN];
  bool together = n + TN <= F.N;
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const uint32_t nn = n + j < F.N ? n + j : 0, img = F.plane.div(nn), p = nn - img * F.plane.d, r = F.width.div(p), c = p - r * F.width.d;
    const unsigned o = lane_at + ((static_cast<int>(img) - img0) * static_cast<unsigned>(P.out_img_stride) + (F.out_a0 + 2 * r) * P.out_w + 2 * c) * 4u;
    off[j] = n + j < F.N ? o : kOobOffset;
    off_odd[j] = n + j < F.N && 2 * static_cast<int>(c) + 1 < P.out_w ? o + 4u : kOobOffset;
    if (j == 0) together = together && 2 * (static_cast<int>(c) + TN) <= P.out_w;   // all of them in one row
  }
  const bool words = __all(together || n >= F.N), ragged = m + 16 * TM > P.M;
#pragma unroll
  for (int tm = 0; tm < TM; ++tm)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int row = C::step_row(tm, e);
      const bool past = ragged && m + row + C::lane_row() >= P.M;
      const int soff = past ? 0 : row * plane_bytes;   // (past M the product may leave 32 bits)
#pragma unroll
      for (int j = 0; j < TN; j += 2) {
        if (words) {
          const float v[4] = {even[tm][j][e], odd[tm][j][e], even[tm][j + 1][e], odd[tm][j + 1][e]};
          gt::store_words<4>(to, past ? kOobOffset : off[j], soff, v);
        } else {
#pragma unroll
          for (int i = j; i < j + 2; ++i) {
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(even[tm][i][e]), to, (past ? kOobOffset : off[i]) + soff, 0, 0);
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(odd[tm][i][e]), to, (past ? kOobOffset : off_odd[i]) + soff, 0, 0);
          }
        }
      }
    }
}

// The filter in the order of the depth, for every phase: w[w_at + row * K + ((ch / 8) * taps + tap) * 8 + ch % 8], zeros for the
// channels that pad the last block (or, `plain`, w[... + ch * taps + tap]).  Tap (u, v) of the phase is the filter's tap
// (a + s u, b + s v); bwd: rows are C and channels O, else the other way.
struct RelayPhase {
  int w_at, K, a, b;
  FastDiv taps, kw, k;
};
struct Relay {
  const float *w;
  float *out;
  int rows, chans, w_row, w_chan, f_w, s, phases, total;
  bool plain;
  RelayPhase phase[kMaxPhases];
};
static __global__ __launch_bounds__(256) void conv_relay_kernel(Relay R) {
  const int idx = blockIdx.x * 256 + threadIdx.x;
  if (idx >= R.total) return;
  int ip = 0;
  while (ip + 1 < R.phases && idx >= R.phase[ip + 1].w_at) ++ip;
  const RelayPhase &F = R.phase[ip];
  const int i = idx - F.w_at, row = F.k.div(i), k = i - row * F.K;
  int ch, tap;
  if (R.plain) {
    ch = F.taps.div(k);
    tap = k - ch * F.taps.d;
  } else {
    const int block = k >> 3, cb = F.taps.div(block);
    tap = block - cb * F.taps.d;
    ch = 8 * cb + (k & 7);
  }
  const int u = F.kw.div(tap), v = tap - u * F.kw.d;
  R.out[idx] = ch < R.chans ? R.w[row * R.w_row + ch * R.w_chan + (F.a + R.s * u) * R.f_w + F.b + R.s * v] : 0.f;
}

// The same for a filter of one phase with all its taps, kRelayRows rows x kRelayChans channels a block, through LDS: memory
// holds a row's channels (forward) or a channel's rows (data gradient, `across`) side by side, and runs of either are read, and of the
// output's rows written, whole.  One thread a value fetched every value by itself: 512 x 512 x 9 behind other layers 14.5 us, 1.3 TB/s
// (five such layers both ways: 2.117 -> 2.092 ms a step).
constexpr int kRelayRows = 8, kRelayChans = 32;
static __global__ __launch_bounds__(256) void conv_relay_tiles_kernel(const float *__restrict__ w, float *__restrict__ out, int rows, int chans, int padded,
                                                                      FastDiv taps, int64_t w_row, int64_t w_chan, FastDiv tiles) {
  extern __shared__ float lds[];   // [row][channel][tap], a channel to spare a row
  const int n_taps = taps.d, pitch = (kRelayChans + 1) * n_taps;
  const uint32_t tr = tiles.div(blockIdx.x);
  const int r0 = tr * kRelayRows, c0 = (blockIdx.x - tr * tiles.d) * kRelayChans;
  const bool across = w_row < w_chan;   // a channel's rows lie side by side
  for (int e = threadIdx.x; e < kRelayRows * kRelayChans * n_taps; e += 256) {
    const int i = taps.div(e), tap = e - i * n_taps;
    const int r = across ? i % kRelayRows : i / kRelayChans, c = across ? i / kRelayRows : i % kRelayChans;
    lds[r * pitch + c * n_taps + tap] = r0 + r < rows && c0 + c < chans ? w[(r0 + r) * w_row + (c0 + c) * w_chan + tap] : 0.f;
  }
  __syncthreads();
  const int here = min(kRelayChans, padded - c0) * n_taps;   // values of a row, side by side in the output
  for (int e = threadIdx.x; e < kRelayRows * kRelayChans * n_taps; e += 256) {
    const int i = taps.div(e >> 3), tap = (e >> 3) - i * n_taps;   // i: block of 8 channels, of row i / 4
    const int r = i / (kRelayChans / 8), b = i % (kRelayChans / 8), at = (b * n_taps + tap) * 8 + (e & 7);
    if (r0 + r < rows && at < here)
      out[(static_cast<int64_t>(r0 + r) * padded + c0) * n_taps + at] = lds[r * pitch + (8 * b + (e & 7)) * n_taps + tap];
  }
}

}  // namespace ct
}  // namespace tsplit
