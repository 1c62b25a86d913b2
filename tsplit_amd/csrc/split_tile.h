// The tile kernel of products of which one operand is small enough to be prepared: fp32 products taken as bf16 matrix products.
//
// An fp32 number is the exact sum of three bf16 numbers, a = a0 + a1 + a2: a0 = bf16(a), rounded to nearest; a1 the upper half word of
// the fp32 number a - a0; a2 = a - a0 - a1, which has 8 significant bits left.  |a1| <= 2^-8 |a|, |a2| < 2^-15 |a| (2^-16 and less
// on the average), and the signs of a1 and a2 are independent of a's.  Of the nine products of a b the six with i + j <= 2 are taken;
// what is left out is below the rounding of one fp32 multiplication, and the sum is rounded six times for every 32 values of the depth
// where v_mfma_f32_16x16x4_f32 rounds for each.  Against 64 bits, relative 2-norm of the error: 8192 x 512 over 512 3.4e-7 (fp32 instruction
// 4.1e-7), over 2048 7.0e-7 (8.1e-7), 64 x 1000 over 4096 2.5e-7 (3.0e-7), 128 x 256 over 784 1.2e-7 (1.6e-7).
//
// The bf16 instruction multiplies 16 times as much per clock, so six take 3/8 of the fp32 instruction's time, and, unlike it, they run
// beside vector instructions (issue_probe).  What bounds such a kernel is those: splitting an element takes 5.5 of them.  With both
// operands split by every wave that reads them, 8192 x 512 over 2048 took 115-132 us (fp32 instruction 123-138); the same loop without
// the splitting 80.  So the operand with fewer rows, the weights, is split once beforehand (planes_kernel), into 3 KB chunks in the order in
// which the lanes take them, and goes from memory to LDS as it lies; the other one stays fp32 on the way into LDS (gemm_tile.h's loaders), and
// each wave splits the columns it multiplies.  Splitting it on the way into LDS instead made LDS the bound (stores take 64 bytes a clock:
// 104-124 us), loading the columns into registers in the lanes' order the loads (105-130 us).
//
// A number below 2^-102 has parts that bf16 does not hold; one that is infinite, not a number or above the largest bf16 number has no
// split, and makes every result it enters infinite or not a number.  Columns are tested for the first as they are split, the
// prepared operand holds not a number in their place, and results are tested for that: a block that finds one computes its tile again with
// the fp32 instruction, from the operands themselves.
#pragma once
#include "fastdiv.h"
#include "gemm_tile.h"

namespace tsplit {
namespace st {

using gt::BK;
using gt::f32x4;
using gt::i32x4;
using mg::kOobOffset;
using mg::u32x4;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

constexpr int kChunk = 3072;            // bytes of 16 rows of one step: three planes of 64 lanes x 8 values
constexpr unsigned kTiny = 25u << 24;   // twice the bits of 2^-102

// (x, y) -> packed pairs of their three parts
__device__ __forceinline__ void split_pair(float x, float y, unsigned &p, unsigned &q, unsigned &r) {
  p = __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2{x, y}), bf16x2));
  x -= __uint_as_float(p << 16);
  y -= __uint_as_float(p & 0xffff0000u);
  q = __builtin_amdgcn_perm(__float_as_uint(y), __float_as_uint(x), 0x07060302u);
  x -= __uint_as_float(__float_as_uint(x) & 0xffff0000u);
  y -= __uint_as_float(__float_as_uint(y) & 0xffff0000u);
  r = __builtin_amdgcn_perm(__float_as_uint(y), __float_as_uint(x), 0x07060302u);
}
// eight values, a lane's k of both halves of a step; least: the smallest of twice the bits less one, zeros being the largest
__device__ __forceinline__ void split(const float (&lo)[4], const float (&hi)[4], bf16x8 (&out)[3], unsigned &least) {
  u32x4 w[3];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float x = i < 2 ? lo[2 * i] : hi[2 * i - 4], y = i < 2 ? lo[2 * i + 1] : hi[2 * i - 3];
    unsigned p, q, r;
    split_pair(x, y, p, q, r);
    w[0][i] = p;
    w[1][i] = q;
    w[2][i] = r;
    least = min(least, min((__float_as_uint(x) << 1) - 1u, (__float_as_uint(y) << 1) - 1u));
  }
#pragma unroll
  for (int s = 0; s < 3; ++s) out[s] = __builtin_bit_cast(bf16x8, w[s]);
}

// Rows of the prepared operand: chunk (row / 16, k / 32), lane (k / 4 % 4) * 16 + row % 16 of a chunk holds k % 4 of both halves.
struct PlanesParams {
  const char *p;
  int tiles, steps;   // chunks along the rows and along the depth
};
template <int BM>
struct Planes {
  static constexpr int kBytes = BM / 16 * kChunk, kTiles = BM / 64;   // of a wave's loads
  i32x4 rsrc;
  int row_bytes;
  __device__ __forceinline__ void init(const PlanesParams &P, int m0) {
    row_bytes = P.steps * kChunk;
    const int64_t at = static_cast<int64_t>(m0 / 16) * row_bytes;
    rsrc = gt::raw_buffer(reinterpret_cast<const float *>(P.p + at), static_cast<int64_t>(P.tiles) * row_bytes - at);
  }
  // rows past the last chunk are out of range
  __device__ __forceinline__ void load(int k0, unsigned lds) const {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const unsigned lane16 = 16u * (threadIdx.x & 63);
#pragma unroll
    for (int t = 0; t < kTiles; ++t)
#pragma unroll
      for (int s = 0; s < 3; ++s) {
        const int tile = wave * kTiles + t;
        gt::load_to_lds(rsrc, lane16, tile * row_bytes + k0 / BK * kChunk + 1024 * s, lds + tile * kChunk + 1024 * s);
      }
  }
};

// The block's verdict on its results and on the values it has split: false if the fp32 instruction has to compute the tile.  By way of
// LDS that no wave reads any more.
template <int TM, int TN>
__device__ __forceinline__ bool clean(const f32x4 (&acc)[TM][TN], unsigned least, char *lds) {
  float probe = 0.f;   // not a number once a result is infinite or not one
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) probe = fmaf(acc[i][j][e], 0.f, probe);
  int *votes = reinterpret_cast<int *>(lds);
  const bool bad = __any(least < kTiny || probe != 0.f);
  if ((threadIdx.x & 63) == 0) votes[threadIdx.x >> 6] = bad;
  __syncthreads();
  return (votes[0] | votes[1] | votes[2] | votes[3]) == 0;
}

// c + a b for one step: six products, the smallest first
template <int R, int TN>
__device__ __forceinline__ void products(const bf16x8 (&a)[R][3], const bf16x8 (&b)[TN][3], f32x4 (*acc)[TN]) {
  constexpr int kA[6] = {2, 0, 1, 1, 0, 0}, kB[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
  for (int i = 0; i < 6; ++i)
#pragma unroll
    for (int u = 0; u < R; ++u)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[u][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[u][kA[i]], b[j][kB[i]], acc[u][j], 0, 0, 0);
}

// The k-loop of one tile: rows from planes, columns from a loader BL of fp32 values.
template <int TM, int TN, int WM, int WN, class BL>
struct Core {
  static_assert(WM * WN == 4 && TM % 2 == 0, "four waves, pairs of row tiles");
  static constexpr int BM = 16 * TM * WM, BN = 16 * TN * WN;
  using AL = Planes<BM>;
  static constexpr int kStage = AL::kBytes + BL::kFloats * 4;
  static constexpr int kLdsFloats = kStage / 2;

  static __device__ __forceinline__ int wave_m0() { return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) / WN * 16 * TM; }
  static __device__ __forceinline__ int wave_n0() { return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) % WN * 16 * TN; }
  // register e of product tile tm holds row lane_row() + step_row(tm, e) of the wave's 16 TM
  static __device__ __forceinline__ int lane_row() { return 4 * (threadIdx.x >> 4 & 3); }
  static __device__ __forceinline__ constexpr int step_row(int tm, int e) { return 16 * tm + e; }

  static __device__ __forceinline__ unsigned offset_of(char *lds) {
    return static_cast<unsigned>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char *)lds));
  }
  static __device__ __forceinline__ void clear(f32x4 (&acc)[TM][TN]) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  }

  // false: the tile has to be computed with the fp32 instruction
  static __device__ __forceinline__ bool run(const AL &la, const BL &lb, int kbegin, int kend, char *lds, f32x4 (&acc)[TM][TN]) {
    const int lane = threadIdx.x & 63, wm0 = wave_m0(), wn0 = wave_n0();
    const unsigned lds_at = offset_of(lds);
    clear(acc);
    if (kbegin >= kend) return true;
    unsigned least = ~0u;
    la.load(kbegin, lds_at);
    lb.load(kbegin, kend, lds_at + AL::kBytes);
    int stage = 0;
    for (int k0 = kbegin; k0 < kend; k0 += BK) {
      char *now = lds + stage * kStage;
      float *columns = reinterpret_cast<float *>(now + AL::kBytes);
      if (lb.cut(k0, kend)) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        lb.clear_tail(k0, kend, columns);
      }
      gt::lds_ready();
      stage ^= 1;
      if (k0 + BK < kend) {
        la.load(k0 + BK, lds_at + stage * kStage);
        lb.load(k0 + BK, kend, lds_at + stage * kStage + AL::kBytes);
      }
      float b0[TN][4], b1[TN][4];
      BL::frag(columns, wn0, 0, lane, b0);
      BL::frag(columns, wn0, 1, lane, b1);
      bf16x8 b[TN][3];
#pragma unroll
      for (int j = 0; j < TN; ++j) split(b0[j], b1[j], b[j], least);
      const char *rows = now + wm0 / 16 * kChunk + 16 * lane;
#pragma unroll
      for (int tm = 0; tm < TM; tm += 2) {
        bf16x8 a[2][3];
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int s = 0; s < 3; ++s) a[u][s] = *reinterpret_cast<const bf16x8 *>(rows + (tm + u) * kChunk + 1024 * s);
        products<2, TN>(a, b, acc + tm);
      }
    }
    return clean<TM, TN>(acc, least, lds + stage * kStage);
  }

  // The same tile with the fp32 instruction, the rows element by element from `src`.
  template <class Src>
  static __device__ __forceinline__ void exact(const Src &src, int m0, const BL &lb, int kbegin, int kend, char *lds, f32x4 (&acc)[TM][TN]) {
    const int lane = threadIdx.x & 63, wm0 = wave_m0(), wn0 = wave_n0();
    float *columns = reinterpret_cast<float *>(lds);
    clear(acc);
    for (int k0 = kbegin; k0 < kend; k0 += BK) {
      __syncthreads();
      lb.load(k0, kend, offset_of(lds));
      if (lb.cut(k0, kend)) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        lb.clear_tail(k0, kend, columns);
      }
      gt::lds_ready();
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        float b[TN][4];
        BL::frag(columns, wn0, h, lane, b);
#pragma unroll
        for (int tm = 0; tm < TM; ++tm)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float a = src.at(m0 + wm0 + 16 * tm + (lane & 15), k0 + 16 * h + 4 * (lane >> 4) + i);
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[tm][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b[j][i], acc[tm][j], 0, 0, 0);
          }
      }
    }
  }
};

// The k-loop of one tile of two fp32 operands, both split by the waves that multiply them; loaders and tile as in gt::Core.
template <int TM, int TN, int WM, int WN, class AL, class BL>
struct CoreBoth : gt::Core<TM, TN, WM, WN, AL, BL> {
  using F = gt::Core<TM, TN, WM, WN, AL, BL>;   // the fp32 instruction's

  // false: the tile has to be computed with the fp32 instruction, F::run
  static __device__ __forceinline__ bool run(AL &la, BL &lb, int kbegin, int kend, float *lds, f32x4 (&acc)[TM][TN]) {
    const int lane = threadIdx.x & 63, wm0 = F::wave_m0(), wn0 = F::wave_n0();
    const unsigned lds_at = static_cast<unsigned>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) float *)lds));
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (kbegin >= kend) return true;
    unsigned least = ~0u;
    la.load(kbegin, kend, lds_at);
    lb.load(kbegin, kend, lds_at + AL::kFloats * 4);
    int stage = 0;
    for (int k0 = kbegin; k0 < kend; k0 += BK) {
      float *sa = lds + stage * F::kStage, *sb = sa + AL::kFloats;
      if (la.cut(k0, kend) || lb.cut(k0, kend)) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        la.clear_tail(k0, kend, sa);
        lb.clear_tail(k0, kend, sb);
      }
      gt::lds_ready();
      stage ^= 1;
      if (k0 + BK < kend) {
        la.load(k0 + BK, kend, lds_at + stage * F::kStage * 4);
        lb.load(k0 + BK, kend, lds_at + (stage * F::kStage + AL::kFloats) * 4);
      }
      float b0[TN][4], b1[TN][4], a0[TM][4], a1[TM][4];
      BL::frag(sb, wn0, 0, lane, b0);
      BL::frag(sb, wn0, 1, lane, b1);
      AL::frag(sa, wm0, 0, lane, a0);
      AL::frag(sa, wm0, 1, lane, a1);
      bf16x8 b[TN][3];
#pragma unroll
      for (int j = 0; j < TN; ++j) split(b0[j], b1[j], b[j], least);
#pragma unroll
      for (int tm = 0; tm < TM; ++tm) {
        bf16x8 a[1][3];
        split(a0[tm], a1[tm], a[0], least);
        products<1, TN>(a, b, acc + tm);
      }
    }
    return clean<TM, TN>(acc, least, reinterpret_cast<char *>(lds + stage * F::kStage));
  }
};

// A dense operand's element (row, k); zeros outside it
struct DenseRows {
  const float *p;
  int64_t row, step;   // distance of rows and of values along the depth
  int rows, depth;
  bool words;          // four values from a multiple of 4 on are one aligned word
  __device__ __forceinline__ float at(int r, int k) const { return r < rows && k < depth ? p[r * row + k * step] : 0.f; }
  // values k to k + 3 of a row, k a multiple of 4
  __device__ __forceinline__ void four(int r, int k, float (&v)[4]) const {
    if (words) {
      const f32x4 w = r < rows && k < depth ? *reinterpret_cast<const f32x4 *>(p + r * row + k) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = w[j];
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = at(r, k + j);
    }
  }
};
inline DenseRows dense_rows(const float *p, int64_t row, int64_t step, int rows, int depth) {
  return DenseRows{p, row, step, rows, depth, step == 1 && row % 4 == 0 && depth % 4 == 0 && (reinterpret_cast<uintptr_t>(p) & 15) == 0};
}

// one lane's eight values of a chunk, row and first k as they fall to it
template <class Src>
__device__ __forceinline__ void put_planes(const Src &src, int row, int k, char *chunk, int lane) {
  float lo[4], hi[4];
  src.four(row, k, lo);
  src.four(row, k + 16, hi);
  bf16x8 w[3];
  unsigned least = ~0u;
  split(lo, hi, w, least);
  if (least < kTiny) w[0][0] = __builtin_bit_cast(__bf16, static_cast<unsigned short>(0x7fc0));   // not a number
#pragma unroll
  for (int s = 0; s < 3; ++s) *reinterpret_cast<bf16x8 *>(chunk + 1024 * s + 16 * lane) = w[s];
}
// A block a chunk, so that small operands spread over the chip.  blockIdx.y: one of a batch of operands, `stride` values apart, and its planes
static __global__ __launch_bounds__(64) void planes_kernel(DenseRows src, int64_t stride, char *__restrict__ out, FastDiv steps) {
  src.p += blockIdx.y * stride;
  out += static_cast<int64_t>(blockIdx.y) * gridDim.x * kChunk;
  const int lane = threadIdx.x, chunk = blockIdx.x, tile = steps.div(chunk);
  put_planes(src, 16 * tile + (lane & 15), (chunk - tile * steps.d) * BK + 4 * (lane >> 4), out + static_cast<int64_t>(chunk) * kChunk, lane);
}

// ---- dense products.  C[M,N] = rows x columns: the rows of A and the columns of B, or (ACROSS) the columns of B and the rows of A.
// XMN: the columns' operand is stored with the depth as its rows.  Batch z's operands and result begin z strides further on; with
// kchunk < K (a batch of one) z is a range of the depth.
struct SplitStrides {
  int64_t planes, src, x, out;
};
template <int TM, int TN, int WM, int WN, bool XMN, bool ACROSS>
__global__ __launch_bounds__(gt::kThreads, 2) void gemm_split_kernel(PlanesParams rows, DenseRows src, mg::DenseParams xp, float *__restrict__ out,
                                                                     SplitStrides zs, bool wide, int P, int X, int K, int kchunk, mg::TileGrid tg) {
  using BL = typename std::conditional<XMN, gt::MnContig<16 * TN * WN, TN>, gt::KContig<16 * TN * WN, TN, !ACROSS>>::type;
  using C = Core<TM, TN, WM, WN, BL>;
  __shared__ __attribute__((aligned(1024))) float lds_f[C::kLdsFloats];
  char *const lds = reinterpret_cast<char *>(lds_f);
  int z, tile_m, tile_n;
  if (!mg::block_tile(tg, z, tile_m, tile_n)) return;
  const int m0 = tile_m * C::BM, n0 = tile_n * C::BN, kbegin = kchunk < K ? z * kchunk : 0, kend = min(K, kbegin + kchunk);
  rows.p += z * zs.planes;
  src.p += z * zs.src;
  xp.p += z * zs.x;
  typename C::AL la;
  BL lb;
  la.init(rows, m0);
  lb.init(xp, n0);
  f32x4 acc[TM][TN];
  if (!C::run(la, lb, kbegin, kend, lds, acc)) C::exact(src, m0, lb, kbegin, kend, lds, acc);

  float *o = out + z * zs.out;
  const int lane = threadIdx.x & 63, idx = lane & 15;
  if constexpr (!ACROSS) {
    const int64_t ldc = X;
    const int m = m0 + C::wave_m0(), n = n0 + C::wave_n0() + TN * idx;
    if (m >= P) return;
    const __amdgpu_buffer_rsrc_t to = gt::output_buffer(o + static_cast<int64_t>(m) * ldc, static_cast<int64_t>(P - m) * ldc * 4);
    const int row_bytes = static_cast<int>(ldc) * 4;
    const unsigned at = (static_cast<unsigned>(C::lane_row()) * static_cast<unsigned>(ldc) + static_cast<unsigned>(n)) * 4u;
    unsigned off[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) off[j] = n + j < X ? at + 4u * j : kOobOffset;
#pragma unroll
    for (int tm = 0; tm < TM; ++tm)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int soff = C::step_row(tm, e) * row_bytes;
        if (wide) {
          float v[TN];
#pragma unroll
          for (int j = 0; j < TN; ++j) v[j] = acc[tm][j][e];
          gt::store_words<TN>(to, off[0], soff, v);
        } else {
#pragma unroll
          for (int j = 0; j < TN; ++j) __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(acc[tm][j][e]), to, off[j], soff, 0);
        }
      }
  } else {
    // a lane holds four neighbouring columns of C in each of TN rows
    const int64_t ldc = P;
    const int x = n0 + C::wave_n0(), p = m0 + C::wave_m0() + C::lane_row();
    if (x >= X) return;
    const __amdgpu_buffer_rsrc_t to = gt::output_buffer(o + static_cast<int64_t>(x) * ldc, static_cast<int64_t>(X - x) * ldc * 4);
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int row = XMN ? TN * idx + j : 16 * j + idx;
      const unsigned at = (static_cast<unsigned>(row) * static_cast<unsigned>(ldc) + static_cast<unsigned>(p)) * 4u;
#pragma unroll
      for (int tm = 0; tm < TM; ++tm) {
        if (wide) {
          const float v[4] = {acc[tm][j][0], acc[tm][j][1], acc[tm][j][2], acc[tm][j][3]};
          gt::store_words<4>(to, p + 16 * tm < P ? at : kOobOffset, 64 * tm, v);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(acc[tm][j][e]), to, p + 16 * tm + e < P ? at + 64u * tm + 4u * e : kOobOffset, 0, 0);
        }
      }
    }
  }
}

// A tile's accumulators as Core lays them, to rows of C.  (gemm_tile_kernel keeps the same lines in its body: taken out into a function there they
// changed the order of its loop, 64 x 4096 over 4096, second operand transposed, 23.8 -> 25.5 us.)
template <class C, int TM, int TN>
__device__ __forceinline__ void store_rows(const f32x4 (&acc)[TM][TN], float *__restrict__ o, int64_t ldc, bool wide, int M, int N, int m0, int n0) {
  // the wave's rows to the end of C: rows past it are out of range
  const int m = m0 + C::wave_m0(), n = n0 + C::wave_n0() + TN * (threadIdx.x & 15);
  if (m >= M) return;
  const __amdgpu_buffer_rsrc_t to = gt::output_buffer(o + static_cast<int64_t>(m) * ldc, static_cast<int64_t>(M - m) * ldc * 4);
  const int row_bytes = static_cast<int>(ldc) * 4;
  const unsigned at = (static_cast<unsigned>(C::lane_row()) * static_cast<unsigned>(ldc) + static_cast<unsigned>(n)) * 4u;
  unsigned off[TN];
#pragma unroll
  for (int j = 0; j < TN; ++j) off[j] = n + j < N ? at + 4u * j : kOobOffset;
#pragma unroll
  for (int tm = 0; tm < TM; ++tm)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int soff = C::step_row(tm, e) * row_bytes;
      if (wide) {   // N is a multiple of TN: a word lies inside its row or behind it
        float v[TN];
#pragma unroll
        for (int j = 0; j < TN; ++j) v[j] = acc[tm][j][e];
        gt::store_words<TN>(to, off[0], soff, v);
      } else {
#pragma unroll
        for (int j = 0; j < TN; ++j) __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(acc[tm][j][e]), to, off[j], soff, 0);
      }
    }
}

// Both operands split by the waves: batch z % batch of operands `zs.a` and `zs.b` values apart, range z / batch of the depth; result z begins
// z * zs.c values further on.
template <int TM, int TN, int WM, int WN, bool TA, bool TB>
__global__ __launch_bounds__(gt::kThreads, 2) void gemm_both_kernel(mg::DenseParams ap, mg::DenseParams bp, float *__restrict__ out, gt::Strides zs, int batch,
                                                                    bool wide, int M, int N, int K, int kchunk, mg::TileGrid tg) {
  using T = gt::Tile<TM, TN, WM, WN, TA, TB>;
  using C = CoreBoth<TM, TN, WM, WN, typename T::AL, typename T::BL>;
  __shared__ __attribute__((aligned(1024))) float lds[T::C::kLdsFloats];
  int z, tile_m, tile_n;
  if (!mg::block_tile(tg, z, tile_m, tile_n)) return;
  const int range = z / batch, m0 = tile_m * T::BM, n0 = tile_n * T::BN, kbegin = range * kchunk, kend = min(K, kbegin + kchunk);
  ap.p += (z - range * batch) * zs.a;
  bp.p += (z - range * batch) * zs.b;
  typename T::AL la;
  typename T::BL lb;
  la.init(ap, m0);
  lb.init(bp, n0);
  f32x4 acc[TM][TN];
  if (!C::run(la, lb, kbegin, kend, lds, acc)) {
    __syncthreads();   // the verdict lies where the first step goes
    C::F::run(la, lb, kbegin, kend, lds, acc);
  }
  store_rows<typename T::C>(acc, out + z * zs.c, N, wide, M, N, m0, n0);
}

}  // namespace st
}  // namespace tsplit
