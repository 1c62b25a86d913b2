// fp32 MFMA tile kernel of the matrix products: C[M,N] = op(A) op(B) with v_mfma_f32_16x16x4_f32.
//
// 256 threads, four waves on a WM x WN grid; each wave owns 16 TM x 16 TN of the tile (64 x 64 at most: wider wave tiles leave
// one wave per SIMD, and 128 x 256 block tiles ran at 133 TFLOP/s where 128 x 128 run at 149).  K advances in steps of 32
// through two LDS stages.  A step is two 16-deep halves; the operand words of a half are read while the half before
// multiplies, so neither LDS nor the barrier, one a step, stands between two bursts of products.
//
// What bounds it is the matrix pipe, and what takes time from the matrix pipe is every other instruction that moves vector
// registers.  So the operands go from memory to LDS without passing through registers (buffer loads with LDS as their
// destination, 16 bytes a lane, out-of-range lanes write zeros): the same loop with loads into registers and LDS stores
// reached 130-138 TFLOP/s at 8192^3, this one 145-150 (fp32 matrix peak 157).
//
// Each operand is staged in the orientation it has in memory, [mn][32] where K is contiguous, [32][mn] where the M or N
// index is; both supply lane group g of 16 lanes with k = 4 g + i of a half.  The columns of the result are dealt to the
// product tiles so that a lane holds TN neighbouring ones and the result leaves in 16-byte (TN = 2: 8-byte) words.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "activations.h"
#include "mfma_gemm.h"

namespace tsplit {
namespace gt {

constexpr int BK = 32;
constexpr int kThreads = 256;

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
using mg::kOobOffset;

// A raw buffer as the four words the load takes (base, size in bytes, format word of mg::kBufFlags)
__device__ __forceinline__ i32x4 raw_buffer(const float *p, int64_t bytes) {
  const uint64_t a = reinterpret_cast<uint64_t>(p);
  return i32x4{__builtin_amdgcn_readfirstlane(static_cast<int>(a)), __builtin_amdgcn_readfirstlane(static_cast<int>(a >> 32) & 0xffff),
               __builtin_amdgcn_readfirstlane(static_cast<int>(bytes < 0x7fffffffll ? bytes : 0x7fffffffll)), mg::kBufFlags};
}

// 64 lanes x 16 bytes from the buffer straight into LDS, at `lds` + 16 * lane (bytes); voff: the lane's byte offset, soff:
// the wave's.  Lanes out of range write zeros.  The compiler does not see the LDS write (lds_ready() orders it) nor that a vector
// memory instruction reads the scalar registers, which may have been written by a vector instruction just before: five wait states.
// (m0 is declared although the compiler never keeps a value of its own there and says so: it does merge equal writes of it.)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void load_to_lds(i32x4 rsrc, unsigned voff, int soff, unsigned lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 3\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"(__builtin_amdgcn_readfirstlane(lds)), "v"(voff),
               "s"(rsrc), "s"(__builtin_amdgcn_readfirstlane(soff))
               : "memory", "m0");
}
// the same with 4 bytes a lane, at `lds` + 4 * lane
__device__ __forceinline__ void load_word_to_lds(i32x4 rsrc, unsigned voff, int soff, unsigned lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 3\n\tbuffer_load_dword %1, %2, %3 offen lds" ::"s"(__builtin_amdgcn_readfirstlane(lds)), "v"(voff),
               "s"(rsrc), "s"(__builtin_amdgcn_readfirstlane(soff))
               : "memory", "m0");
}
#pragma clang diagnostic pop
// Everything this wave has asked for lies in LDS, every operand word it has read is in registers; then the block's barrier.
// The wait comes twice: the compiler counts LDS reads only from the one it knows.  Without it scalar loads from before the
// k-loop counted as outstanding through every step, and each half's reads were waited for in full before the half before
// multiplied (8192 x 8192 x 8192 with B transposed: 7.88 ms, with it 7.60).
__device__ __forceinline__ void lds_ready() {
  __builtin_amdgcn_s_waitcnt(0x0070);   // vmcnt(0) lgkmcnt(0)
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// Operand with K contiguous: element (mn, k) at p[mn * ld + k].  LDS: [MN][32], word q of row s holds k-word q ^ (s / 2 % 8)
// (the 16 rows a product tile's lanes read then start on 16 different bank groups).  PERM: LDS row s of a wave's 16 T rows
// holds matrix row (s % 16) * T + s / 16, so that tile t's lane c supplies index T c + t.
template <int MN, int T, bool PERM>
struct KContig {
  static constexpr bool kDense = true;
  static constexpr int kParts = 1;
  static constexpr bool kDealt = PERM;   // tile t's lane r supplies index T r + t, not 16 t + r
  static constexpr int kFloats = MN * BK;
  static constexpr int kLoads = MN / 32;   // a wave's loads a step, 8 rows each
  unsigned voff[kLoads];
  i32x4 rsrc;
  int lane, wave;
  __device__ __forceinline__ void init(const mg::DenseParams &P, int mn0) {
    lane = threadIdx.x & 63;
    wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int rows_left = P.mn_total - mn0;
    // (rows that are part of longer ones end with their own last value)
    rsrc = raw_buffer(P.p + static_cast<int64_t>(mn0) * P.ld, (static_cast<int64_t>(rows_left - 1) * P.ld + P.k_total) * 4);
    const int slot0 = wave * kLoads * 8 + (lane >> 3);
    const unsigned row_bytes = static_cast<unsigned>(P.ld) * 4u;
    if constexpr (PERM) {
#pragma unroll
      for (int s = 0; s < kLoads; ++s) {
        const int slot = slot0 + 8 * s, row = slot / (16 * T) * (16 * T) + slot % 16 * T + slot / 16 % T;
        voff[s] = row < rows_left ? static_cast<unsigned>(row) * row_bytes + 16u * word_of(slot) : kOobOffset;
      }
    } else {
      const unsigned at = static_cast<unsigned>(slot0) * row_bytes;
#pragma unroll
      for (int s = 0; s < kLoads; ++s) voff[s] = slot0 + 8 * s < rows_left ? at + 8u * s * row_bytes + 16u * word_of(slot0 + 8 * s) : kOobOffset;
    }
  }
  // the k-word this lane fetches for an LDS row
  __device__ __forceinline__ unsigned word_of(int slot) const { return (lane & 7) ^ (slot >> 1 & 7); }
  // words beyond kend read as zeros; the word that kend cuts is cut by clear_tail()
  __device__ __forceinline__ void load(int k0, int kend, unsigned lds) const {
    lds += wave * kLoads * 1024;
    if (k0 + BK <= kend) {
#pragma unroll
      for (int s = 0; s < kLoads; ++s) load_to_lds(rsrc, voff[s], k0 * 4, lds + 1024 * s);
    } else {
#pragma unroll
      for (int s = 0; s < kLoads; ++s) {
        const int slot = (wave * kLoads + s) * 8 + (lane >> 3);
        const int word = (lane & 7) ^ (slot >> 1 & 7);
        load_to_lds(rsrc, k0 + 4 * word < kend ? voff[s] : kOobOffset, k0 * 4, lds + 1024 * s);
      }
    }
  }
  // this step's last word holds values past kend
  __device__ __forceinline__ bool cut(int k0, int kend) const { return k0 + BK > kend && (kend & 3) != 0; }
  // zeroes the values at and beyond kend of the words this lane has fetched (they belong to the next row)
  __device__ __forceinline__ void clear_tail(int k0, int kend, float *lds) const {
#pragma unroll
    for (int s = 0; s < kLoads; ++s) {
      const int slot = (wave * kLoads + s) * 8 + (lane >> 3);
      const int word = (lane & 7) ^ (slot >> 1 & 7), keep = kend - (k0 + 4 * word);
      if (keep > 0)
        for (int i = keep; i < 4; ++i) lds[slot * BK + 4 * (lane & 7) + i] = 0.f;
    }
  }
  static __device__ __forceinline__ void frag(const float *lds, int mn0, int h, int lane, float (&v)[T][4]) {
#pragma unroll
    for (int t = 0; t < T; ++t) {
      const int slot = mn0 + 16 * t + (lane & 15);
      const f32x4 q = *reinterpret_cast<const f32x4 *>(lds + slot * BK + 4 * ((4 * h + (lane >> 4)) ^ (slot >> 1 & 7)));
#pragma unroll
      for (int i = 0; i < 4; ++i) v[t][i] = q[i];
    }
  }
};

// Operand with M or N contiguous: element (k, mn) at p[k * ld + mn].  LDS: [32][MN].  A word past a row's end holds the next
// row's first values: they belong to rows or columns of C that do not exist.
template <int MN, int T>
struct MnContig {
  static constexpr bool kDense = true, kDealt = true;
  static constexpr int kParts = 1;
  static constexpr int kFloats = BK * MN;
  static constexpr int kLoads = MN / 32;
  static constexpr int kWords = MN / 4;            // 16-byte words of a row
  static constexpr int kRows = 64 / kWords;        // rows of one load
  static_assert(kWords <= 64, "a load covers whole rows");
  unsigned voff;
  i32x4 rsrc;
  int row_bytes, wave;
  __device__ __forceinline__ void init(const mg::DenseParams &P, int mn0) {
    const int lane = threadIdx.x & 63;
    wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    row_bytes = static_cast<int>(P.ld) * 4;
    rsrc = raw_buffer(P.p, (static_cast<int64_t>(P.k_total - 1) * P.ld + P.mn_total) * 4);
    const int col = mn0 + 4 * (lane % kWords);
    voff = col < P.mn_total ? (static_cast<unsigned>(lane / kWords) * static_cast<unsigned>(P.ld) + static_cast<unsigned>(col)) * 4u : kOobOffset;
  }
  // rows past the matrix' end are out of range
  __device__ __forceinline__ void load(int k0, int /*kend*/, unsigned lds) const {
#pragma unroll
    for (int s = 0; s < kLoads; ++s)
      load_to_lds(rsrc, voff, (k0 + (wave * kLoads + s) * kRows) * row_bytes, lds + (wave * kLoads + s) * 1024);
  }
  __device__ __forceinline__ bool cut(int, int) const { return false; }
  __device__ __forceinline__ void clear_tail(int, int, float *) const {}
  static __device__ __forceinline__ void frag(const float *lds, int mn0, int h, int lane, float (&v)[T][4]) {
    typedef float vec __attribute__((ext_vector_type(T)));
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const vec q = *reinterpret_cast<const vec *>(lds + (16 * h + 4 * (lane >> 4) + i) * MN + mn0 + T * (lane & 15));
#pragma unroll
      for (int t = 0; t < T; ++t) v[t][i] = q[t];
    }
  }
};

template <int TM, int TN>
__device__ __forceinline__ void products(const float (&a)[TM][4], const float (&b)[TN][4], f32x4 (&acc)[TM][TN]) {
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int tm = 0; tm < TM; ++tm)
#pragma unroll
      for (int tn = 0; tn < TN; ++tn) acc[tm][tn] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[tm][i], b[tn][i], acc[tm][tn], 0, 0, 0);
}
// the same with between(i) behind each quarter
template <int TM, int TN, class Between>
__device__ __forceinline__ void products_and(const float (&a)[TM][4], const float (&b)[TN][4], f32x4 (&acc)[TM][TN], Between between) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
#pragma unroll
    for (int tm = 0; tm < TM; ++tm)
#pragma unroll
      for (int tn = 0; tn < TN; ++tn) acc[tm][tn] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[tm][i], b[tn][i], acc[tm][tn], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
    between(i);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// Output words: T neighbouring columns of a row, at voff + step bytes (kOobOffset: nowhere).  The step is added to the lane's
// offset and not passed as the scalar offset: with a scalar register there, 16-byte stores whose data registers the next
// instruction writes again lost values (the wait state such a store needs is only inserted for the other form).
template <int T>
__device__ __forceinline__ void store_words(__amdgpu_buffer_rsrc_t to, unsigned voff, int step, const float (&v)[T]) {
  voff += step;   // (kOobOffset stays out of range: steps are below 2 GiB)
  if constexpr (T == 4)
    __builtin_amdgcn_raw_buffer_store_b128(mg::u32x4{__float_as_uint(v[0]), __float_as_uint(v[1]), __float_as_uint(v[2]), __float_as_uint(v[3])}, to,
                                           voff, 0, 0);
  else
    __builtin_amdgcn_raw_buffer_store_b64(u32x2{__float_as_uint(v[0]), __float_as_uint(v[1])}, to, voff, 0, 0);
}
template <int T>
__device__ __forceinline__ void load_words(__amdgpu_buffer_rsrc_t from, unsigned voff, int step, float (&v)[T]) {
  if constexpr (T == 4) {
    const mg::u32x4 r = __builtin_amdgcn_raw_buffer_load_b128(from, voff + step, 0, 0);
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = __uint_as_float(r[j]);
  } else {
    const u32x2 r = __builtin_amdgcn_raw_buffer_load_b64(from, voff + step, 0, 0);
#pragma unroll
    for (int j = 0; j < 2; ++j) v[j] = __uint_as_float(r[j]);
  }
}
__device__ __forceinline__ __amdgpu_buffer_rsrc_t output_buffer(float *p, int64_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(p, 0, static_cast<int>(bytes < 0x7fffffffll ? bytes : 0x7fffffffll), mg::kBufFlags);
}

// The k-loop of one tile with operand loaders AL, BL: acc = sum over [kbegin, kend).
template <int TM, int TN, int WM, int WN, class AL, class BL, bool SPREAD = (BL::kParts > 1)>
struct Core {
  static_assert(WM * WN == 4, "four waves");
  static constexpr int BM = 16 * TM * WM, BN = 16 * TN * WN;
  static constexpr int kStage = AL::kFloats + BL::kFloats;
  static constexpr int kLdsFloats = 2 * kStage;

  static __device__ __forceinline__ int wave_m0() { return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) / WN * 16 * TM; }
  static __device__ __forceinline__ int wave_n0() { return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) % WN * 16 * TN; }
  // register e of product tile tm holds row lane_row() + step_row(tm, e) of the wave's 16 TM
  static __device__ __forceinline__ int lane_row() { return (AL::kDealt ? 4 * TM : 4) * (threadIdx.x >> 4 & 3); }
  static __device__ __forceinline__ constexpr int step_row(int tm, int e) { return AL::kDealt ? TM * e + tm : 16 * tm + e; }

  static __device__ __forceinline__ void run(AL &la, BL &lb, int kbegin, int kend, float *lds, f32x4 (&acc)[TM][TN]) {
    float none[TN];
    run<false>(la, lb, kbegin, kend, lds, acc, false, none);
  }
  // SUMS, where `on`: col[t] is also the sum over the range of what this lane supplies of B's column of tile t (of lane group g the
  // k = 4 g + i of every half).  Eight of a step are added pairwise, eight steps one by one, then those: in ranges of up to
  // 16 K rows no longer a chain of roundings than a reduction in slices has.
  template <bool SUMS>
  static __device__ __forceinline__ void run(AL &la, BL &lb, int kbegin, int kend, float *lds, f32x4 (&acc)[TM][TN], bool on, float (&col)[TN]) {
    const int lane = threadIdx.x & 63, wm0 = wave_m0(), wn0 = wave_n0();
    const unsigned lds_at = static_cast<unsigned>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) float *)lds));
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    float some[TN];
    if constexpr (SUMS) {
#pragma unroll
      for (int j = 0; j < TN; ++j) col[j] = some[j] = 0.f;
    }
    if (kbegin >= kend) return;
    float a0[TM][4], b0[TN][4], a1[TM][4], b1[TN][4];
    auto add = [&](const float (&b)[TN][4]) {
      if constexpr (SUMS)
        if (on) {
#pragma unroll
          for (int j = 0; j < TN; ++j) some[j] += (b[j][0] + b[j][1]) + (b[j][2] + b[j][3]);
        }
    };
    la.load(kbegin, kend, lds_at);
    lb.load(kbegin, kend, lds_at + AL::kFloats * 4);
    int stage = 0;
    // SPREAD: the next step's loads of B between the products.  A load takes the memory pipeline 16 clocks whatever its width, and a wave
    // issues in order: 8 to 16 loads of 4 bytes a lane in one burst behind the barrier kept it from its next product until the last
    // was taken.  Two to four behind each quarter of the products: 3x3 of 35 x 35 70.1 -> 63.5 us, 17 x 17 of several taps 69.1 -> 59.5,
    // 512 -> 512 of 28 x 28, 18 images 558 -> 497, its filter gradient 570 -> 525, stride-2 data gradients 0.91-0.94 of the time, filter
    // gradients 0.92-0.97.  Operands in words (2 to 8 loads a step) and one-tap gathers, which have no choice of offsets to make, gained
    // nothing either way, nor did the LDS reads between products.  The first step has no products to put loads between, the last none to
    // ask for: forms of their own (`first`, `more` are types then), since a branch between products costs registers (108 -> 149 on 128 x 64).
    static_assert(!(SPREAD && SUMS), "loads between products leave no column sums");
    auto step = [&](int k0, auto first, auto more) {
      if (la.cut(k0, kend) || lb.cut(k0, kend)) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        la.clear_tail(k0, kend, lds + stage * kStage);
        lb.clear_tail(k0, kend, lds + stage * kStage + AL::kFloats);
      }
      lds_ready();
      const float *sa = lds + stage * kStage, *sb = sa + AL::kFloats;
      stage ^= 1;
      const unsigned next_a = lds_at + stage * kStage * 4, next_b = next_a + AL::kFloats * 4;
      if (more) {
        if constexpr (SPREAD) {
          lb.prepare(k0 + BK, kend, next_b);
        } else {
          la.load(k0 + BK, kend, next_a);
          lb.load(k0 + BK, kend, next_b);
        }
      }
      AL::frag(sa, wm0, 0, lane, a0);
      BL::frag(sb, wn0, 0, lane, b0);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (SPREAD) {
        auto part = [&](int i) {
          if (!more) return;
          if (i == 0) la.load(k0 + BK, kend, next_a);
          lb.part(i);
        };
        if (first) {
#pragma unroll
          for (int i = 0; i < 4; ++i) part(i);
        } else {
          products_and<TM, TN>(a1, b1, acc, part);
        }
      } else if (!first) {
        products<TM, TN>(a1, b1, acc);
        add(b1);
        if constexpr (SUMS)
          if (((k0 - kbegin) & (8 * BK - 1)) == 0) {
#pragma unroll
            for (int j = 0; j < TN; ++j) {
              col[j] += some[j];
              some[j] = 0.f;
            }
          }
      }
      __builtin_amdgcn_sched_barrier(0);
      AL::frag(sa, wm0, 1, lane, a1);
      BL::frag(sb, wn0, 1, lane, b1);
      __builtin_amdgcn_sched_barrier(0);
      products<TM, TN>(a0, b0, acc);
      add(b0);
      __builtin_amdgcn_sched_barrier(0);
    };
    if constexpr (SPREAD) {
      const std::true_type yes{};
      const std::false_type no{};
      int k0 = kbegin;
      if (k0 + BK >= kend) {
        step(k0, yes, no);
      } else {
        step(k0, yes, yes);
        for (k0 += BK; k0 + BK < kend; k0 += BK) step(k0, no, yes);
        step(k0, no, no);
      }
    } else {
      for (int k0 = kbegin; k0 < kend; k0 += BK) step(k0, k0 == kbegin, k0 + BK < kend);
    }
    // (a depth whose last half step is all zeros: 100 x 4096' x 4096 46 -> 43 us; convolutions' depths are cut and padded otherwise, and gained
    // nothing)
    if (!BL::kDense || ((kend - kbegin - 1) & (BK - 1)) >= BK / 2) products<TM, TN>(a1, b1, acc);
    add(b1);
    if constexpr (SUMS) {
#pragma unroll
      for (int j = 0; j < TN; ++j) col[j] += some[j];
    }
  }
};

// ---- dense products.  TA: A is stored [K][M]; TB: B is stored [N][K]
template <int TM, int TN, int WM, int WN, bool TA, bool TB>
struct Tile {
  static constexpr int BM = 16 * TM * WM, BN = 16 * TN * WN;
  using AL = typename std::conditional<TA, MnContig<BM, TM>, KContig<BM, TM, false>>::type;
  using BL = typename std::conditional<TB, KContig<BN, TN, true>, MnContig<BN, TN>>::type;
  using C = Core<TM, TN, WM, WN, AL, BL>;

  // SUMS: the tiles of the first row also leave the sums of B's columns over the range
  template <bool SUMS = false>
  static __device__ __forceinline__ void run(const mg::DenseParams &ap, const mg::DenseParams &bp, float *__restrict__ o, int64_t ldc,
                                             bool wide, int M, int N, int m0, int n0, int kbegin, int kend, float *lds, float *__restrict__ sums = nullptr) {
    AL la;
    BL lb;
    la.init(ap, m0);
    lb.init(bp, n0);
    f32x4 acc[TM][TN];
    if constexpr (SUMS) {
      float col[TN];
      const bool on = m0 == 0 && C::wave_m0() == 0;   // two waves have all columns between them
      C::template run<true>(la, lb, kbegin, kend, lds, acc, on, col);
      if (on) {
        const int lane = threadIdx.x & 63, c = n0 + C::wave_n0() + TN * (lane & 15);
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          col[j] += __shfl_xor(col[j], 16, 64);
          col[j] += __shfl_xor(col[j], 32, 64);
          if (lane < 16 && c + j < N) sums[c + j] = col[j];
        }
      }
    } else {
      C::run(la, lb, kbegin, kend, lds, acc);
    }
    // the wave's rows to the end of C: rows past it are out of range
    const int m = m0 + C::wave_m0(), n = n0 + C::wave_n0() + TN * (threadIdx.x & 15);
    if (m >= M) return;
    const __amdgpu_buffer_rsrc_t to = output_buffer(o + static_cast<int64_t>(m) * ldc, static_cast<int64_t>(M - m) * ldc * 4);
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
          store_words<TN>(to, off[0], soff, v);
        } else {
#pragma unroll
          for (int j = 0; j < TN; ++j) __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(acc[tm][j][e]), to, off[j], soff, 0);
        }
      }
  }
};

// Batch z's operands and result begin z strides further on; with kchunk < K (a batch of one) z is a split and covers
// k in [z * kchunk, (z + 1) * kchunk).
struct Strides {
  int64_t a, b, c;
};
template <int TM, int TN, int WM, int WN, bool TA, bool TB>
__global__ __launch_bounds__(kThreads, 2) void gemm_tile_kernel(mg::DenseParams ap, mg::DenseParams bp, float *__restrict__ out, Strides zs,
                                                                bool wide, int M, int N, int K, int kchunk, mg::TileGrid tg) {
  using T = Tile<TM, TN, WM, WN, TA, TB>;
  __shared__ __attribute__((aligned(1024))) float lds[T::C::kLdsFloats];
  int z, tile_m, tile_n;
  if (!mg::block_tile(tg, z, tile_m, tile_n)) return;
  ap.p += z * zs.a;
  bp.p += z * zs.b;
  const int kbegin = kchunk < K ? z * kchunk : 0;
  T::run(ap, bp, out + z * zs.c, N, wide, M, N, tile_m * T::BM, tile_n * T::BN, kbegin, min(K, kbegin + kchunk), lds);
}

// C = A^T B and the sums of B's columns (a linear layer's two parameter gradients from its input and the gradient of its output): the
// blocks of the first row of tiles have every column of B in their registers on the way.  As a reduction of its own the sums take two
// launches, 10.5 us for 8192 x 512 where the product takes 35.  Column sums of range z go to sums + z * zs.
template <int TM, int TN>
__global__ __launch_bounds__(kThreads, 2) void gemm_sums_kernel(mg::DenseParams ap, mg::DenseParams bp, float *__restrict__ out, float *__restrict__ sums,
                                                                int64_t zs, bool wide, int M, int N, int K, int kchunk, mg::TileGrid tg) {
  using T = Tile<TM, TN, 2, 2, true, false>;
  __shared__ __attribute__((aligned(1024))) float lds[T::C::kLdsFloats];
  int z, tile_m, tile_n;
  if (!mg::block_tile(tg, z, tile_m, tile_n)) return;
  T::template run<true>(ap, bp, out + z * zs, N, wide, M, N, tile_m * T::BM, tile_n * T::BN, z * kchunk, min(K, (z + 1) * kchunk), lds, sums + z * zs);
}

// The ranges of both added: first[i] for i < split, second[i - split] behind that, of `n` values a range (split and n multiples of VEC)
template <int VEC>
static __global__ __launch_bounds__(256) void fold_two_kernel(const float *__restrict__ part, float *__restrict__ first, float *__restrict__ second,
                                                              int64_t split, int64_t n, int S) {
  typedef float vec __attribute__((ext_vector_type(VEC)));
  const int64_t i = (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x) * VEC;
  if (i >= n) return;
  auto read = [&](int z) { return *reinterpret_cast<const vec *>(part + z * n + i); };
  vec s = read(0);
  int z = 1;
  for (; z + 4 <= S; z += 4) {
    const vec a = read(z), b = read(z + 1), c = read(z + 2), d = read(z + 3);
    s += a;
    s += b;
    s += c;
    s += d;
  }
  for (; z < S; ++z) s += read(z);
  *reinterpret_cast<vec *>(i < split ? first + i : second + (i - split)) = s;
}

// ---- products whose result is worked on before it is stored
// What follows the sum of products, in this order and with a rounding each, as the operators behind a product would do it (but for alpha *
// sum + mask_value, rounded once; alpha is 1 where there is a bias):
// v = alpha * sum; + bias[column]; + mask_value where mask[column] is 0; fill where the column lies right of the row; + add; stored, and
// max(v, 0) stored as well; or the result, as the gradient behind a Relu, taken through it: as a second array or in place of the result.
// Each of these as an operator of its own reads and writes the whole result again: scores of 32 x 8 x 256 x
// 256 (67 MB) took 29 us as a product and 175 with a scale, a mask and a causal selection behind it, a projection of 8192 x 512 over 512
// 36 and 64 us with its bias and a residual.
struct Epilogue {
  float alpha;
  const float *bias;     // of N; null: none
  const float *mask;     // of N, for the outer batch index; null: none
  float mask_value;
  int causal;
  float fill;
  const float *add;      // laid out as the result, which it may be (a lane reads a value before it writes it); null: none
  float *relu;           // likewise; null: not stored
  const float *gate;     // the input of the Relu that the result is taken through, laid out as the result and no array written; null: none
  // the second value of v: Relu, or its gradient where it let x through
  __device__ __forceinline__ float second(float v, float x) const { return gate ? relu_grad_of(x, v) : fmaxf(v, 0.f); }
  __device__ __forceinline__ float at(float v, int m, int n, float b, bool masked) const {
    v *= alpha;
    if (bias) v += b;
    if (mask) v += masked ? mask_value : 0.f;
    if (causal && n > m) v = fill;
    return v;
  }
};
// Batch z is (z / inner, z % inner); an operand's matrices lie `o` apart by the first index and `i` by the second (heads that share the rows
// of one array lie a head's width apart).
struct BatchOf {
  int inner;
  int64_t ao, ai, bo, bi, co, ci;
};

template <int TM, int TN, bool TA, bool TB>
__global__ __launch_bounds__(kThreads, 2) void gemm_epilogue_kernel(mg::DenseParams ap, mg::DenseParams bp, float *out, int64_t ldc,
                                                                    BatchOf zs, Epilogue ep, bool wide, int M, int N, int K, mg::TileGrid tg) {
  using T = Tile<TM, TN, 2, 2, TA, TB>;
  using C = typename T::C;
  __shared__ __attribute__((aligned(1024))) float lds[C::kLdsFloats];
  int z, tile_m, tile_n;
  if (!mg::block_tile(tg, z, tile_m, tile_n)) return;
  const int zo = z / zs.inner, zi = z - zo * zs.inner;
  ap.p += zo * zs.ao + zi * zs.ai;
  bp.p += zo * zs.bo + zi * zs.bi;
  const int64_t c_at = zo * zs.co + zi * zs.ci;
  const int m0 = tile_m * T::BM, n0 = tile_n * T::BN;
  typename T::AL la;
  typename T::BL lb;
  la.init(ap, m0);
  lb.init(bp, n0);
  f32x4 acc[TM][TN];
  C::run(la, lb, 0, K, lds, acc);
  const int m = m0 + C::wave_m0(), n = n0 + C::wave_n0() + TN * (threadIdx.x & 15);
  if (m >= M) return;
  // rows past the last one are out of range; a row's columns past N go nowhere
  const int64_t from = c_at + static_cast<int64_t>(m) * ldc, bytes = (static_cast<int64_t>(M - m - 1) * ldc + N) * 4;
  const __amdgpu_buffer_rsrc_t to = output_buffer(out + from, bytes);
  const __amdgpu_buffer_rsrc_t add = output_buffer(const_cast<float *>(ep.add ? ep.add + from : out + from), bytes);
  const __amdgpu_buffer_rsrc_t relu = output_buffer(ep.relu ? ep.relu + from : out + from, bytes);
  const __amdgpu_buffer_rsrc_t gate = output_buffer(const_cast<float *>(ep.gate ? ep.gate + from : out + from), bytes);
  const bool first = !ep.gate || ep.relu, second = ep.gate || ep.relu;   // which of the two values leave
  const int row_bytes = static_cast<int>(ldc) * 4, row0 = m + C::lane_row();
  const unsigned at = (static_cast<unsigned>(C::lane_row()) * static_cast<unsigned>(ldc) + static_cast<unsigned>(n)) * 4u;
  unsigned off[TN];
  float b[TN];
  bool masked[TN];
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    off[j] = n + j < N ? at + 4u * j : kOobOffset;
    b[j] = ep.bias && n + j < N ? ep.bias[n + j] : 0.f;
    masked[j] = ep.mask && n + j < N && ep.mask[static_cast<int64_t>(zo) * N + n + j] == 0.f;
  }
#pragma unroll
  for (int tm = 0; tm < TM; ++tm)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int step = C::step_row(tm, e), soff = step * row_bytes;
      float v[TN];
#pragma unroll
      for (int j = 0; j < TN; ++j) v[j] = ep.at(acc[tm][j][e], row0 + step, n + j, b[j], masked[j]);
      if (wide) {   // N and ldc are multiples of 4: a word lies inside its row or behind it
        if (ep.add) {
          float r[TN];
          load_words<TN>(add, off[0], soff, r);
#pragma unroll
          for (int j = 0; j < TN; ++j) v[j] += r[j];
        }
        if (first) store_words<TN>(to, off[0], soff, v);
        if (second) {
          float x[TN] = {};
          if (ep.gate) load_words<TN>(gate, off[0], soff, x);
#pragma unroll
          for (int j = 0; j < TN; ++j) v[j] = ep.second(v[j], x[j]);
          store_words<TN>(relu, off[0], soff, v);
        }
      } else {
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          if (ep.add) v[j] += __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(add, off[j] + soff, 0, 0));
          if (first) __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v[j]), to, off[j] + soff, 0, 0);
          if (second) {
            const float x = ep.gate ? __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(gate, off[j] + soff, 0, 0)) : 0.f;
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(ep.second(v[j], x)), relu, off[j] + soff, 0, 0);
          }
        }
      }
    }
}

// out[i] = what follows the sum over the S ranges' results (a bias, an addend, Relu's second result), VEC values a thread
template <int VEC>
static __global__ __launch_bounds__(256) void fold_epilogue_kernel(const float *part, float *out, int64_t n, int N, int S,
                                                                   Epilogue ep) {
  const int64_t i = (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x) * VEC;
  if (i >= n) return;
  typedef float vec __attribute__((ext_vector_type(VEC)));
  auto read = [](const float *p) { return *reinterpret_cast<const vec *>(p); };
  vec s = read(part + i);
  int z = 1;
  for (; z + 4 <= S; z += 4) {
    const vec a = read(part + z * n + i), b = read(part + (z + 1) * n + i), c = read(part + (z + 2) * n + i), d = read(part + (z + 3) * n + i);
    s += a;
    s += b;
    s += c;
    s += d;
  }
  for (; z < S; ++z) s += read(part + z * n + i);
  s *= ep.alpha;
  const int col = static_cast<int>(i % N);
  if (ep.bias) {
#pragma unroll
    for (int j = 0; j < VEC; ++j) s[j] += ep.bias[col + j];
  }
  if (ep.add) s += read(ep.add + i);
  if (!ep.gate || ep.relu) *reinterpret_cast<vec *>(out + i) = s;
  if (ep.gate || ep.relu) {
    vec x = s;
    if (ep.gate) x = read(ep.gate + i);
#pragma unroll
    for (int j = 0; j < VEC; ++j) s[j] = ep.second(s[j], x[j]);
    *reinterpret_cast<vec *>((ep.relu ? ep.relu : out) + i) = s;
  }
}

// out[i] = sum_z part[z * n + i], z ascending, four values a thread (n a multiple of 4)
static __global__ __launch_bounds__(256) void fold_splits_kernel(const f32x4 *__restrict__ part, f32x4 *__restrict__ out, int64_t n4, int S) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= n4) return;
  f32x4 s = part[i];
  int z = 1;
  for (; z + 4 <= S; z += 4) {
    const f32x4 a = part[z * n4 + i], b = part[(z + 1) * n4 + i], c = part[(z + 2) * n4 + i], d = part[(z + 3) * n4 + i];
    s += a;
    s += b;
    s += c;
    s += d;
  }
  for (; z < S; ++z) s += part[z * n4 + i];
  out[i] = s;
}

// out[i] = sum over the S ranges' results, n values apart in `part`, + add[i] where given (it may be out)
inline void launch_fold(const float *part, float *out, int64_t n, int S, hipStream_t st, const float *add = nullptr) {
  if (add) {
    const Epilogue ep{1.f, nullptr, nullptr, 0.f, 0, 0.f, add, nullptr, nullptr};
    if (n % 4 == 0 && ((reinterpret_cast<uintptr_t>(out) | reinterpret_cast<uintptr_t>(add)) & 15) == 0)
      hipLaunchKernelGGL((fold_epilogue_kernel<4>), dim3(static_cast<unsigned>((n / 4 + 255) / 256)), dim3(256), 0, st, part, out, n, 4, S, ep);
    else
      hipLaunchKernelGGL((fold_epilogue_kernel<1>), dim3(static_cast<unsigned>((n + 255) / 256)), dim3(256), 0, st, part, out, n, 1, S, ep);
    return;
  }
  if (n % 4 == 0 && (reinterpret_cast<uintptr_t>(out) & 15) == 0)
    hipLaunchKernelGGL(fold_splits_kernel, dim3(static_cast<unsigned>((n / 4 + 255) / 256)), dim3(256), 0, st,
                       reinterpret_cast<const f32x4 *>(part), reinterpret_cast<f32x4 *>(out), n / 4, S);
  else
    hipLaunchKernelGGL(mg::splitk_fold_kernel, dim3(static_cast<unsigned>((n + 255) / 256)), dim3(256), 0, st, part, out, n, n, S);
}

}  // namespace gt
}  // namespace tsplit
