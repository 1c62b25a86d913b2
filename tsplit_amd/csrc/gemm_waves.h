// Small products in one launch: the waves of a block share the depth of one small tile.
//
// A product of a few hundred rows and columns has few 64 x 64 tiles, so on the kernel of gemm_tile.h its depth was cut into ranges and a
// second launch added them; either launch takes what any launch takes, and a range of one or two steps is a chain of memory latencies
// behind one barrier each.  Here a block owns 16 TM x 16 TN of the result, its two to four waves take the ranges of the depth in turn (the tile
// kernel's own ranges: the bits of that kernel and its fold; batches in up to four, see plan_waves), 32 values at a time, operands go from
// memory to the registers the matrix instruction reads (no LDS, no barrier on the way), and the ranges' results are added through LDS in
// ascending order.  What bounds it is latency: one for the operands, one for LDS, and the launch.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "gemm_tile.h"

namespace tsplit {
namespace gw {

using gt::f32x4;
using mg::kOobOffset;
constexpr int kDeep = 32;       // of the depth at a time: whole 128-byte lines of an operand with K contiguous
constexpr int kGroups = kDeep / 16;

// What a lane supplies of one operand: index T (lane & 15) + t of tile t, k = 16 u + 4 (lane >> 4) + i of kDeep.
template <int T, bool KCONTIG>
struct Operand {
  float v[kGroups][T][4];
};

template <int T, bool KCONTIG>
struct Loader {
  __amdgpu_buffer_rsrc_t rsrc;
  unsigned voff[KCONTIG ? T : 1];
  int step;   // bytes to the next value of k
  __device__ __forceinline__ void init(const mg::DenseParams &P, int mn0) {
    const int lane = threadIdx.x & 63, at = T * (lane & 15), g = lane >> 4;
    if constexpr (KCONTIG) {
      const int left = P.mn_total - mn0;
      rsrc = gt::output_buffer(const_cast<float *>(P.p) + static_cast<int64_t>(mn0) * P.ld, (static_cast<int64_t>(left - 1) * P.ld + P.k_total) * 4);
      step = 4;
#pragma unroll
      for (int t = 0; t < T; ++t)
        voff[t] = at + t < left ? static_cast<unsigned>(at + t) * static_cast<unsigned>(P.ld) * 4u + 16u * g : kOobOffset;
    } else {
      rsrc = gt::output_buffer(const_cast<float *>(P.p), (static_cast<int64_t>(P.k_total - 1) * P.ld + P.mn_total) * 4);
      step = static_cast<int>(P.ld) * 4;
      voff[0] = mn0 + at < P.mn_total ? static_cast<unsigned>(4 * g) * static_cast<unsigned>(step) + static_cast<unsigned>(mn0 + at) * 4u : kOobOffset;
    }
  }
  __device__ __forceinline__ void load(int k0, Operand<T, KCONTIG> &o) const {
#pragma unroll
    for (int u = 0; u < kGroups; ++u)
      if constexpr (KCONTIG) {
#pragma unroll
        for (int t = 0; t < T; ++t) {
          const mg::u32x4 r = __builtin_amdgcn_raw_buffer_load_b128(rsrc, voff[t], (k0 + 16 * u) * 4, 0);
#pragma unroll
          for (int i = 0; i < 4; ++i) o.v[u][t][i] = __uint_as_float(r[i]);
        }
      } else {   // rows of k past the last one are out of range
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int soff = (k0 + 16 * u + i) * step;
          if constexpr (T == 1) {
            o.v[u][0][i] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rsrc, voff[0], soff, 0));
          } else {
            const gt::u32x2 r = __builtin_amdgcn_raw_buffer_load_b64(rsrc, voff[0], soff, 0);
            o.v[u][0][i] = __uint_as_float(r[0]);
            o.v[u][1][i] = __uint_as_float(r[1]);
          }
        }
      }
  }
  // values past the depth's end: of the next row
  static __device__ __forceinline__ void cut(int k0, int K, Operand<T, KCONTIG> &o) {
    if constexpr (KCONTIG) {
      const int g = threadIdx.x >> 4 & 3;
#pragma unroll
      for (int u = 0; u < kGroups; ++u)
#pragma unroll
        for (int t = 0; t < T; ++t)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (k0 + 16 * u + 4 * g + i >= K) o.v[u][t][i] = 0.f;
    }
  }
};

// SUMS: the blocks of the first row of tiles also leave the sums of B's columns, added as gt::Core adds them.
template <int TM, int TN, bool TA, bool TB, bool SUMS>
__global__ __launch_bounds__(256) void gemm_waves_kernel(mg::DenseParams ap, mg::DenseParams bp, float *out, int64_t ldc, gt::BatchOf zs,
                                                          gt::Epilogue ep, float *sums, bool wide, int M, int N, int K, int S, int kchunk,
                                                          mg::TileGrid tg) {
  extern __shared__ __attribute__((aligned(16))) float lds[];   // [range][tm][e][lane][tn]; with SUMS [range][16 TN] behind it
  int z, tile_m, tile_n;
  if (!mg::block_tile(tg, z, tile_m, tile_n)) return;
  const int zo = z / zs.inner, zi = z - zo * zs.inner;
  ap.p += zo * zs.ao + zi * zs.ai;
  bp.p += zo * zs.bo + zi * zs.bi;
  const int m0 = tile_m * 16 * TM, n0 = tile_n * 16 * TN;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = blockDim.x >> 6;
  Loader<TM, !TA> la;
  Loader<TN, TB> lb;
  la.init(ap, m0);
  lb.init(bp, n0);
  constexpr int kTile = 256 * TM * TN;
  typedef float vec __attribute__((ext_vector_type(TN)));
  f32x4 acc[TM][TN];
  float col[TN], some[TN];
  const bool on = SUMS && tile_m == 0;
  auto clear = [&] {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < TN; ++j) col[j] = some[j] = 0.f;
  };
  // a share of the wave's: k in [k, k + kDeep) of range r, which ends with share `end`
  struct Share {
    int k, r, end;
  };
  auto first_of = [&](int r) { return Share{r * kchunk, r, min(K, (r + 1) * kchunk)}; };
  auto behind = [&](const Share &s) { return s.k + kDeep < s.end ? Share{s.k + kDeep, s.r, s.end} : first_of(s.r + waves); };
  // last: of the wave's (the others end before the depth does)
  auto multiply = [&](const Share &s, Operand<TM, !TA> &x, Operand<TN, TB> &y, auto last) {
    if constexpr (decltype(last)::value)
      if (s.k + kDeep > K) {
        Loader<TM, !TA>::cut(s.k, K, x);
        Loader<TN, TB>::cut(s.k, K, y);
      }
    if (SUMS && (s.k - s.r * kchunk) % (8 * kDeep) == 0) {
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        col[j] += some[j];
        some[j] = 0.f;
      }
    }
#pragma unroll
    for (int u = 0; u < kGroups; ++u) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int tm = 0; tm < TM; ++tm)
#pragma unroll
          for (int tn = 0; tn < TN; ++tn) acc[tm][tn] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.v[u][tm][i], y.v[u][tn][i], acc[tm][tn], 0, 0, 0);
      if (on) {
#pragma unroll
        for (int j = 0; j < TN; ++j) some[j] += (y.v[u][j][0] + y.v[u][j][1]) + (y.v[u][j][2] + y.v[u][j][3]);
      }
    }
    if (s.k + kDeep < s.end) return;
    // the range's result
#pragma unroll
    for (int tm = 0; tm < TM; ++tm)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        vec v;
#pragma unroll
        for (int j = 0; j < TN; ++j) v[j] = acc[tm][j][e];
        *reinterpret_cast<vec *>(lds + s.r * kTile + ((tm * 4 + e) * 64 + lane) * TN) = v;
      }
    if constexpr (SUMS)
      if (on) {
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          float v = col[j] + some[j];
          v += __shfl_xor(v, 16, 64);
          v += __shfl_xor(v, 32, 64);
          if (lane < 16) lds[S * kTile + s.r * 16 * TN + TN * lane + j] = v;
        }
      }
    clear();
  };
  clear();
  Operand<TM, !TA> a[2];
  Operand<TN, TB> b[2];
  auto load = [&](const Share &s, int to) {
    la.load(s.k, a[to]);
    lb.load(s.k, b[to]);
    __builtin_amdgcn_sched_barrier(0);
  };
  auto use = [&](const Share &s, int from, auto last) {
    multiply(s, a[from], b[from], last);
    __builtin_amdgcn_sched_barrier(0);
  };
  // Two shares a turn, the next one's loads in front of either's products.  (No load under a condition of its own: where the paths meet the
  // compiler waits for as many as the shorter one has, which then are the next share's too.)
  const std::true_type yes{};
  const std::false_type no{};
  Share now = first_of(wave);
  if (now.r < S) {
    load(now, 0);
    for (;;) {
      const Share next = behind(now);
      if (next.r >= S) {
        use(now, 0, yes);
        break;
      }
      load(next, 1);
      use(now, 0, no);
      now = behind(next);
      if (now.r >= S) {
        use(next, 1, yes);
        break;
      }
      load(now, 0);
      use(next, 1, no);
    }
  }
  __syncthreads();
  if constexpr (SUMS)
    if (on && threadIdx.x < 16 * TN && n0 + static_cast<int>(threadIdx.x) < N) {
      float s = lds[S * kTile + threadIdx.x];
      for (int r = 1; r < S; ++r) s += lds[S * kTile + r * 16 * TN + threadIdx.x];
      sums[n0 + threadIdx.x] = s;
    }
  const int64_t c_at = zo * zs.co + zi * zs.ci;
  for (int q = threadIdx.x; q < TM * 256; q += blockDim.x) {
    const int l = q & 63, m = m0 + TM * (4 * (l >> 4) + (q >> 6 & 3)) + (q >> 8), n = n0 + TN * (l & 15);
    vec s = *reinterpret_cast<const vec *>(lds + q * TN);
    for (int r = 1; r < S; ++r) s += *reinterpret_cast<const vec *>(lds + r * kTile + q * TN);
    if (m >= M) continue;
    const int64_t at = c_at + m * ldc + n;
    float v[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j)
      v[j] = ep.at(s[j], m, n + j, ep.bias && n + j < N ? ep.bias[n + j] : 0.f, ep.mask && n + j < N && ep.mask[static_cast<int64_t>(zo) * N + n + j] == 0.f);
    const bool first = !ep.gate || ep.relu, second = ep.gate || ep.relu;
    if (wide && n + TN <= N) {
      vec r;
      if (ep.add) r = *reinterpret_cast<const vec *>(ep.add + at);
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        if (ep.add) v[j] += r[j];
        r[j] = v[j];
      }
      if (first) *reinterpret_cast<vec *>(out + at) = r;
      if (second) {
        vec x = r;
        if (ep.gate) x = *reinterpret_cast<const vec *>(ep.gate + at);
#pragma unroll
        for (int j = 0; j < TN; ++j) r[j] = ep.second(v[j], x[j]);
        *reinterpret_cast<vec *>((ep.relu ? ep.relu : out) + at) = r;
      }
    } else {
#pragma unroll
      for (int j = 0; j < TN; ++j)
        if (n + j < N) {
          if (ep.add) v[j] += ep.add[at + j];
          if (first) out[at + j] = v[j];
          if (second) (ep.relu ? ep.relu : out)[at + j] = ep.second(v[j], ep.gate ? ep.gate[at + j] : v[j]);
        }
    }
  }
}

}  // namespace gw
}  // namespace tsplit
