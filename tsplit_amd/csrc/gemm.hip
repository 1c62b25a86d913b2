// DLGpuMatrixMultiply and DLGpuBatchMatrixMultiply: row-major C = op(A) op(B) on the fp32 MFMA
// tile kernel of gemm_tile.h.
//
// The four transpose combinations only change which way each operand is staged (a transposed
// operand is simply one whose other index is contiguous); nothing is ever transposed in memory.
// The tile (128x128, 64x128, 128x64 or 64x64) and the number of ranges K is cut into come from a
// small model of the chip (tile_plan.h); the ranges' results are added in ascending order by a
// second kernel.  Small products run on the kernel of gemm_waves.h, in one launch.  The batched form runs every leading index
// as one more grid dimension of the same kernel.  Operands of 2 GiB and more, and results whose 64 rows reach that far, stay on the engine
// of mfma_gemm.h, which takes 64-bit addresses, with its own tiles and ranges.
#include <algorithm>

#include "common.h"
#include "gemm_tile.h"
#include "mfma_gemm.h"
#include "gemm_split.h"
#include "gemm_waves.h"
#include "tile_plan.h"

namespace tsplit {
namespace {

using namespace mg;

// stored rows of an operand: (M or N, K) by (transposed or not)
inline int64_t stored_rows(bool k_rows, int mn, int K) { return k_rows ? K : mn; }

struct Plan {
  int tile, S, kchunk;
  WavesPlan waves;   // with waves: one launch of gemm_waves.h instead, S is 1
};

Plan best_plan(int M, int N, int K, int batch, bool may_split) {
  const int64_t cols = N;
  const int steps = std::max(1, (K + gt::BK - 1) / gt::BK);
  const TilePlan t = plan_tiles(M, &cols, &steps, 1, batch, may_split ? 64 : 1, static_cast<double>(M) * N, kProductCost);
  const WavesPlan waves = plan_waves(M, N, K, batch, t, !may_split);
  if (waves.waves) return {0, 1, waves.kchunk, waves};
  Plan p{t.tile, 1, (steps + t.S - 1) / t.S * gt::BK, waves};
  p.S = std::max(1, (K + p.kchunk - 1) / p.kchunk);
  if (p.S == 1) p.kchunk = K;
  return p;
}

// the plans of the shapes this thread asked for last (working one out takes about 2 us of host time)
Plan plan_product(int M, int N, int K, int batch, bool may_split) {
  struct Entry {
    int M, N, K, batch;
    bool may_split;
    Plan plan;
  };
  static thread_local Entry known[256] = {};
  // (multiplied through: sums of small multiples put every shape of a net of power-of-two sizes into two places)
  const unsigned mix = ((static_cast<unsigned>(M) * 31u + static_cast<unsigned>(N)) * 31u + static_cast<unsigned>(K)) * 31u + static_cast<unsigned>(batch);
  Entry &e = known[(mix * 2654435769u) >> 24];
  if (e.M != M || e.N != N || e.K != K || e.batch != batch || e.may_split != may_split) e = {M, N, K, batch, may_split, best_plan(M, N, K, batch, may_split)};
  return e.plan;
}

template <int TM, int TN, bool TA, bool TB>
void launch_tile(const float *A, int64_t lda, int64_t sa, const float *B, int64_t ldb, int64_t sb, float *out, int64_t sc, int batch, int M,
                 int N, int K, const Plan &plan, hipStream_t s) {
  using T = gt::Tile<TM, TN, 2, 2, TA, TB>;
  const int tm = (M + T::BM - 1) / T::BM, tn = (N + T::BN - 1) / T::BN, z = plan.S > 1 ? plan.S : batch;
  const bool wide = N % 4 == 0 && sc % 4 == 0 && aligned16(out);
  hipLaunchKernelGGL((gt::gemm_tile_kernel<TM, TN, 2, 2, TA, TB>), dim3(grid_blocks(tm, tn, z)), dim3(gt::kThreads), 0, s,
                     DenseParams{A, lda, M, K}, DenseParams{B, ldb, N, K}, out, gt::Strides{sa, sb, sc}, wide, M, N, K, plan.kchunk,
                     TileGrid{tm, tn, tm * tn * z});
}

template <bool TA, bool TB>
void launch_planned(const float *A, int64_t lda, int64_t sa, const float *B, int64_t ldb, int64_t sb, float *out, int64_t sc, int batch, int M,
                    int N, int K, const Plan &plan, hipStream_t s) {
  switch (plan.tile) {
    case 0: return launch_tile<4, 4, TA, TB>(A, lda, sa, B, ldb, sb, out, sc, batch, M, N, K, plan, s);
    case 1: return launch_tile<2, 4, TA, TB>(A, lda, sa, B, ldb, sb, out, sc, batch, M, N, K, plan, s);
    case 2: return launch_tile<4, 2, TA, TB>(A, lda, sa, B, ldb, sb, out, sc, batch, M, N, K, plan, s);
    default: return launch_tile<2, 2, TA, TB>(A, lda, sa, B, ldb, sb, out, sc, batch, M, N, K, plan, s);
  }
}

// the same tiles with something behind the products (S = 1)
template <int TM, int TN, bool TA, bool TB>
void launch_epilogue_tile(const float *A, int64_t lda, const float *B, int64_t ldb, float *out, int64_t ldc, const gt::BatchOf &zs, int batch, int M,
                          int N, int K, const gt::Epilogue &ep, hipStream_t s) {
  using T = gt::Tile<TM, TN, 2, 2, TA, TB>;
  const int tm = (M + T::BM - 1) / T::BM, tn = (N + T::BN - 1) / T::BN;
  const bool wide = N % 4 == 0 && ldc % 4 == 0 && zs.co % 4 == 0 && zs.ci % 4 == 0 && aligned16(out) && aligned16(ep.add) && aligned16(ep.relu) && aligned16(ep.gate);
  hipLaunchKernelGGL((gt::gemm_epilogue_kernel<TM, TN, TA, TB>), dim3(grid_blocks(tm, tn, batch)), dim3(gt::kThreads), 0, s, DenseParams{A, lda, M, K},
                     DenseParams{B, ldb, N, K}, out, ldc, zs, ep, wide, M, N, K, TileGrid{tm, tn, tm * tn * batch});
}

template <bool TA, bool TB>
void launch_epilogue(int tile, const float *A, int64_t lda, const float *B, int64_t ldb, float *out, int64_t ldc, const gt::BatchOf &zs, int batch,
                     int M, int N, int K, const gt::Epilogue &ep, hipStream_t s) {
  switch (tile) {
    case 0: return launch_epilogue_tile<4, 4, TA, TB>(A, lda, B, ldb, out, ldc, zs, batch, M, N, K, ep, s);
    case 1: return launch_epilogue_tile<2, 4, TA, TB>(A, lda, B, ldb, out, ldc, zs, batch, M, N, K, ep, s);
    case 2: return launch_epilogue_tile<4, 2, TA, TB>(A, lda, B, ldb, out, ldc, zs, batch, M, N, K, ep, s);
    default: return launch_epilogue_tile<2, 2, TA, TB>(A, lda, B, ldb, out, ldc, zs, batch, M, N, K, ep, s);
  }
}

constexpr gt::Epilogue kNothingMore{1.f, nullptr, nullptr, 0.f, 0, 0.f, nullptr, nullptr, nullptr};
constexpr gt::BatchOf kOneProduct{1, 0, 0, 0, 0, 0, 0};

// small products: the depth shared by the waves of a block (gemm_waves.h)
template <int TM, int TN, bool TA, bool TB, bool SUMS>
void launch_waves_tile(const float *A, int64_t lda, const float *B, int64_t ldb, float *out, int64_t ldc, const gt::BatchOf &zs, int batch, int M, int N,
                       int K, const gt::Epilogue &ep, float *sums, const WavesPlan &p, hipStream_t s) {
  const int tm = (M + 16 * TM - 1) / (16 * TM), tn = (N + 16 * TN - 1) / (16 * TN);
  const bool wide = TN > 1 && N % 2 == 0 && ldc % 2 == 0 && zs.co % 2 == 0 && zs.ci % 2 == 0 && aligned16(out) && aligned16(ep.add) &&
                    aligned16(ep.relu) && aligned16(ep.gate);
  const size_t lds = static_cast<size_t>(p.S) * (256 * TM * TN + (SUMS ? 16 * TN : 0)) * sizeof(float);
  hipLaunchKernelGGL((gw::gemm_waves_kernel<TM, TN, TA, TB, SUMS>), dim3(grid_blocks(tm, tn, batch)), dim3(64 * p.waves), lds, s, DenseParams{A, lda, M, K},
                     DenseParams{B, ldb, N, K}, out, ldc, zs, ep, sums, wide, M, N, K, p.S, p.kchunk, TileGrid{tm, tn, tm * tn * batch});
}
template <bool TA, bool TB, bool SUMS = false>
void launch_waves(const WavesPlan &p, const float *A, int64_t lda, const float *B, int64_t ldb, float *out, int64_t ldc, const gt::BatchOf &zs, int batch,
                  int M, int N, int K, const gt::Epilogue &ep, float *sums, hipStream_t s) {
  switch (p.tile) {
    case 0: return launch_waves_tile<1, 1, TA, TB, SUMS>(A, lda, B, ldb, out, ldc, zs, batch, M, N, K, ep, sums, p, s);
    case 1: return launch_waves_tile<1, 2, TA, TB, SUMS>(A, lda, B, ldb, out, ldc, zs, batch, M, N, K, ep, sums, p, s);
    case 2: return launch_waves_tile<2, 1, TA, TB, SUMS>(A, lda, B, ldb, out, ldc, zs, batch, M, N, K, ep, sums, p, s);
    default: return launch_waves_tile<2, 2, TA, TB, SUMS>(A, lda, B, ldb, out, ldc, zs, batch, M, N, K, ep, sums, p, s);
  }
}

// the results of S ranges (or of one) summed, with what follows
int launch_epilogue_fold(const float *part, float *out, int64_t mn, int N, int S, const gt::Epilogue &ep, hipStream_t s) {
  if (N % 4 == 0 && aligned16(part) && aligned16(out) && aligned16(ep.add) && aligned16(ep.relu) && aligned16(ep.gate))
    hipLaunchKernelGGL(gt::fold_epilogue_kernel<4>, dim3(static_cast<unsigned>((mn / 4 + 255) / 256)), dim3(256), 0, s, part, out, mn, N, S, ep);
  else
    hipLaunchKernelGGL(gt::fold_epilogue_kernel<1>, dim3(static_cast<unsigned>((mn + 255) / 256)), dim3(256), 0, s, part, out, mn, N, S, ep);
  return 0;
}

template <bool TA, bool TB>
int launch_product(const float *A, int64_t lda, const float *B, int64_t ldb, float *C, int M, int N, int K, hipStream_t s, int64_t *ws_elems) {
  const Plan plan = plan_product(M, N, K, 1, true);
  if (plan.waves.waves) {
    launch_waves<TA, TB>(plan.waves, A, lda, B, ldb, C, N, kOneProduct, 1, M, N, K, kNothingMore, nullptr, s);
    return 0;
  }
  const int64_t mn = static_cast<int64_t>(M) * N;
  float *out = C;
  if (plan.S > 1) {
    out = static_cast<float *>(scratch_get(s, 2, static_cast<size_t>(plan.S) * mn * 4));
    TS_REQUIRE(out, "DLGpuMatrixMultiply: no scratch memory for split-K");
    *ws_elems = plan.S * mn;
  }
  launch_planned<TA, TB>(A, lda, 0, B, ldb, 0, out, mn, 1, M, N, K, plan, s);
  if (plan.S > 1) gt::launch_fold(out, C, mn, plan.S, s);
  return 0;
}

// C = A^T B and the column sums of B, in ranges of up to kSumsRange rows: on either kernel a lane's sums of a range are a chain of a
// rounding every 256 rows (the same bits), the reduction's are cut finer the more rows there are.  Error of the sums against float64 (normal values, as a share of
// the root of the rows) in ranges of 11 K rows 1.6e-7, as a reduction 2.4e-7; of 33 K 2.3 and 2.2, of 87 K 3.7 and 3.1.  Nor is there time to be
// gained beyond: 262144 x 1024 and 1024 columns 4145 us, as two calls 4029.
constexpr int kSumsRange = 16384;
template <int TM, int TN>
void launch_sums_tile(const float *A, int64_t lda, const float *B, int64_t ldb, float *out, float *sums, int64_t zs, int M, int N, int K,
                      const Plan &plan, hipStream_t s) {
  using T = gt::Tile<TM, TN, 2, 2, true, false>;
  const int tm = (M + T::BM - 1) / T::BM, tn = (N + T::BN - 1) / T::BN;
  const bool wide = N % 4 == 0 && zs % 4 == 0 && aligned16(out);
  hipLaunchKernelGGL((gt::gemm_sums_kernel<TM, TN>), dim3(grid_blocks(tm, tn, plan.S)), dim3(gt::kThreads), 0, s, DenseParams{A, lda, M, K},
                     DenseParams{B, ldb, N, K}, out, sums, zs, wide, M, N, K, plan.kchunk, TileGrid{tm, tn, tm * tn * plan.S});
}
int launch_sums(const float *A, int64_t lda, const float *B, int64_t ldb, float *C, float *sums, int M, int N, int K, hipStream_t s) {
  const Plan plan = plan_product(M, N, K, 1, true);
  if (plan.waves.waves) {
    launch_waves<true, false, true>(plan.waves, A, lda, B, ldb, C, N, kOneProduct, 1, M, N, K, kNothingMore, sums, s);
    return 0;
  }
  const int64_t mn = static_cast<int64_t>(M) * N, n = mn + N;
  float *out = C, *to = sums;
  if (plan.S > 1) {
    out = static_cast<float *>(scratch_get(s, 2, static_cast<size_t>(plan.S) * n * 4));
    TS_REQUIRE(out, "TSplit_MatrixMultiplySums: no scratch memory for split-K");
    to = out + mn;
  }
  const int64_t zs = plan.S > 1 ? n : 0;
  switch (plan.tile) {
    case 0: launch_sums_tile<4, 4>(A, lda, B, ldb, out, to, zs, M, N, K, plan, s); break;
    case 1: launch_sums_tile<2, 4>(A, lda, B, ldb, out, to, zs, M, N, K, plan, s); break;
    case 2: launch_sums_tile<4, 2>(A, lda, B, ldb, out, to, zs, M, N, K, plan, s); break;
    default: launch_sums_tile<2, 2>(A, lda, B, ldb, out, to, zs, M, N, K, plan, s); break;
  }
  if (plan.S > 1) {
    const int vec = N % 4 == 0 && aligned16(C) && aligned16(sums) ? 4 : 1;
    hipLaunchKernelGGL((vec == 4 ? gt::fold_two_kernel<4> : gt::fold_two_kernel<1>), dim3(static_cast<unsigned>((n / vec + 255) / 256)), dim3(256), 0, s,
                       out, C, sums, mn, n, plan.S);
  }
  return 0;
}

// operands or rows of the result beyond 32-bit offsets: the loaders with 64-bit addresses
template <int BM, int BN, bool TA, bool TB>
struct Far {
  using AL = typename std::conditional<TA, MnContigLoader<BM>, KContigLoader<BM>>::type;
  using BL = typename std::conditional<TB, KContigLoader<BN>, MnContigLoader<BN>>::type;
  typename AL::Params ap;
  typename BL::Params bp;
  int tm, tn;
  Far(const float *A, int64_t lda, int64_t sa, const float *B, int64_t ldb, int64_t sb, int M, int N)
      : ap{A, lda, M, lda % 4 == 0 && sa % 4 == 0 && aligned16(A)},
        bp{B, ldb, N, ldb % 4 == 0 && sb % 4 == 0 && aligned16(B)},
        tm((M + BM - 1) / BM),
        tn((N + BN - 1) / BN) {}
};

// K in ranges where the tiles alone leave the chip idle (512 x 512 over 1.1 million rows is 16 tiles: 5.2 ms in ranges, 101 whole)
template <int BM, int BN, int WM, int WN, bool TA, bool TB>
int launch_far(const float *A, int64_t lda, const float *B, int64_t ldb, float *C, int M, int N, int K, hipStream_t s, int64_t *ws_elems) {
  using F = Far<BM, BN, TA, TB>;
  const F f(A, lda, 0, B, ldb, 0, M, N);
  static const int occ = blocks_per_cu(mfma_gemm_kernel<BM, BN, WM, WN, typename F::AL, typename F::BL, RowMajorCols>);
  int S, kchunk;
  plan_splitk(f.tm * f.tn, K, 64, occ, S, kchunk);
  float *out = C;
  const int64_t mn = static_cast<int64_t>(M) * N;
  if (S > 1) {
    out = static_cast<float *>(scratch_get(s, 2, static_cast<size_t>(S) * mn * 4));
    TS_REQUIRE(out, "DLGpuMatrixMultiply: no scratch memory for split-K");
    *ws_elems = S * mn;
  }
  hipLaunchKernelGGL((mfma_gemm_kernel<BM, BN, WM, WN, typename F::AL, typename F::BL, RowMajorCols>), dim3(grid_blocks(f.tm, f.tn, S)),
                     dim3(kThreads), 0, s, f.ap, f.bp, out, mn, static_cast<int64_t>(N), RowMajorCols{}, M, N, K, kchunk,
                     TileGrid{f.tm, f.tn, f.tm * f.tn * S});
  if (S > 1) gt::launch_fold(out, C, mn, S, s);
  return 0;
}

template <int BM, int BN, int WM, int WN, bool TA, bool TB>
int launch_far_batched(const float *A, int64_t lda, int64_t sa, const float *B, int64_t ldb, int64_t sb, float *C, int batch, int M, int N,
                       int K, hipStream_t s) {
  using F = Far<BM, BN, TA, TB>;
  const F f(A, lda, sa, B, ldb, sb, M, N);
  hipLaunchKernelGGL((mfma_batched_gemm_kernel<BM, BN, WM, WN, typename F::AL, typename F::BL>), dim3(grid_blocks(f.tm, f.tn, batch)),
                     dim3(kThreads), 0, s, f.ap, f.bp, C, sa, sb, static_cast<int64_t>(M) * N, M, N, K, TileGrid{f.tm, f.tn, f.tm * f.tn * batch});
  return 0;
}

template <bool TA, bool TB>
int dispatch_far(const float *A, int64_t lda, const float *B, int64_t ldb, float *C, int M, int N, int K, hipStream_t s, int64_t *ws) {
  if (M <= 64) return launch_far<64, 256, 1, 4, TA, TB>(A, lda, B, ldb, C, M, N, K, s, ws);
  return launch_far<128, 128, 2, 2, TA, TB>(A, lda, B, ldb, C, M, N, K, s, ws);
}

// the same product with split-bf16 terms (opt-in): 128 x 128 tiles whatever M, the split-K plan and fold of above
template <bool TA, bool TB>
int launch_gemm_split(const float *A, int64_t lda, const float *B, int64_t ldb, float *C, int M, int N, int K,
                      hipStream_t s, int64_t *ws_elems) {
  using AL = typename std::conditional<TA, SplitMnContigLoader, SplitKContigLoader>::type;
  using BL = typename std::conditional<TB, SplitKContigLoader, SplitMnContigLoader>::type;
  const typename AL::Params ap{A, lda, M, K};
  const typename BL::Params bp{B, ldb, N, K};
  const int tm = (M + 127) / 128, tn = (N + 127) / 128;
  int S, kchunk;
  plan_splitk(tm * tn, K, 64, 3, S, kchunk);
  float *out = C;
  const int64_t mn = static_cast<int64_t>(M) * N;
  if (S > 1) {
    out = static_cast<float *>(scratch_get(s, 2, static_cast<size_t>(S) * mn * 4));
    TS_REQUIRE(out, "DLGpuMatrixMultiply: no scratch memory for split-K");
    *ws_elems = S * mn;
  }
  hipLaunchKernelGGL((mfma_gemm_split_kernel<AL, BL>), dim3(grid_blocks(tm, tn, S)), dim3(kThreads), 0, s, ap, bp, out, mn,
                     M, N, K, kchunk, TileGrid{tm, tn, tm * tn * S});
  if (S > 1) gt::launch_fold(out, C, mn, S, s);
  return 0;
}

// both operands within reach of 32-bit byte offsets
template <bool TA, bool TB>
bool near(int64_t lda, int64_t ldb, int M, int N, int K) {
  return K < (1 << 29) && dense_fits_buffer(stored_rows(TA, M, K), lda, 128) && dense_fits_buffer(stored_rows(!TB, N, K), ldb, 128);
}

// a wave stores its 64 rows of the result, and the columns of one more, by 32-bit byte offsets
bool rows_reach(int N) { return 65ll * 4 * N < (1ll << 31); }

template <bool TA, bool TB>
int dispatch_product(const float *A, int64_t lda, const float *B, int64_t ldb, float *C, int M, int N, int K, hipStream_t s, int64_t *ws) {
  if (!near<TA, TB>(lda, ldb, M, N, K)) return dispatch_far<TA, TB>(A, lda, B, ldb, C, M, N, K, s, ws);
  // split-bf16 products where asked for: K a multiple of 4 (a loaded word lies inside a row or outside it)
  if (split_bf16_enabled() && K % 4 == 0 && K >= BK) return launch_gemm_split<TA, TB>(A, lda, B, ldb, C, M, N, K, s, ws);
  if (!rows_reach(N)) return dispatch_far<TA, TB>(A, lda, B, ldb, C, M, N, K, s, ws);
  return launch_product<TA, TB>(A, lda, B, ldb, C, M, N, K, s, ws);
}

// A product with something behind it: on the tile kernel in one launch, or, where K is cut into ranges, in the launch that adds them up.
// Operands that other kernels take (beyond 32-bit offsets, split-bf16) are multiplied there and the rest follows by a pass over the result.
template <bool TA, bool TB>
int dispatch_epilogue(const float *A, int64_t lda, const float *B, int64_t ldb, float *C, int M, int N, int K, const gt::Epilogue &ep, hipStream_t s) {
  const int64_t mn = static_cast<int64_t>(M) * N;
  if (near<TA, TB>(lda, ldb, M, N, K) && rows_reach(N) && !(split_bf16_enabled() && K % 4 == 0 && K >= BK)) {
    const Plan plan = plan_product(M, N, K, 1, true);
    if (plan.waves.waves) {
      launch_waves<TA, TB>(plan.waves, A, lda, B, ldb, C, N, kOneProduct, 1, M, N, K, ep, nullptr, s);
      return 0;
    }
    if (plan.S == 1) {
      launch_epilogue<TA, TB>(plan.tile, A, lda, B, ldb, C, N, kOneProduct, 1, M, N, K, ep, s);
      return 0;
    }
    float *part = static_cast<float *>(scratch_get(s, 2, static_cast<size_t>(plan.S) * mn * 4));
    TS_REQUIRE(part, "TSplit_MatrixMultiplyAdd: no scratch memory for split-K");
    launch_planned<TA, TB>(A, lda, 0, B, ldb, 0, part, mn, 1, M, N, K, plan, s);
    return launch_epilogue_fold(part, C, mn, N, plan.S, ep, s);
  }
  int64_t ws = 0;
  float *product = C;
  if (ep.add == C) {   // read by the pass behind the product
    product = static_cast<float *>(scratch_get(s, 3, static_cast<size_t>(mn) * 4));
    TS_REQUIRE(product, "TSplit_MatrixMultiplyAdd: no scratch memory for the product");
  }
  if (const int rc = dispatch_product<TA, TB>(A, lda, B, ldb, product, M, N, K, s, &ws)) return rc;
  return launch_epilogue_fold(product, C, mn, N, 1, ep, s);
}

template <bool TA, bool TB>
int dispatch_batched(const float *A, int64_t lda, int64_t sa, const float *B, int64_t ldb, int64_t sb, float *C,
                     int batch, int M, int N, int K, hipStream_t s) {
  const int64_t tiles = static_cast<int64_t>((M + 63) / 64) * ((N + 63) / 64) * batch;
  TS_REQUIRE(tiles < (1ll << 31) - 8, "DLGpuBatchMatrixMultiply: too many tiles");
  if (!near<TA, TB>(lda, ldb, M, N, K) || !rows_reach(N)) {   // (batches of 1.1M x 64 x 512 on 256 x 64 tiles 0.79 ms, on 128 x 128 0.92)
    if (M <= 64) return launch_far_batched<64, 256, 1, 4, TA, TB>(A, lda, sa, B, ldb, sb, C, batch, M, N, K, s);
    if (N <= 64) return launch_far_batched<256, 64, 4, 1, TA, TB>(A, lda, sa, B, ldb, sb, C, batch, M, N, K, s);
    return launch_far_batched<128, 128, 2, 2, TA, TB>(A, lda, sa, B, ldb, sb, C, batch, M, N, K, s);
  }
  const Plan plan = plan_product(M, N, K, batch, false);
  if (plan.waves.waves) {
    launch_waves<TA, TB>(plan.waves, A, lda, B, ldb, C, N, gt::BatchOf{1, sa, 0, sb, 0, static_cast<int64_t>(M) * N, 0}, batch, M, N, K, kNothingMore, nullptr, s);
    return 0;
  }
  launch_planned<TA, TB>(A, lda, sa, B, ldb, sb, C, static_cast<int64_t>(M) * N, batch, M, N, K, plan, s);
  return 0;
}

// an array as a matrix of its last axis' columns
void rows_by_cols(const DLArray *a, int64_t &rows, int64_t &cols) {
  rows = 1;
  for (int d = 0; d + 1 < a->ndim; ++d) rows *= a->shape[d];
  cols = a->shape[a->ndim - 1];
}

// One operand or result of a product over heads: [n, heads, rows, cols], or [n, rows, heads * cols] with a head's columns side by side
struct HeadArray {
  float *p;
  int64_t n, rows, cols, ld, outer, inner;
};
bool head_array(const DLArray *a, int heads, HeadArray &h) {
  const int64_t *s = a->shape;
  if (a->ndim == 4 && s[1] == heads)
    h = {static_cast<float *>(a->data), s[0], s[2], s[3], s[3], s[1] * s[2] * s[3], s[2] * s[3]};
  else if (a->ndim == 3 && s[2] % heads == 0)
    h = {static_cast<float *>(a->data), s[0], s[1], s[2] / heads, s[2], s[1] * s[2], s[2] / heads};
  else
    return false;
  return true;
}

template <bool TA, bool TB>
int dispatch_heads(const HeadArray &a, const HeadArray &b, const HeadArray &c, int heads, int M, int N, int K, const gt::Epilogue &ep, hipStream_t s) {
  TS_REQUIRE((near<TA, TB>(a.ld, b.ld, M, N, K) && 65ll * 4 * c.ld < (1ll << 31)),
             "TSplit_HeadsMatrixMultiply: a matrix reaches beyond 32-bit byte offsets");
  const int batch = static_cast<int>(c.n) * heads;
  const Plan plan = plan_product(M, N, K, batch, false);
  const gt::BatchOf zs{heads, a.outer, a.inner, b.outer, b.inner, c.outer, c.inner};
  if (plan.waves.waves)
    launch_waves<TA, TB>(plan.waves, a.p, a.ld, b.p, b.ld, c.p, c.ld, zs, batch, M, N, K, ep, nullptr, s);
  else
    launch_epilogue<TA, TB>(plan.tile, a.p, a.ld, b.p, b.ld, c.p, c.ld, zs, batch, M, N, K, ep, s);
  return 0;
}

}  // namespace
}  // namespace tsplit

using namespace tsplit;

extern "C" int TSplit_MatrixMultiplyAdd(const DLArrayHandle matA, int transposeA, const DLArrayHandle matB, int transposeB,
                                        const DLArrayHandle bias, const DLArrayHandle addend, const DLArrayHandle gate, DLArrayHandle matC,
                                        DLArrayHandle relu, DLStreamHandle stream_handle) {
  const char *who = "TSplit_MatrixMultiplyAdd";
  TS_REQUIRE(matA && matB && matC, "%s: NULL array", who);
  TS_REQUIRE(matA->ndim >= 2 && matB->ndim >= 2 && matC->ndim >= 2, "%s: arrays of two axes or more only", who);
  int64_t a_rows, lda, b_rows, ldb, M, N;
  rows_by_cols(matA, a_rows, lda);
  rows_by_cols(matB, b_rows, ldb);
  rows_by_cols(matC, M, N);
  const int64_t K = transposeA ? a_rows : lda;
  TS_REQUIRE((transposeA ? lda : a_rows) == M && (transposeB ? b_rows : ldb) == N && (transposeB ? ldb : b_rows) == K, "%s: shapes do not conform",
             who);
  TS_REQUIRE(M < (1ll << 31) && N < (1ll << 31) && K < (1ll << 31) - 64, "%s: dimension too large", who);
  TS_REQUIRE(!bias || numel(bias) == N, "%s: the bias has %lld values for %lld columns", who, (long long)(bias ? numel(bias) : 0), (long long)N);
  TS_REQUIRE(!addend || numel(addend) == M * N, "%s: the addend is of the result's size", who);
  TS_REQUIRE(!relu || (numel(relu) == M * N && relu->data != matC->data), "%s: Relu's result is another array of the result's size", who);
  TS_REQUIRE(!gate || (numel(gate) == M * N && gate->data != matC->data && (!relu || gate->data != relu->data)),
             "%s: the gate is another array of the result's size", who);
  hipStream_t s = stream_of(stream_handle);
  ProfileScope ps(nullptr, s, 0, 0, 0);
  int rc = 0;
  if (M > 0 && N > 0) {
    const float *A = static_cast<const float *>(matA->data), *B = static_cast<const float *>(matB->data);
    float *C = static_cast<float *>(matC->data);
    const int m = static_cast<int>(M), n = static_cast<int>(N), k = static_cast<int>(K);
    const gt::Epilogue ep{1.f, bias ? static_cast<const float *>(bias->data) : nullptr, nullptr, 0.f, 0, 0.f,
                          addend ? static_cast<const float *>(addend->data) : nullptr, relu ? static_cast<float *>(relu->data) : nullptr,
                          gate ? static_cast<const float *>(gate->data) : nullptr};
    if (!transposeA && !transposeB) rc = dispatch_epilogue<false, false>(A, lda, B, ldb, C, m, n, k, ep, s);
    if (!transposeA && transposeB) rc = dispatch_epilogue<false, true>(A, lda, B, ldb, C, m, n, k, ep, s);
    if (transposeA && !transposeB) rc = dispatch_epilogue<true, false>(A, lda, B, ldb, C, m, n, k, ep, s);
    if (transposeA && transposeB) rc = dispatch_epilogue<true, true>(A, lda, B, ldb, C, m, n, k, ep, s);
  }
  if (rc) return rc;
  return ps.finish();
}

extern "C" int TSplit_MatrixMultiplySums(const DLArrayHandle matA, const DLArrayHandle matB, DLArrayHandle matC, DLArrayHandle sums,
                                         DLStreamHandle stream_handle) {
  const char *who = "TSplit_MatrixMultiplySums";
  TS_REQUIRE(matA && matB && matC && sums, "%s: NULL array", who);
  TS_REQUIRE(matA->ndim >= 2 && matB->ndim >= 2 && matC->ndim == 2, "%s: operands of two axes or more, a result of two", who);
  int64_t K, lda, b_rows, ldb;
  rows_by_cols(matA, K, lda);
  rows_by_cols(matB, b_rows, ldb);
  const int64_t M = matC->shape[0], N = matC->shape[1];
  TS_REQUIRE(K == b_rows && lda == M && ldb == N && numel(sums) == N, "%s: shapes do not conform", who);
  TS_REQUIRE(M < (1ll << 31) && N < (1ll << 31) && K < (1ll << 31) - 64, "%s: dimension too large", who);
  const int m = static_cast<int>(M), n = static_cast<int>(N), k = static_cast<int>(K);
  const bool here = M > 0 && N > 0 && K > 0 && near<true, false>(lda, ldb, m, n, k) && rows_reach(n) && !(split_bf16_enabled() && K % 4 == 0 && K >= BK) &&
                    plan_product(m, n, k, 1, true).kchunk <= kSumsRange;
  if (!here) {   // the product by itself, on whichever kernel takes it, and the sums by themselves
    int64_t ashape[2] = {K, M}, bshape[2] = {K, N};
    DLArray A{matA->data, matA->ctx, 2, ashape}, B{matB->data, matB->ctx, 2, bshape};
    if (const int rc = DLGpuMatrixMultiply(&A, true, &B, false, matC, stream_handle, nullptr)) return rc;
    return DLGpuReduceSumAxisZero(&B, sums, stream_handle, nullptr);
  }
  hipStream_t s = stream_of(stream_handle);
  ProfileScope ps(nullptr, s, 0, 0, 0);
  if (const int rc = launch_sums(static_cast<const float *>(matA->data), lda, static_cast<const float *>(matB->data), ldb,
                                 static_cast<float *>(matC->data), static_cast<float *>(sums->data), m, n, k, s))
    return rc;
  return ps.finish();
}

extern "C" int TSplit_HeadsMatrixMultiply(const DLArrayHandle matA, int transposeA, const DLArrayHandle matB, int transposeB, DLArrayHandle matC,
                                          int heads, float alpha, const DLArrayHandle mask, float mask_value, int causal, float fill,
                                          const DLArrayHandle addend, DLStreamHandle stream_handle) {
  const char *who = "TSplit_HeadsMatrixMultiply";
  TS_REQUIRE(matA && matB && matC, "%s: NULL array", who);
  HeadArray a, b, c;
  TS_REQUIRE(heads > 0 && head_array(matA, heads, a) && head_array(matB, heads, b) && head_array(matC, heads, c),
             "%s: arrays are [n, heads, rows, columns] or [n, rows, heads * columns]", who);
  const int64_t M = c.rows, N = c.cols, K = transposeA ? a.rows : a.cols;
  TS_REQUIRE(a.n == c.n && b.n == c.n && (transposeA ? a.cols : a.rows) == M && (transposeB ? b.rows : b.cols) == N &&
                 (transposeB ? b.cols : b.rows) == K,
             "%s: shapes do not conform", who);
  TS_REQUIRE(M < (1ll << 31) && N < (1ll << 31) && K < (1ll << 31) - 64, "%s: dimension too large", who);
  TS_REQUIRE((M + 63) / 64 * ((N + 63) / 64) < (1ll << 31) / heads && c.n <= ((1ll << 31) - 9) / heads / ((M + 63) / 64 * ((N + 63) / 64) + 1),
             "%s: too many tiles", who);
  TS_REQUIRE(!mask || numel(mask) == c.n * N, "%s: the mask has a value for every column of every n", who);
  TS_REQUIRE(!addend || (addend->ndim == matC->ndim && numel(addend) == numel(matC) && addend->data != matC->data),
             "%s: the addend is another array of the result's layout", who);
  hipStream_t s = stream_of(stream_handle);
  ProfileScope ps(nullptr, s, 0, 0, 0);
  int rc = 0;
  if (M > 0 && N > 0 && c.n > 0) {
    const int m = static_cast<int>(M), n = static_cast<int>(N), k = static_cast<int>(K);
    const gt::Epilogue ep{alpha, nullptr, mask ? static_cast<const float *>(mask->data) : nullptr, mask_value, causal, fill,
                          addend ? static_cast<const float *>(addend->data) : nullptr, nullptr, nullptr};
    if (!transposeA && !transposeB) rc = dispatch_heads<false, false>(a, b, c, heads, m, n, k, ep, s);
    if (!transposeA && transposeB) rc = dispatch_heads<false, true>(a, b, c, heads, m, n, k, ep, s);
    if (transposeA && !transposeB) rc = dispatch_heads<true, false>(a, b, c, heads, m, n, k, ep, s);
    if (transposeA && transposeB) rc = dispatch_heads<true, true>(a, b, c, heads, m, n, k, ep, s);
  }
  if (rc) return rc;
  return ps.finish();
}

extern "C" int DLGpuMatrixMultiply(const DLArrayHandle matA, bool transposeA, const DLArrayHandle matB,
                                   bool transposeB, DLArrayHandle matC, DLStreamHandle stream_handle,
                                   ProfilerHandle p) {
  TS_REQUIRE(matA && matB && matC, "DLGpuMatrixMultiply: NULL array");
  TS_REQUIRE(matA->ndim == 2 && matB->ndim == 2 && matC->ndim == 2, "DLGpuMatrixMultiply: 2-D arrays only");
  const int64_t M = matC->shape[0], N = matC->shape[1];
  const int64_t K = transposeA ? matA->shape[0] : matA->shape[1];
  const int64_t Am = transposeA ? matA->shape[1] : matA->shape[0];
  const int64_t Bk = transposeB ? matB->shape[1] : matB->shape[0];
  const int64_t Bn = transposeB ? matB->shape[0] : matB->shape[1];
  TS_REQUIRE(Am == M && Bn == N && Bk == K, "DLGpuMatrixMultiply: shapes do not conform: op(A) %lldx%lld, op(B) %lldx%lld, C %lldx%lld",
             (long long)Am, (long long)K, (long long)Bk, (long long)Bn, (long long)M, (long long)N);
  TS_REQUIRE(M < (1ll << 31) && N < (1ll << 31) && K < (1ll << 31) - 64, "DLGpuMatrixMultiply: dimension too large");
  hipStream_t s = stream_of(stream_handle);
  int64_t ws = 0;
  ProfileScope ps(p, s, numel(matA) + numel(matB), M * N, 0);
  int rc = 0;
  if (M > 0 && N > 0) {
    const float *A = static_cast<const float *>(matA->data), *B = static_cast<const float *>(matB->data);
    float *C = static_cast<float *>(matC->data);
    const int64_t lda = matA->shape[1], ldb = matB->shape[1];
    const int m = static_cast<int>(M), n = static_cast<int>(N), k = static_cast<int>(K);
    if (!transposeA && !transposeB) rc = dispatch_product<false, false>(A, lda, B, ldb, C, m, n, k, s, &ws);
    if (!transposeA && transposeB) rc = dispatch_product<false, true>(A, lda, B, ldb, C, m, n, k, s, &ws);
    if (transposeA && !transposeB) rc = dispatch_product<true, false>(A, lda, B, ldb, C, m, n, k, s, &ws);
    if (transposeA && transposeB) rc = dispatch_product<true, true>(A, lda, B, ldb, C, m, n, k, s, &ws);
  }
  if (p) p->workspace_memory = mib(ws);
  if (rc) return rc;
  return ps.finish();
}

extern "C" int DLGpuBatchMatrixMultiply(const DLArrayHandle matA, bool transposeA, const DLArrayHandle matB,
                                        bool transposeB, DLArrayHandle matC, DLStreamHandle stream_handle) {
  TS_REQUIRE(matA && matB && matC, "DLGpuBatchMatrixMultiply: NULL array");
  const int nd = matC->ndim;
  TS_REQUIRE(nd >= 2 && matA->ndim == nd && matB->ndim == nd, "DLGpuBatchMatrixMultiply: ranks must agree and be >= 2");
  int64_t batch = 1;
  for (int d = 0; d < nd - 2; ++d) {
    TS_REQUIRE(matA->shape[d] == matC->shape[d] && matB->shape[d] == matC->shape[d],
               "DLGpuBatchMatrixMultiply: leading axis %d differs between the operands", d);
    batch *= matC->shape[d];
  }
  const int64_t a0 = matA->shape[nd - 2], a1 = matA->shape[nd - 1], b0 = matB->shape[nd - 2], b1 = matB->shape[nd - 1];
  const int64_t M = matC->shape[nd - 2], N = matC->shape[nd - 1];
  const int64_t K = transposeA ? a0 : a1, Am = transposeA ? a1 : a0;
  const int64_t Bk = transposeB ? b1 : b0, Bn = transposeB ? b0 : b1;
  TS_REQUIRE(Am == M && Bn == N && Bk == K,
             "DLGpuBatchMatrixMultiply: shapes do not conform: op(A) %lldx%lld, op(B) %lldx%lld, C %lldx%lld", (long long)Am,
             (long long)K, (long long)Bk, (long long)Bn, (long long)M, (long long)N);
  TS_REQUIRE(M < (1ll << 31) && N < (1ll << 31) && K < (1ll << 31) - 64 && batch < (1ll << 31),
             "DLGpuBatchMatrixMultiply: dimension too large");
  hipStream_t s = stream_of(stream_handle);
  ProfileScope ps(nullptr, s, 0, 0, 0);
  int rc = 0;
  if (M > 0 && N > 0 && batch > 0) {
    const float *A = static_cast<const float *>(matA->data), *B = static_cast<const float *>(matB->data);
    float *C = static_cast<float *>(matC->data);
    const int m = static_cast<int>(M), n = static_cast<int>(N), k = static_cast<int>(K), b = static_cast<int>(batch);
    const int64_t sa = a0 * a1, sb = b0 * b1;
    if (!transposeA && !transposeB) rc = dispatch_batched<false, false>(A, a1, sa, B, b1, sb, C, b, m, n, k, s);
    if (!transposeA && transposeB) rc = dispatch_batched<false, true>(A, a1, sa, B, b1, sb, C, b, m, n, k, s);
    if (transposeA && !transposeB) rc = dispatch_batched<true, false>(A, a1, sa, B, b1, sb, C, b, m, n, k, s);
    if (transposeA && transposeB) rc = dispatch_batched<true, true>(A, a1, sa, B, b1, sb, C, b, m, n, k, s);
  }
  if (rc) return rc;
  return ps.finish();
}
