// Row softmax and softmax-cross-entropy (forward, gradient).
//
// Softmax: one wavefront owns one row: max and sum are wave64 shuffle reductions, no LDS and
// no block barrier; a 256-thread block handles 4 rows.  The cross-entropy mean is a second,
// single-block deterministic reduction over the per-row losses (the reference does that
// mean serially in thread 0 of its only block: src/ops/SoftmaxCrossEntropy.cu:33-41).
// The cross-entropy kernels hold a row in registers, a wave or a block of 512 threads a row.
#include <algorithm>
#include <mutex>

#include "common.h"
#include "reduce.h"

// Per-row losses of TSplit_SoftmaxCrossEntropyNoAlloc (below): a fixed array in the code object, so
// that call needs no device allocation.  No kernel names it: kernels get its address as an argument.
// The host code's reference to it (hipGetSymbolAddress below) is what makes the compiler give this
// static variable a symbol the runtime can find; it must NOT carry __attribute__((used)), which keeps
// the symbol local to the code object, and looking up a local symbol ends the process.
constexpr int kNoAllocMaxRows = 1 << 18;
static __device__ __align__(256) float scratch[kNoAllocMaxRows];

namespace tsplit {
namespace {

constexpr int kRowsPerBlock = 4;

__device__ __forceinline__ void row_max_sum(const float *row, int ncol, int lane, float &mx, float &sum) {
  float m = -INFINITY;
  for (int j = lane; j < ncol; j += kWave) m = fmaxf(m, row[j]);
  m = wave_max(m);
  float s = 0.f;
  for (int j = lane; j < ncol; j += kWave) s += expf(row[j] - m);
  mx = m;
  sum = wave_sum(s);
}

__global__ __launch_bounds__(256) void softmax_kernel(const float *__restrict__ x, float *__restrict__ y,
                                                      int64_t nrow, int ncol) {
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t r = static_cast<int64_t>(blockIdx.x) * kRowsPerBlock + threadIdx.x / kWave;
  if (r >= nrow) return;
  const float *row = x + r * ncol;
  float m, s;
  row_max_sum(row, ncol, lane, m, s);
  const float inv = 1.f / s;
  float *out = y + r * ncol;
  for (int j = lane; j < ncol; j += kWave) out[j] = expf(row[j] - m) * inv;
}

// ---- cross-entropy: loss_r = sum_j label[j] * (log(sum) - (y[j] - max)), gradient (softmax - label) * scale
typedef float f32x4 __attribute__((ext_vector_type(4)));

// Where a row's labels come from: an array of the logits' shape, or one class index a row (as the reference stores them: a float), smoothed:
// label[j] = on * (j == id) + off.
struct LabelArray {
  static constexpr bool kIds = false;
  const float *p;
  template <int VEC>
  __device__ __forceinline__ void get(int64_t row, int ncol, int j, float (&l)[VEC]) const {
    if constexpr (VEC == 4) {
      const f32x4 v = __builtin_nontemporal_load(reinterpret_cast<const f32x4 *>(p + row * ncol + j));
#pragma unroll
      for (int i = 0; i < 4; ++i) l[i] = v[i];
    } else {
      l[0] = p[row * ncol + j];
    }
  }
};
struct LabelIds {
  static constexpr bool kIds = true;
  const float *ids;
  float on, off;
  template <int VEC>
  __device__ __forceinline__ void get(int64_t row, int /*ncol*/, int j, float (&l)[VEC]) const {
    const float id = ids[row];
#pragma unroll
    for (int i = 0; i < VEC; ++i) l[i] = (static_cast<float>(j + i) == id ? on : 0.f) + off;
  }
};

// One block a row.  What bounds it is memory: so a row's logits are read once, into registers, and maximum, sum and result are taken from
// there (8192 rows of 32 000: with two reads of the logits and one of a label array the loss took 328 us and the gradient 677; from
// registers the gradient takes 549, with class indices 458 and the loss 190; 250 rows of 5003, which a wave each used to take value by
// value: 33 -> 9 and 39 -> 6).  WORDS vectors of VEC values a thread hold rows of up to THREADS * VEC * WORDS columns; WORDS = 0 is the
// form for longer ones, which reads the row again.  GRAD: out is the gradient, scaled by g[0] * inv_batch; else out[row] is the row's loss.
template <int THREADS, int VEC, int WORDS, bool GRAD, class Label>
__global__ __launch_bounds__(THREADS == kWave ? 4 * kWave : THREADS) __attribute__((amdgpu_waves_per_eu(4))) void ce_kernel(const float *__restrict__ y, Label lab,
                                                                                    const float *__restrict__ g, float *__restrict__ out,
                                                                                    int64_t nrow, int ncol, float inv_batch) {
  constexpr int kWaves = THREADS / kWave, kRows = kWaves == 1 ? 4 : 1;   // (rows of a wave: four a block)
  __shared__ float sm[kWaves];
  const int thread = kRows > 1 ? threadIdx.x % THREADS : threadIdx.x;
  const int wave = kRows > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x / THREADS) : 0;
  for (int64_t r = static_cast<int64_t>(blockIdx.x) * kRows + wave; r < nrow; r += static_cast<int64_t>(gridDim.x) * kRows) {
    const float *row = y + r * ncol;
    constexpr int kHeld = WORDS ? WORDS : 1;
    float v[kHeld][VEC];
    auto fetch = [&](int w, float(&x)[VEC]) {
      const int j = (w * THREADS + thread) * VEC;
      if constexpr (VEC == 4) {
        f32x4 q = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};
        if (j < ncol) q = *reinterpret_cast<const f32x4 *>(row + j);   // ncol is a multiple of 4
#pragma unroll
        for (int i = 0; i < 4; ++i) x[i] = q[i];
      } else {
        x[0] = j < ncol ? row[j] : -INFINITY;
      }
    };
    const int words = WORDS ? WORDS : (ncol + THREADS * VEC - 1) / (THREADS * VEC);
    auto each = [&](auto &&f) {
#pragma unroll
      for (int w = 0; w < words; ++w) {
        if constexpr (WORDS) {
          f(w, v[w]);
        } else {
          float x[VEC];
          fetch(w, x);
          f(w, x);
        }
      }
    };
    if constexpr (WORDS) {
#pragma unroll
      for (int w = 0; w < WORDS; ++w) fetch(w, v[w]);
    }
    float m = -INFINITY;
    each([&](int, float(&x)[VEC]) {
#pragma unroll
      for (int i = 0; i < VEC; ++i) m = fmaxf(m, x[i]);
    });
    m = wave_max(m);
    if constexpr (kWaves > 1) {
      if (threadIdx.x % kWave == 0) sm[threadIdx.x / kWave] = m;
      __syncthreads();
      m = sm[0];
#pragma unroll
      for (int i = 1; i < kWaves; ++i) m = fmaxf(m, sm[i]);
    }
    // the loss, sum of label * (lse - (x - m)), is lse * sum(label) - sum(label * (x - m)): two terms of one sign.  Of class indices
    // label is `off` (and one value more): weighted as they are added, so that logits masked with the type's lowest value add up.
    float s = 0.f, labels = 0.f, below = 0.f;
    each([&](int w, float(&x)[VEC]) {
      const int j = (w * THREADS + thread) * VEC;
      float l[VEC] = {};
      if constexpr (!GRAD && !Label::kIds) {
        if (j < ncol) lab.template get<VEC>(r, ncol, j, l);
      }
#pragma unroll
      for (int i = 0; i < VEC; ++i) {
        const float e = j < ncol ? expf(x[i] - m) : 0.f;
        if constexpr (GRAD && WORDS != 0) x[i] = e;
        if constexpr (!GRAD && Label::kIds) below = j < ncol ? fmaf(lab.off, x[i] - m, below) : below;
        if constexpr (!GRAD && !Label::kIds) {
          labels += l[i];
          below += j < ncol ? l[i] * (x[i] - m) : 0.f;
        }
        s += e;
      }
    });
    s = kWaves > 1 ? block_sum<float, kWaves>(s, sm) : wave_sum(s);
    if constexpr (GRAD) {
      const float inv = 1.f / s, scale = g[0] * inv_batch;
      each([&](int w, float(&x)[VEC]) {
        const int j = (w * THREADS + thread) * VEC;
        if (j >= ncol) return;
        float l[VEC];
        lab.template get<VEC>(r, ncol, j, l);
#pragma unroll
        for (int i = 0; i < VEC; ++i) {
          float e = x[i];
          if constexpr (WORDS == 0) e = expf(e - m);
          l[i] = (e * inv - l[i]) * scale;
        }
        if constexpr (VEC == 4)
          __builtin_nontemporal_store(f32x4{l[0], l[1], l[2], l[3]}, reinterpret_cast<f32x4 *>(out + r * ncol + j));
        else
          out[r * ncol + j] = l[0];
      });
    } else {
      below = kWaves > 1 ? block_sum<float, kWaves>(below, sm) : wave_sum(below);
      if constexpr (!Label::kIds) labels = kWaves > 1 ? block_sum<float, kWaves>(labels, sm) : wave_sum(labels);
      if (thread == 0) {
        const float lse = logf(s);
        if constexpr (Label::kIds) {
          const float id = lab.ids[r];
          const int hit = id >= 0.f && id < static_cast<float>(ncol) ? static_cast<int>(id) : -1;
          float loss = lab.off * static_cast<float>(ncol) * lse - below;
          if (hit >= 0 && static_cast<float>(hit) == id) loss += lab.on * (lse - (row[hit] - m));
          out[r] = loss;
        } else {
          out[r] = lse * labels - below;
        }
      }
    }
    if constexpr (kWaves > 1) __syncthreads();   // the next row's maxima go where this row's sums are read
  }
}

__global__ __launch_bounds__(256) void mean_kernel(const float *__restrict__ v, float *__restrict__ out, int64_t n) {
  __shared__ double sm[4];
  double acc = 0.0;
  for (int64_t i = threadIdx.x; i < n; i += 256) acc += static_cast<double>(v[i]);
  acc = block_sum<double, 4>(acc, sm);
  if (threadIdx.x == 0) out[0] = static_cast<float>(acc / static_cast<double>(n));
}

// The loss of a label array of more columns than that: running (max, scaled sum) pairs and the label sums in one pass over both arrays,
// loss_r = (log s + m) * sum(l) - sum(l * y).  8192 rows of 32 000: 328 us; labels beside logits in registers 550, the row read again 440.
struct MaxSum {
  float m, s;     // s = sum of exp(x - m) over the elements seen so far
};

__device__ __forceinline__ void ms_add(MaxSum &a, float x) {
  if (x > a.m) {
    a.s = a.s * expf(a.m - x) + 1.f;      // expf(-inf) = 0 covers the first element
    a.m = x;
  } else {
    a.s += expf(x - a.m);
  }
}

__device__ __forceinline__ MaxSum ms_merge(MaxSum a, MaxSum b) {
  const float m = fmaxf(a.m, b.m);
  if (m == -INFINITY) return MaxSum{m, 0.f};
  return MaxSum{m, a.s * expf(a.m - m) + b.s * expf(b.m - m)};
}

__device__ __forceinline__ MaxSum ms_block(MaxSum v, float *smem /* 8 floats */) {
#pragma unroll
  for (int d = kWave / 2; d > 0; d >>= 1) {
    MaxSum o{__shfl_xor(v.m, d, kWave), __shfl_xor(v.s, d, kWave)};
    v = ms_merge(v, o);
  }
  const int wave = threadIdx.x / kWave, lane = threadIdx.x & (kWave - 1);
  if (lane == 0) {
    smem[2 * wave] = v.m;
    smem[2 * wave + 1] = v.s;
  }
  __syncthreads();
  MaxSum r{smem[0], smem[1]};
#pragma unroll
  for (int w = 1; w < 4; ++w) r = ms_merge(r, MaxSum{smem[2 * w], smem[2 * w + 1]});
  __syncthreads();
  return r;
}

__global__ __launch_bounds__(256) void ce_rows_wide_kernel(const float *__restrict__ y, const float *__restrict__ lab,
                                                           float *__restrict__ row_loss, int64_t nrow, int ncol) {
  __shared__ float sm[8];
  __shared__ float sm2[8];
  for (int64_t r = blockIdx.x; r < nrow; r += gridDim.x) {
    const f32x4 *row = reinterpret_cast<const f32x4 *>(y + r * ncol);
    const f32x4 *l = reinterpret_cast<const f32x4 *>(lab + r * ncol);
    MaxSum ms{-INFINITY, 0.f};
    float sl = 0.f, sly = 0.f;
    for (int j = threadIdx.x; j < ncol / 4; j += 256) {
      const f32x4 v = row[j], w = __builtin_nontemporal_load(l + j);
      ms_add(ms, v.x);
      ms_add(ms, v.y);
      ms_add(ms, v.z);
      ms_add(ms, v.w);
      sl += (w.x + w.y) + (w.z + w.w);
      sly += (w.x * v.x + w.y * v.y) + (w.z * v.z + w.w * v.w);
    }
    ms = ms_block(ms, sm);
    sl = block_sum<float, 4>(sl, sm2);
    __syncthreads();
    sly = block_sum<float, 4>(sly, sm2);
    if (threadIdx.x == 0) row_loss[r] = (logf(ms.s) + ms.m) * sl - sly;
    __syncthreads();
  }
}

// Rows of up to 1024 columns: a wave each (nothing waits for a barrier); longer ones: 512 threads.
template <bool GRAD, class Label>
void launch_ce(const float *y, const Label &lab, const float *g, float *out, int64_t nrow, int ncol, float inv_batch, bool words, hipStream_t s) {
  auto run = [&](auto *kernel, int threads) {
    const int64_t blocks = std::min<int64_t>(threads == 64 ? (nrow + 3) / 4 : nrow, 1 << 20);
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(blocks)), dim3(threads == 64 ? 256 : threads), 0, s, y, lab, g, out, nrow, ncol, inv_batch);
  };
  if (ncol <= 64 * 4) return run(ce_kernel<64, 1, 4, GRAD, Label>, 64);
  if (ncol <= 64 * 16) return run(ce_kernel<64, 1, 16, GRAD, Label>, 64);
  constexpr bool kLong = GRAD || Label::kIds;
  if (words) {
    if (ncol <= 2048 * 4) return run(ce_kernel<512, 4, 4, GRAD, Label>, 512);
    if (kLong && ncol <= 2048 * 16) return run(ce_kernel<512, 4, kLong ? 16 : 4, GRAD, Label>, 512);
    if constexpr (kLong) {
      return run(ce_kernel<512, 4, 0, GRAD, Label>, 512);
    } else {
      hipLaunchKernelGGL(ce_rows_wide_kernel, dim3(static_cast<unsigned>(std::min<int64_t>(nrow, 1 << 20))), dim3(256), 0, s, y, lab.p, out, nrow, ncol);
      return;
    }
  }
  if (ncol <= 512 * 16) return run(ce_kernel<512, 1, 16, GRAD, Label>, 512);
  if (kLong && ncol <= 512 * 64) return run(ce_kernel<512, 1, kLong ? 64 : 16, GRAD, Label>, 512);
  return run(ce_kernel<512, 1, 0, GRAD, Label>, 512);
}
inline bool in_words(int ncol, const void *a, const void *b) { return ncol % 4 == 0 && aligned16(a) && aligned16(b); }

inline bool rows_cols(const DLArray *a, int64_t &nrow, int &ncol) {
  if (a->ndim < 1) return false;
  nrow = 1;
  for (int i = 0; i + 1 < a->ndim; ++i) nrow *= a->shape[i];
  ncol = static_cast<int>(a->shape[a->ndim - 1]);
  return nrow > 0 && ncol > 0;
}

// ---------------------------------------------------------------- entry point that allocates nothing
// Each GPU holds its own copy of `scratch` (1 MiB) at its own address, from the time the library is
// loaded on it until the process ends.
constexpr int kNoAllocMaxDevices = 64;
std::mutex g_noalloc_mu;
float *g_noalloc_ptr[kNoAllocMaxDevices] = {};

}  // namespace

// Device address of `scratch` on device `dev`, looked up once per device with that device current.
// (In host code the array's name is only a handle for this lookup, never a device address.)
float *softmax_noalloc_scratch(int dev) {
  if (dev < 0 || dev >= kNoAllocMaxDevices) return nullptr;
  std::lock_guard<std::mutex> lk(g_noalloc_mu);
  if (g_noalloc_ptr[dev]) return g_noalloc_ptr[dev];
  int caller_dev = -1;
  if (hipGetDevice(&caller_dev) != hipSuccess) {
    (void)hipGetLastError();
    caller_dev = -1;
  }
  if (hipSetDevice(dev) != hipSuccess) {
    (void)hipGetLastError();
    return nullptr;
  }
  void *ptr = nullptr;
  const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
  if (caller_dev >= 0 && caller_dev != dev) (void)hipSetDevice(caller_dev);   // the caller's device stays current
  if (e != hipSuccess || ptr == nullptr) {
    (void)hipGetLastError();
    std::fprintf(stderr, "[libc_runtime_api] hipGetSymbolAddress(scratch) failed on device %d: %s\n", dev,
                 hipGetErrorString(e));
    return nullptr;
  }
  g_noalloc_ptr[dev] = static_cast<float *>(ptr);
  return g_noalloc_ptr[dev];
}

// Called from the library's per-device init call so that the first operator call finds the address.
void softmax_noalloc_setup(int dev) { (void)softmax_noalloc_scratch(dev); }

}  // namespace tsplit

using namespace tsplit;

extern "C" {

int TSplit_SoftmaxCrossEntropyNoAlloc(const DLArrayHandle input_a, const DLArrayHandle input_b, DLArrayHandle output,
                                      DLStreamHandle stream_handle) {
  const char *who = "TSplit_SoftmaxCrossEntropyNoAlloc";
  TS_REQUIRE(input_a && input_b && output, "%s: NULL array", who);
  TS_REQUIRE(numel(input_a) == numel(input_b), "%s: logits and labels differ in size", who);
  TS_REQUIRE(numel(output) >= 1, "%s: output must hold one element", who);
  int64_t nrow;
  int ncol;
  TS_REQUIRE(rows_cols(input_a, nrow, ncol), "%s: empty input", who);
  TS_REQUIRE(nrow <= kNoAllocMaxRows, "%s: %lld rows, the fixed scratch array holds %d; use DLGpuSoftmaxCrossEntropy", who,
             static_cast<long long>(nrow), kNoAllocMaxRows);
  float *row_loss = softmax_noalloc_scratch(input_a->ctx.device_id);
  TS_REQUIRE(row_loss, "%s: the scratch array of device %d could not be located", who, input_a->ctx.device_id);
  hipStream_t s = stream_of(stream_handle);
  // every row's entry is written by the first kernel before the second reads rows [0, nrow): nothing of
  // an earlier call's contents is read, so nothing has to be cleared
  launch_ce<false>(static_cast<const float *>(input_a->data), LabelArray{static_cast<const float *>(input_b->data)}, nullptr, row_loss, nrow, ncol,
                   0.f, in_words(ncol, input_a->data, input_b->data), s);
  hipLaunchKernelGGL(mean_kernel, dim3(1), dim3(256), 0, s, row_loss, static_cast<float *>(output->data), nrow);
  const hipError_t le = hipGetLastError();
  TS_REQUIRE(le == hipSuccess, "%s: kernel launch failed: %s", who, hipGetErrorString(le));
  return 0;
}

int DLGpuSoftmax(const DLArrayHandle input, DLArrayHandle output, DLStreamHandle stream_handle, ProfilerHandle p) {
  TS_REQUIRE(input && output, "DLGpuSoftmax: NULL array");
  TS_REQUIRE(input->ndim == 2 && output->ndim == 2, "DLGpuSoftmax: 2-D arrays only");
  TS_REQUIRE(numel(input) == numel(output), "DLGpuSoftmax: sizes differ");
  int64_t nrow;
  int ncol;
  TS_REQUIRE(rows_cols(input, nrow, ncol), "DLGpuSoftmax: empty input");
  hipStream_t s = stream_of(stream_handle);
  ProfileScope ps(p, s, numel(input), numel(output), 0);
  const unsigned blocks = static_cast<unsigned>((nrow + kRowsPerBlock - 1) / kRowsPerBlock);
  hipLaunchKernelGGL(softmax_kernel, dim3(blocks), dim3(256), 0, s, static_cast<const float *>(input->data),
                     static_cast<float *>(output->data), nrow, ncol);
  return ps.finish();
}

int DLGpuSoftmaxCrossEntropy(const DLArrayHandle input_a, const DLArrayHandle input_b, DLArrayHandle output,
                             DLStreamHandle stream_handle, ProfilerHandle p) {
  TS_REQUIRE(input_a && input_b && output, "DLGpuSoftmaxCrossEntropy: NULL array");
  TS_REQUIRE(numel(input_a) == numel(input_b), "DLGpuSoftmaxCrossEntropy: logits and labels differ in size");
  TS_REQUIRE(numel(output) >= 1, "DLGpuSoftmaxCrossEntropy: output must hold one element");
  int64_t nrow;
  int ncol;
  TS_REQUIRE(rows_cols(input_a, nrow, ncol), "DLGpuSoftmaxCrossEntropy: empty input");
  hipStream_t s = stream_of(stream_handle);
  float *row_loss = static_cast<float *>(scratch_get(s, 0, static_cast<size_t>(nrow) * 4));
  TS_REQUIRE(row_loss, "DLGpuSoftmaxCrossEntropy: no scratch memory");
  ProfileScope ps(p, s, 2 * numel(input_a), 1, nrow);
  launch_ce<false>(static_cast<const float *>(input_a->data), LabelArray{static_cast<const float *>(input_b->data)}, nullptr, row_loss, nrow, ncol,
                   0.f, in_words(ncol, input_a->data, input_b->data), s);
  hipLaunchKernelGGL(mean_kernel, dim3(1), dim3(256), 0, s, row_loss, static_cast<float *>(output->data), nrow);
  return ps.finish();
}

int DLGpuSoftmaxCrossEntropy_Gradient(const DLArrayHandle input_a, const DLArrayHandle input_b,
                                      const DLArrayHandle input_c, DLArrayHandle output,
                                      DLStreamHandle stream_handle, ProfilerHandle p) {
  TS_REQUIRE(input_a && input_b && input_c && output, "DLGpuSoftmaxCrossEntropy_Gradient: NULL array");
  TS_REQUIRE(numel(input_a) == numel(input_b) && numel(input_a) == numel(output),
             "DLGpuSoftmaxCrossEntropy_Gradient: operand sizes differ");
  TS_REQUIRE(numel(input_c) >= 1, "DLGpuSoftmaxCrossEntropy_Gradient: upstream gradient is empty");
  int64_t nrow;
  int ncol;
  TS_REQUIRE(rows_cols(input_a, nrow, ncol), "DLGpuSoftmaxCrossEntropy_Gradient: empty input");
  hipStream_t s = stream_of(stream_handle);
  ProfileScope ps(p, s, 2 * numel(input_a) + 1, numel(output), 0);
  // scaled by 1/shape[0] (not 1/rows), as src/ops/SoftmaxCrossEntropy.cu:101,120 does
  const float inv_batch = 1.f / static_cast<float>(input_a->shape[0]);
  launch_ce<true>(static_cast<const float *>(input_a->data), LabelArray{static_cast<const float *>(input_b->data)},
                  static_cast<const float *>(input_c->data), static_cast<float *>(output->data), nrow, ncol, inv_batch,
                  in_words(ncol, input_a->data, input_b->data) && aligned16(output->data), s);
  return ps.finish();
}

int TSplit_SoftmaxCrossEntropyIds(const DLArrayHandle logits, const DLArrayHandle ids, float on, float off, DLArrayHandle output,
                                  DLStreamHandle stream_handle) {
  const char *who = "TSplit_SoftmaxCrossEntropyIds";
  TS_REQUIRE(logits && ids && output, "%s: NULL array", who);
  int64_t nrow;
  int ncol;
  TS_REQUIRE(rows_cols(logits, nrow, ncol), "%s: empty input", who);
  TS_REQUIRE(numel(ids) == nrow && numel(output) >= 1, "%s: one class index a row and a loss of one element", who);
  hipStream_t s = stream_of(stream_handle);
  float *row_loss = static_cast<float *>(scratch_get(s, 0, static_cast<size_t>(nrow) * 4));
  TS_REQUIRE(row_loss, "%s: no scratch memory", who);
  ProfileScope ps(nullptr, s, 0, 0, 0);
  launch_ce<false>(static_cast<const float *>(logits->data), LabelIds{static_cast<const float *>(ids->data), on, off}, nullptr, row_loss, nrow, ncol,
                   0.f, in_words(ncol, logits->data, nullptr), s);
  hipLaunchKernelGGL(mean_kernel, dim3(1), dim3(256), 0, s, row_loss, static_cast<float *>(output->data), nrow);
  return ps.finish();
}

int TSplit_SoftmaxCrossEntropyIds_Gradient(const DLArrayHandle logits, const DLArrayHandle ids, float on, float off, const DLArrayHandle adjoint,
                                           DLArrayHandle output, DLStreamHandle stream_handle) {
  const char *who = "TSplit_SoftmaxCrossEntropyIds_Gradient";
  TS_REQUIRE(logits && ids && adjoint && output, "%s: NULL array", who);
  int64_t nrow;
  int ncol;
  TS_REQUIRE(rows_cols(logits, nrow, ncol), "%s: empty input", who);
  TS_REQUIRE(numel(ids) == nrow && numel(adjoint) >= 1 && numel(output) == numel(logits), "%s: sizes differ", who);
  hipStream_t s = stream_of(stream_handle);
  ProfileScope ps(nullptr, s, 0, 0, 0);
  launch_ce<true>(static_cast<const float *>(logits->data), LabelIds{static_cast<const float *>(ids->data), on, off},
                  static_cast<const float *>(adjoint->data), static_cast<float *>(output->data), nrow, ncol,
                  1.f / static_cast<float>(logits->shape[0]), in_words(ncol, logits->data, output->data), s);
  return ps.finish();
}

}  // extern "C"
