// A sequence of LSTM cells with separate gates (examples/LSTM.py:21-90 node by node: per step a slice, eight products, bias
// broadcasts, sums, three Sigmoids, two Tanhs and four products of elements), as one launch a step.
//
// z_g = h W'_g + frame W_g + b_g is one product of rows [h | frame | 1 | 0...] with the weights below one another, so a step is
// that product for four gates with the cell behind it in registers; its h goes into the rows of the next step.  The reverse sweep
// has dh = dz_{t+1} U' with the cell's gradient behind it, and the parameters' gradients are one product over all steps of the
// rows with dz.
//
// What bounds a step is latency: the launch, one trip to memory for h (written on other XCDs a launch ago) and the products' own
// chain.  So a block is a tile of 16 samples x 16 units (64 blocks at 128 x 128), a wave is one gate of it, everything a wave
// multiplies is asked for before the first product, and the weights lie in the order of the matrix instruction's lanes, 16 bytes a
// lane.  v_mfma_f32_16x16x4_f32 sums k = 4 (lane / 16) + i with i its number of four: any order of k will do as long as both
// operands have it, and this one loads float4 on both sides.
#include "activations.h"
#include "common.h"

using namespace tsplit;

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
constexpr int kThreads = 256;
constexpr int kGates = 4;          // forget, input, output, candidate
constexpr int kAhead = 16;         // 16-deep chunks asked for at once: 256 deep, 128 registers

struct Weights {
  const float *w[kGates], *u[kGates], *b[kGates];
};
struct Grads {
  float *w[kGates], *u[kGates], *b[kGates];
};
struct Sizes {
  int n, steps, d, h;
  int depth;     // of the rows: h + d + 1 in whole 16s
  int hp;        // h in whole 16s
};

int up16(int64_t v) { return static_cast<int>((v + 15) / 16 * 16); }

// row k of the weights below one another: U, W, the bias, zeros
__device__ __forceinline__ float stacked(const Weights &q, const Sizes &z, int g, int k, int unit) {
  if (unit >= z.h) return 0.f;
  if (k < z.h) return q.u[g][static_cast<int64_t>(k) * z.h + unit];
  k -= z.h;
  if (k < z.d) return q.w[g][static_cast<int64_t>(k) * z.h + unit];
  return k == z.d ? q.b[g][unit] : 0.f;
}

// Before the first step: both directions' weights in lane order, the frames and ones in their rows, h of the first step.
// Fragment (gate, tile of 16 units, chunk of 16 k): lane l has k = 16 chunk + 4 (l / 16) .. + 3 of unit 16 tile + l % 16.
__global__ __launch_bounds__(kThreads) void prepare_kernel(Weights q, Sizes z, const float *__restrict__ x, const float *__restrict__ initial,
                                                           float *__restrict__ fwd, float *__restrict__ bwd, float *__restrict__ rows) {
  const int64_t nf = static_cast<int64_t>(kGates) * z.hp * z.depth, nb = static_cast<int64_t>(kGates) * z.hp * z.hp;
  const int64_t nr = static_cast<int64_t>(z.n) * z.steps * z.depth;
  const float first = initial[0];
  for (int64_t e = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x; e < nf + nb + nr; e += static_cast<int64_t>(gridDim.x) * kThreads) {
    if (e < nf + nb) {
      const bool back = e >= nf;
      const int64_t f = back ? e - nf : e;
      const int i = f & 3, lane = (f >> 2) & 63;
      const int chunks = (back ? z.hp : z.depth) / 16, tiles = z.hp / 16;
      const int64_t frag = f >> 8;
      const int k = static_cast<int>(frag % chunks) * 16 + 4 * (lane >> 4) + i;
      const int unit = static_cast<int>(frag / chunks % tiles) * 16 + (lane & 15), g = static_cast<int>(frag / chunks / tiles);
      if (back)
        bwd[f] = k < z.h && unit < z.h ? q.u[g][static_cast<int64_t>(unit) * z.h + k] : 0.f;
      else
        fwd[f] = stacked(q, z, g, k, unit);
    } else {
      const int64_t f = e - nf - nb, row = f / z.depth;
      const int k = static_cast<int>(f % z.depth);
      const int c = k - z.h;
      if (c >= 0)
        rows[f] = c < z.d ? x[row * z.d + c] : c == z.d ? 1.f : 0.f;
      else if (row % z.steps == 0)
        rows[f] = first;
    }
  }
}

// acc += rows of `a` (the lane's row and its 4 k) times the fragments at `b`, `chunks` 16-deep chunks
__device__ __forceinline__ f32x4 multiply(const float *__restrict__ a, const float *__restrict__ b, int chunks) {
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int j0 = 0; j0 < chunks; j0 += kAhead) {
    f32x4 av[kAhead], bv[kAhead];
#pragma unroll
    for (int j = 0; j < kAhead; ++j)
      if (j0 + j < chunks) {
        av[j] = *reinterpret_cast<const f32x4 *>(a + 16 * (j0 + j));
        bv[j] = *reinterpret_cast<const f32x4 *>(b + 256 * static_cast<int64_t>(j0 + j));
      }
#pragma unroll
    for (int j = 0; j < kAhead; ++j)
      if (j0 + j < chunks) {
#pragma unroll
        for (int i = 0; i < 4; ++i) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(av[j][i], bv[j][i], acc, 0, 0, 0);
      }
  }
  return acc;
}

// a wave's 16 x 16 results into LDS, for the thread (row, unit) that has the cell
__device__ __forceinline__ void put(float (&z)[kGates][16][17], const f32x4 &acc) {
  const int lane = threadIdx.x & 63, g = threadIdx.x >> 6;
#pragma unroll
  for (int i = 0; i < 4; ++i) z[g][4 * (lane >> 4) + i][lane & 15] = acc[i];
}

// A block's tile: units within samples.  Rows of samples beyond the last read the last one's and store nothing.
struct Tile {
  int unit, sample;   // its first ones / 16
  __device__ explicit Tile(const Sizes &z) : unit(blockIdx.x % (z.hp / 16)), sample(blockIdx.x / (z.hp / 16)) {}
};

__global__ __launch_bounds__(kThreads) void step_kernel(Sizes z, int t, float *rows, const float *__restrict__ fwd, float *__restrict__ gates,
                                                        float *__restrict__ cells, const float *__restrict__ initial, float *__restrict__ last) {
  __shared__ float lds[kGates][16][17];
  const Tile tile(z);
  const int lane = threadIdx.x & 63, g = threadIdx.x >> 6;
  const int64_t row = min(tile.sample * 16 + (lane & 15), z.n - 1);
  put(lds, multiply(rows + (row * z.steps + t) * z.depth + 4 * (lane >> 4),
                    fwd + (static_cast<int64_t>(g) * (z.hp / 16) + tile.unit) * (z.depth / 16) * 256 + 4 * lane, z.depth / 16));
  __syncthreads();
  const int r = threadIdx.x >> 4, c = threadIdx.x & 15;
  const int i = tile.sample * 16 + r, unit = tile.unit * 16 + c;
  if (i >= z.n || unit >= z.h) return;
  const int64_t at = static_cast<int64_t>(i) * z.steps + t;
  const float before = t ? cells[(at - 1) * z.h + unit] : initial[0];
  const float f = sigmoid_of(lds[0][r][c]), in = sigmoid_of(lds[1][r][c]), o = sigmoid_of(lds[2][r][c]), cand = tanh_of(lds[3][r][c]);
  const float cell = before * f + in * cand;
  const float h = tanh_of(cell) * o;
  float *act = gates + at * kGates * z.hp + unit;
  act[0] = f;
  act[z.hp] = in;
  act[2 * z.hp] = o;
  act[3 * z.hp] = cand;
  cells[at * z.h + unit] = cell;
  if (t + 1 < z.steps)
    rows[(at + 1) * z.depth + unit] = h;
  else
    last[static_cast<int64_t>(i) * z.h + unit] = h;
}

// dz of step t from that of step t + 1 (from dlast at the end); `carry` holds the gradient of the cell between launches
__global__ __launch_bounds__(kThreads) void step_gradient_kernel(Sizes z, int t, const float *__restrict__ dlast, const float *__restrict__ bwd,
                                                                 const float *__restrict__ gates, const float *__restrict__ cells,
                                                                 const float *__restrict__ initial, float *carry, float *dz) {
  __shared__ float lds[kGates][16][17];
  const Tile tile(z);
  const bool end = t + 1 == z.steps;
  const int lane = threadIdx.x & 63, g = threadIdx.x >> 6;
  if (!end) {
    const int64_t row = min(tile.sample * 16 + (lane & 15), z.n - 1);
    put(lds, multiply(dz + ((row * z.steps + t + 1) * kGates + g) * z.hp + 4 * (lane >> 4),
                      bwd + (static_cast<int64_t>(g) * (z.hp / 16) + tile.unit) * (z.hp / 16) * 256 + 4 * lane, z.hp / 16));
  }
  __syncthreads();
  const int r = threadIdx.x >> 4, c = threadIdx.x & 15;
  const int i = tile.sample * 16 + r, unit = tile.unit * 16 + c;
  if (i >= z.n) return;
  const int64_t at = static_cast<int64_t>(i) * z.steps + t;
  float *out = dz + at * kGates * z.hp + unit;
  if (unit >= z.h) {     // the next step and the parameters' product read whole 16s
    out[0] = out[z.hp] = out[2 * z.hp] = out[3 * z.hp] = 0.f;
    return;
  }
  const int64_t flat = static_cast<int64_t>(i) * z.h + unit;
  const float dh = end ? dlast[flat] : ((lds[0][r][c] + lds[1][r][c]) + lds[2][r][c]) + lds[3][r][c];
  const float *act = gates + at * kGates * z.hp + unit;
  const float f = act[0], in = act[z.hp], o = act[2 * z.hp], cand = act[3 * z.hp];
  const float th = tanh_of(cells[at * z.h + unit]), before = t ? cells[(at - 1) * z.h + unit] : initial[0];
  float dc = tanh_grad_of(th, o * dh);
  if (!end) dc = carry[flat] + dc;
  if (t) carry[flat] = f * dc;
  out[0] = sigmoid_grad_of(f, before * dc);
  out[z.hp] = sigmoid_grad_of(in, cand * dc);
  out[2 * z.hp] = sigmoid_grad_of(o, th * dh);
  out[3 * z.hp] = tanh_grad_of(cand, in * dc);
}

// the product's rows [U | W | bias] to the parameters' arrays
__global__ __launch_bounds__(kThreads) void spread_kernel(Sizes z, const float *__restrict__ all, Grads out) {
  const int64_t e = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x, per = static_cast<int64_t>(z.h + z.d + 1) * z.h;
  if (e >= kGates * per) return;
  const int g = static_cast<int>(e / per);
  const int64_t f = e % per;
  const int k = static_cast<int>(f / z.h), unit = static_cast<int>(f % z.h);
  const float v = all[(static_cast<int64_t>(k) * kGates + g) * z.hp + unit];
  if (k < z.h)
    out.u[g][f] = v;
  else if (k < z.h + z.d)
    out.w[g][f - static_cast<int64_t>(z.h) * z.h] = v;
  else
    out.b[g][unit] = v;
}

// params: W, U, b of the forget, input, output and candidate gates in turn
int sizes_of(const char *who, const DLArray *x, const DLArrayHandle *params, int steps, Sizes &z) {
  TS_REQUIRE(x && params && steps > 0, "%s: NULL array or no step", who);
  for (int i = 0; i < 3 * kGates; ++i) TS_REQUIRE(params[i], "%s: NULL parameter", who);
  TS_REQUIRE(x->ndim == 2 && x->shape[1] % steps == 0, "%s: x is [n, steps * frame]", who);
  const DLArray *u = params[1];
  TS_REQUIRE(u->ndim == 2 && u->shape[0] == u->shape[1] && u->shape[0] > 0, "%s: U is square", who);
  const int64_t n = x->shape[0], d = x->shape[1] / steps, h = u->shape[0];
  TS_REQUIRE(n < (1 << 20) && d < (1 << 24) && h < (1 << 20) && d > 0 && n * steps < (1ll << 31) - 64, "%s: dimension too large", who);
  for (int g = 0; g < kGates; ++g) {
    const DLArray *w = params[3 * g], *ug = params[3 * g + 1], *b = params[3 * g + 2];
    TS_REQUIRE(w->ndim == 2 && w->shape[0] == d && w->shape[1] == h && ug->ndim == 2 && ug->shape[0] == h && ug->shape[1] == h && numel(b) == h,
               "%s: the gates' parameters are W [frame, units], U [units, units], b [units]", who);
  }
  z = Sizes{static_cast<int>(n), steps, static_cast<int>(d), static_cast<int>(h), up16(h + d + 1), up16(h)};
  TS_REQUIRE(static_cast<int64_t>(z.hp / 16) * ((n + 15) / 16) < (1ll << 31) - 1, "%s: dimension too large", who);
  return 0;
}

bool holds(const DLArray *a, int64_t n) { return a && numel(a) == n && aligned16(a->data); }
float *fp(const DLArray *a) { return static_cast<float *>(a->data); }

int check_saved(const char *who, const Sizes &z, const DLArray *rows, const DLArray *packed, const DLArray *gates, const DLArray *cells,
                const DLArray *initial) {
  const int64_t at = static_cast<int64_t>(z.n) * z.steps;
  TS_REQUIRE(holds(rows, at * z.depth) && holds(packed, kGates * static_cast<int64_t>(z.hp) * (z.depth + z.hp)) && holds(gates, at * kGates * z.hp) &&
                 holds(cells, at * z.h) && initial && numel(initial) == 1,
             "%s: a saved array is not of its size (TSplit_LstmSizes) or not on 16 bytes", who);
  return 0;
}

}  // namespace

extern "C" int TSplit_LstmSizes(int frame, int units, int *depth, int *units_padded) {
  TS_REQUIRE(frame > 0 && units > 0 && depth && units_padded, "TSplit_LstmSizes: bad argument");
  *depth = up16(static_cast<int64_t>(frame) + units + 1);
  *units_padded = up16(units);
  return 0;
}

extern "C" int TSplit_Lstm(const DLArrayHandle x, const DLArrayHandle *params, const DLArrayHandle initial, int steps, DLArrayHandle rows,
                           DLArrayHandle packed, DLArrayHandle gates, DLArrayHandle cells, DLArrayHandle last, DLStreamHandle stream_handle) {
  Sizes z;
  if (const int rc = sizes_of("TSplit_Lstm", x, params, steps, z)) return rc;
  if (const int rc = check_saved("TSplit_Lstm", z, rows, packed, gates, cells, initial)) return rc;
  TS_REQUIRE(last && numel(last) == static_cast<int64_t>(z.n) * z.h, "TSplit_Lstm: the last state is [n, units]");
  hipStream_t s = stream_of(stream_handle);
  ProfileScope ps(nullptr, s, 0, 0, 0);
  if (z.n == 0) return ps.finish();
  Weights q;
  for (int g = 0; g < kGates; ++g) q.w[g] = fp(params[3 * g]), q.u[g] = fp(params[3 * g + 1]), q.b[g] = fp(params[3 * g + 2]);
  float *fwd = fp(packed), *bwd = fwd + kGates * static_cast<int64_t>(z.hp) * z.depth;
  const int64_t items = numel(packed) + numel(rows), blocks = (items + kThreads - 1) / kThreads;
  hipLaunchKernelGGL(prepare_kernel, dim3(static_cast<unsigned>(blocks < 4096 ? blocks : 4096)), dim3(kThreads), 0, s, q, z, fp(x), fp(initial), fwd, bwd,
                     fp(rows));
  const dim3 grid(static_cast<unsigned>(z.hp / 16 * ((z.n + 15) / 16)));
  for (int t = 0; t < steps; ++t)
    hipLaunchKernelGGL(step_kernel, grid, dim3(kThreads), 0, s, z, t, fp(rows), fwd, fp(gates), fp(cells), fp(initial), fp(last));
  return ps.finish();
}

extern "C" int TSplit_LstmGradient(const DLArrayHandle dlast, const DLArrayHandle x, const DLArrayHandle *params, const DLArrayHandle initial, int steps,
                                   const DLArrayHandle rows, const DLArrayHandle packed, const DLArrayHandle gates, const DLArrayHandle cells,
                                   DLArrayHandle dgates, DLArrayHandle *dparams, DLStreamHandle stream_handle) {
  const char *who = "TSplit_LstmGradient";
  Sizes z;
  if (const int rc = sizes_of(who, x, params, steps, z)) return rc;
  if (const int rc = check_saved(who, z, rows, packed, gates, cells, initial)) return rc;
  TS_REQUIRE(dlast && numel(dlast) == static_cast<int64_t>(z.n) * z.h, "%s: the gradient of the last state is [n, units]", who);
  TS_REQUIRE(holds(dgates, numel(gates)) && dgates->data != gates->data, "%s: dgates is another array of the size of gates", who);
  TS_REQUIRE(dparams, "%s: NULL gradients", who);
  for (int i = 0; i < 3 * kGates; ++i)
    TS_REQUIRE(dparams[i] && numel(dparams[i]) == numel(params[i]), "%s: a gradient is not of its parameter's size", who);
  hipStream_t s = stream_of(stream_handle);
  ProfileScope ps(nullptr, s, 0, 0, 0);
  const int64_t wide = kGates * static_cast<int64_t>(z.hp), carry_n = static_cast<int64_t>(z.n) * z.h;
  const int64_t all_n = static_cast<int64_t>(z.depth) * wide;
  float *all = static_cast<float *>(scratch_get(s, 3, static_cast<size_t>(all_n + carry_n) * 4));
  TS_REQUIRE(all, "%s: no scratch memory", who);
  float *carry = all + all_n;
  const float *bwd = fp(packed) + kGates * static_cast<int64_t>(z.hp) * z.depth;
  const dim3 grid(static_cast<unsigned>(z.hp / 16 * ((z.n + 15) / 16)));
  for (int t = steps - 1; t >= 0 && z.n; --t)
    hipLaunchKernelGGL(step_gradient_kernel, grid, dim3(kThreads), 0, s, z, t, fp(dlast), bwd, fp(gates), fp(cells), fp(initial), carry, fp(dgates));
  // all parameters' gradients: rows' over all samples and steps times dz (zeros for no samples)
  int64_t ashape[2] = {static_cast<int64_t>(z.n) * steps, z.depth}, bshape[2] = {static_cast<int64_t>(z.n) * steps, wide}, cshape[2] = {z.depth, wide};
  DLArray A{rows->data, rows->ctx, 2, ashape}, B{dgates->data, dgates->ctx, 2, bshape}, C{all, rows->ctx, 2, cshape};
  if (const int rc = DLGpuMatrixMultiply(&A, true, &B, false, &C, stream_handle, nullptr)) return rc;
  Grads out;
  for (int g = 0; g < kGates; ++g) out.w[g] = fp(dparams[3 * g]), out.u[g] = fp(dparams[3 * g + 1]), out.b[g] = fp(dparams[3 * g + 2]);
  const int64_t items = kGates * static_cast<int64_t>(z.h + z.d + 1) * z.h;
  TS_REQUIRE(items / kThreads < (1ll << 31) - 1, "%s: too many parameters", who);
  hipLaunchKernelGGL(spread_kernel, dim3(static_cast<unsigned>((items + kThreads - 1) / kThreads)), dim3(kThreads), 0, s, z, all, out);
  return ps.finish();
}
