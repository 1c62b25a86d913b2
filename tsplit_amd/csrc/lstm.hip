// A sequence of LSTM cells with separate gates (examples/LSTM.py:21-90 node by node: per step a slice, eight products, bias
// broadcasts, sums, three Sigmoids, two Tanhs and four products of elements): up to 128 units all steps in one launch (further down),
// beyond that one launch a step.
//
// z_g = h W'_g + frame W_g + b_g is one product of rows [h | frame | 1 | 0...] with the weights below one another, so a step is
// that product for four gates with the cell behind it in registers; its h goes into the rows of the next step.  The reverse sweep
// has dh = dz_{t+1} U' with the cell's gradient behind it, and the parameters' gradients are one product over all steps of the
// rows with dz.
//
// What bounds a launch a step is latency: the launch, one trip to memory for h (written on other XCDs a launch ago) and the products' own
// chain.  So a block is a tile of 16 samples x 16 units (128 blocks at 128 samples and 256 units), a wave is one gate of it, everything a wave
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

// Before the first step: the weights as the steps read them, the frames and ones in their rows, h of the first step.
// A launch a step: fragments (gate, tile of 16 units, chunk of 16 k) in lane order, lane l k = 16 chunk + 4 (l / 16) .. + 3 of unit
// 16 tile + l % 16; `fwd` of the stacked weights, `bwd` of U'.  All steps in one launch (`flat`): fwd the matrices [frame + 1][gate][unit]
// of W and the bias, bwd U' as [gate][k][unit].
__global__ __launch_bounds__(kThreads) void prepare_kernel(Weights q, Sizes z, bool flat, const float *__restrict__ x,
                                                           const float *__restrict__ initial, float *__restrict__ fwd, float *__restrict__ bwd,
                                                           float *__restrict__ rows) {
  const int64_t nf = static_cast<int64_t>(kGates) * z.hp * (flat ? z.d + 1 : z.depth), nb = static_cast<int64_t>(kGates) * z.hp * z.hp;
  const int64_t nr = static_cast<int64_t>(z.n) * z.steps * z.depth;
  const float first = initial[0];
  for (int64_t e = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x; e < nf + nb + nr; e += static_cast<int64_t>(gridDim.x) * kThreads) {
    if (e < nf + nb) {
      const bool back = e >= nf;
      const int64_t f = back ? e - nf : e;
      int g, k, unit;
      if (flat) {
        unit = static_cast<int>(f % z.hp);
        const int64_t rest = f / z.hp;
        g = static_cast<int>(back ? rest / z.hp : rest % kGates);
        k = static_cast<int>(back ? rest % z.hp : rest / kGates + z.h);
      } else {
        const int lane = (f >> 2) & 63, chunks = (back ? z.hp : z.depth) / 16, tiles = z.hp / 16;
        const int64_t frag = f >> 8;
        k = static_cast<int>(frag % chunks) * 16 + 4 * (lane >> 4) + (f & 3);
        unit = static_cast<int>(frag / chunks % tiles) * 16 + (lane & 15);
        g = static_cast<int>(frag / chunks / tiles);
      }
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

// ---- All steps in one launch, where U fits the registers of one CU: up to 128 units (4 x 128 x 128 floats are 64 registers in each
// of 1024 threads).  A block takes four samples through all steps: nothing leaves the CU between steps but what the reverse sweep
// reads, and the frames' product is taken for all steps beforehand.  v_mfma_f32_4x4x1_16b_f32 with one block of A broadcast to all
// sixteen is 4 samples x 64 columns of one k in 8 cycles, the same rate as the larger shapes: lane l holds its column's weights, and
// a register of A has h of sample l % 4 and k = l / 4, sixteen k.  Of a step of 128 units 2 048 cycles are products.
// 28 steps of 128 samples: forward 61 us, gradient 56; a launch a step 144 and 150 (5.1-5.3 us each).
constexpr int kResident = 1024, kSamples = 4;

// acc += A's sixteen k times w[0..15]
__device__ __forceinline__ f32x4 multiply16(float a, const float *w, f32x4 acc) {
#define TS_K(k) acc = __builtin_amdgcn_mfma_f32_4x4x1f32(a, w[k], acc, 4, k, 0);
  TS_K(0) TS_K(1) TS_K(2) TS_K(3) TS_K(4) TS_K(5) TS_K(6) TS_K(7) TS_K(8) TS_K(9) TS_K(10) TS_K(11) TS_K(12) TS_K(13) TS_K(14) TS_K(15)
#undef TS_K
  return acc;
}

// COLS columns and DEPTH k of a product, dealt to the sixteen waves: 64 columns and a range of k each
template <int COLS, int DEPTH>
struct Share {
  static constexpr int kGroups = COLS / 64, kParts = 16 / kGroups, kDepth = DEPTH / kParts, kPitch = COLS + 16;
  int lane, col, part;
  __device__ Share() : lane(threadIdx.x & 63) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    col = wave % kGroups * 64 + lane, part = wave / kGroups;
  }
  // the wave's range of the product of lds[k][sample] with w, into parts[range][sample][column]
  __device__ void multiply(const float *lds, const float (&w)[kDepth], float *parts) const {
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int q = 0; q < kDepth / 16; ++q) acc = multiply16(lds[part * kDepth * kSamples + 64 * q + lane], w + 16 * q, acc);
#pragma unroll
    for (int i = 0; i < kSamples; ++i) parts[(part * kSamples + i) * kPitch + col] = acc[i];
  }
  __device__ static float sum(const float *parts, int sample, int col) {
    float v = parts[sample * kPitch + col];
#pragma unroll
    for (int p = 1; p < kParts; ++p) v += parts[(p * kSamples + sample) * kPitch + col];
    return v;
  }
};

// `gates` holds the frames' products and biases and receives the activations.  HP: units, rounded up.
template <int HP>
__global__ __launch_bounds__(kResident) void resident_kernel(Sizes z, Weights q, float *gates, float *__restrict__ rows, float *__restrict__ cells,
                                                             const float *__restrict__ initial, float *__restrict__ last) {
  using S = Share<kGates * HP, HP>;
  __shared__ float state[HP * kSamples], parts[S::kParts * kSamples * S::kPitch];
  const S me;
  float w[S::kDepth];
  {
    const float *u = q.u[me.col / HP];
    const int unit = me.col % HP, k0 = me.part * S::kDepth;
#pragma unroll
    for (int k = 0; k < S::kDepth; ++k) w[k] = unit < z.h && k0 + k < z.h ? u[(k0 + k) * z.h + unit] : 0.f;
  }
  const float first = initial[0];
  if (threadIdx.x < HP * kSamples) state[threadIdx.x] = static_cast<int>(threadIdx.x) / kSamples < z.h ? first : 0.f;
  // the first threads have a cell each
  const bool cell = threadIdx.x < HP * kSamples;
  const int sample = threadIdx.x / HP, unit = threadIdx.x % HP;
  const int i = blockIdx.x * kSamples + sample;
  const bool live = cell && i < z.n && unit < z.h;
  const int64_t at = static_cast<int64_t>(min(i, z.n - 1)) * z.steps;
  float *mine = gates + at * kGates * z.hp + min(unit, z.h - 1);
  float c = first, next[kGates];
  if (cell)
#pragma unroll
    for (int g = 0; g < kGates; ++g) next[g] = mine[g * z.hp];
  __syncthreads();
  for (int t = 0; t < z.steps; ++t) {
    float pre[kGates];
    float *act = mine + static_cast<int64_t>(t) * kGates * z.hp;
    if (cell) {
      const float *ahead = t + 1 < z.steps ? act + kGates * z.hp : act;
#pragma unroll
      for (int g = 0; g < kGates; ++g) pre[g] = next[g], next[g] = ahead[g * z.hp];
    }
    me.multiply(state, w, parts);
    __syncthreads();
    if (cell) {
#pragma unroll
      for (int g = 0; g < kGates; ++g) pre[g] += S::sum(parts, sample, g * HP + unit);
      const float f = sigmoid_of(pre[0]), in = sigmoid_of(pre[1]), o = sigmoid_of(pre[2]), cand = tanh_of(pre[3]);
      c = c * f + in * cand;
      const float h = tanh_of(c) * o;
      state[unit * kSamples + sample] = unit < z.h ? h : 0.f;
      if (live) {
        act[0] = f;
        act[z.hp] = in;
        act[2 * z.hp] = o;
        act[3 * z.hp] = cand;
        cells[(at + t) * z.h + unit] = c;
        if (t + 1 < z.steps)
          rows[(at + t + 1) * z.depth + unit] = h;
        else
          last[static_cast<int64_t>(i) * z.h + unit] = h;
      }
    }
    __syncthreads();
  }
}

// `ut`: U' as [gate][k][unit]
template <int HP>
__global__ __launch_bounds__(kResident) void resident_gradient_kernel(Sizes z, const float *__restrict__ dlast, const float *__restrict__ ut,
                                                                      const float *__restrict__ gates, const float *__restrict__ cells,
                                                                      const float *__restrict__ initial, float *__restrict__ dz) {
  using S = Share<HP, kGates * HP>;
  __shared__ float state[kGates * HP * kSamples], parts[S::kParts * kSamples * S::kPitch];
  const S me;
  float w[S::kDepth];
  {
    const int k0 = me.part * S::kDepth, g = k0 / HP, kk = k0 % HP;   // a range lies inside one gate
    const float *u = ut + static_cast<int64_t>(g) * z.hp * z.hp;
#pragma unroll
    for (int k = 0; k < S::kDepth; ++k) w[k] = me.col < z.hp && kk + k < z.hp ? u[(kk + k) * z.hp + me.col] : 0.f;
  }
  const bool cell = threadIdx.x < HP * kSamples;
  const int sample = threadIdx.x / HP, unit = threadIdx.x % HP;
  const int i = blockIdx.x * kSamples + sample;
  const int64_t row = min(i, z.n - 1), at = row * z.steps;
  const int u = min(unit, z.h - 1);
  const float *acts = gates + at * kGates * z.hp + u, *cs = cells + at * z.h + u;
  const float first = initial[0], dl = cell ? dlast[row * z.h + u] : 0.f;
  float carry = 0.f, next[kGates] = {}, cnext = 0.f, bnext = 0.f;
  auto load = [&](int t) {
#pragma unroll
    for (int g = 0; g < kGates; ++g) next[g] = acts[(static_cast<int64_t>(t) * kGates + g) * z.hp];
    cnext = cs[static_cast<int64_t>(t) * z.h];
    bnext = t ? cs[static_cast<int64_t>(t - 1) * z.h] : first;
  };
  if (cell) load(z.steps - 1);
  for (int t = z.steps - 1; t >= 0; --t) {
    const bool end = t + 1 == z.steps;
    float f = 0.f, in = 0.f, o = 0.f, cand = 0.f, cc = 0.f, before = 0.f;
    if (cell) {
      f = next[0], in = next[1], o = next[2], cand = next[3], cc = cnext, before = bnext;
      load(t ? t - 1 : 0);
    }
    if (!end) me.multiply(state, w, parts);
    __syncthreads();
    if (cell) {
      const float dh = end ? dl : S::sum(parts, sample, unit);
      const float th = tanh_of(cc);
      const float dc = carry + tanh_grad_of(th, o * dh);
      carry = f * dc;
      const bool real = unit < z.h;
      const float d[kGates] = {real ? sigmoid_grad_of(f, before * dc) : 0.f, real ? sigmoid_grad_of(in, cand * dc) : 0.f,
                               real ? sigmoid_grad_of(o, th * dh) : 0.f, real ? tanh_grad_of(cand, in * dc) : 0.f};
#pragma unroll
      for (int g = 0; g < kGates; ++g) {
        state[(g * HP + unit) * kSamples + sample] = d[g];
        if (i < z.n && unit < z.hp) dz[((at + t) * kGates + g) * z.hp + unit] = d[g];
      }
    }
    __syncthreads();
  }
}

// A CU's registers hold U of 128 units, 256 KB; of more it would come from L2 every step (1 MB at 256 units, 8 us at 64 bytes a clock),
// and a launch a step, with the weights dealt to many CUs, takes 5.
bool resident(const Sizes &z) { return z.h <= 128; }

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
  const bool flat = resident(z);
  const int64_t wide = kGates * static_cast<int64_t>(z.hp), blocks = (numel(packed) + numel(rows) + kThreads - 1) / kThreads;
  hipLaunchKernelGGL(prepare_kernel, dim3(static_cast<unsigned>(blocks < 4096 ? blocks : 4096)), dim3(kThreads), 0, s, q, z, flat, fp(x), fp(initial),
                     fwd, bwd, fp(rows));
  if (flat) {
    int64_t ashape[2] = {static_cast<int64_t>(z.n) * steps, z.d}, bshape[2] = {z.d, wide}, cshape[2] = {static_cast<int64_t>(z.n) * steps, wide};
    DLArray A{x->data, x->ctx, 2, ashape}, B{fwd, x->ctx, 2, bshape}, bias{fwd + z.d * wide, x->ctx, 1, bshape + 1}, C{gates->data, x->ctx, 2, cshape};
    if (const int rc = TSplit_MatrixMultiplyAdd(&A, 0, &B, 0, &bias, nullptr, nullptr, &C, nullptr, stream_handle)) return rc;
    hipLaunchKernelGGL((z.h <= 64 ? resident_kernel<64> : resident_kernel<128>), dim3((z.n + kSamples - 1) / kSamples), dim3(kResident), 0, s, z, q,
                       fp(gates), fp(rows), fp(cells), fp(initial), fp(last));
    return ps.finish();
  }
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
  if (resident(z) && z.n)
    hipLaunchKernelGGL((z.h <= 64 ? resident_gradient_kernel<64> : resident_gradient_kernel<128>), dim3((z.n + kSamples - 1) / kSamples),
                       dim3(kResident), 0, s, z, fp(dlast), bwd, fp(gates), fp(cells), fp(initial), fp(dgates));
  for (int t = steps - 1; t >= 0 && z.n && !resident(z); --t)
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
