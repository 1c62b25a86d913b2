// The scalar functions of Sigmoid, Tanh and Relu, for their own kernels and for kernels that have them inside.
#pragma once
#include <hip/hip_runtime.h>

namespace tsplit {

// 1/(1+1/exp(x)) (src/ops/Sigmoid.cu:6); saturates to 0 and 1 without NaN
__device__ __forceinline__ float sigmoid_of(float x) { return 1.f / (1.f + expf(-x)); }
__device__ __forceinline__ float tanh_of(float x) { return tanhf(x); }
// gradients in the order of the reference's nodes: s * (1 + -1 * s) * g, (1 + (-1 * t) * t) * g
__device__ __forceinline__ float sigmoid_grad_of(float s, float g) { return (s * (1.f - s)) * g; }
__device__ __forceinline__ float tanh_grad_of(float t, float g) { return (1.f - t * t) * g; }

// Relu's gradient: (sign(x) + 1) * 0.5 * dy; keeps +-0 and NaN like np.sign
__device__ __forceinline__ float relu_grad_of(float x, float dy) {
  const float sgn = x > 0.f ? 1.f : (x < 0.f ? -1.f : x);
  return (sgn + 1.f) * 0.5f * dy;
}

}  // namespace tsplit
