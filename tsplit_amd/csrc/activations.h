// The scalar functions of Sigmoid and Tanh, for their own kernels and for kernels that have them inside.
#pragma once
#include <hip/hip_runtime.h>

namespace tsplit {

// 1/(1+1/exp(x)) (src/ops/Sigmoid.cu:6); saturates to 0 and 1 without NaN
__device__ __forceinline__ float sigmoid_of(float x) { return 1.f / (1.f + expf(-x)); }
__device__ __forceinline__ float tanh_of(float x) { return tanhf(x); }
// gradients in the order of the reference's nodes: s * (1 + -1 * s) * g, (1 + (-1 * t) * t) * g
__device__ __forceinline__ float sigmoid_grad_of(float s, float g) { return (s * (1.f - s)) * g; }
__device__ __forceinline__ float tanh_grad_of(float t, float g) { return (1.f - t * t) * g; }

}  // namespace tsplit
