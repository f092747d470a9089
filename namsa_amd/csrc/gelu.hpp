// The tanh form of GELU and its derivative, as the FP32 kernels of the
// corrector network apply them.
#pragma once

#include <hip/hip_runtime.h>

namespace namsa {

// the tanh both share: where a kernel needs both it is computed once
__device__ __forceinline__ float gelu_inner(float x) {
  const float c = 0.7978845608028654f;  // sqrt(2/pi)
  return tanhf(c * (x + 0.044715f * x * x * x));
}

__device__ __forceinline__ float gelu_tanh(float x, float t) { return 0.5f * x * (1.0f + t); }

__device__ __forceinline__ float gelu_tanh(float x) { return gelu_tanh(x, gelu_inner(x)); }

__device__ __forceinline__ float gelu_grad_tanh(float x, float t) {
  const float c = 0.7978845608028654f;
  return 0.5f * (1.0f + t) + 0.5f * x * (1.0f - t * t) * c * (1.0f + 3.0f * 0.044715f * x * x);
}

__device__ __forceinline__ float gelu_grad_tanh(float x) { return gelu_grad_tanh(x, gelu_inner(x)); }

}  // namespace namsa
