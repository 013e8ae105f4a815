// gpt2_device.h — GELU on the device, for the elementwise kernels and the
// linear layers' epilogues.
#pragma once

#include <hip/hip_runtime.h>

namespace dfattn {

// tanh GELU constants: sqrt(2/pi) and the cubic coefficient (elementwise.cu:181-182).
constexpr float kGeluK0 = 0.7978845608028654f;
constexpr float kGeluK1 = 0.044715f;

__device__ __forceinline__ float gelu_f(float v) {
  return 0.5f * v * (1.f + tanhf(kGeluK0 * (v + kGeluK1 * v * v * v)));
}
__device__ __forceinline__ float gelu_grad(float go, float v) {
  const float t = tanhf(kGeluK0 * (v + kGeluK1 * v * v * v));
  const float d_inner = kGeluK0 * (1.f + 3.f * kGeluK1 * v * v);
  return go * (0.5f * (1.f + t) + 0.5f * v * (1.f - t * t) * d_inner);
}

}  // namespace dfattn
