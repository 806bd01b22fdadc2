// The gated units of feed-forwards, on fp32 values: 0 silu(g) u, 1 gelu(g) u in its tanh form, 2 the clamped unit
// min(g, limit) sigmoid(alpha .) (clamp(u, +-limit) + 1)
#pragma once
#include "common.h"

namespace sm {

// tanh form of gelu: 0.5 z (1 + tanh(y)), y = sqrt(2/pi) (z + 0.044715 z^3), evaluated as
// z * sigmoid(2 y), which is the same function (1 + tanh(y) = 2 sigmoid(2 y))
__device__ __forceinline__ float gelu_tanhf_(float z) {
  return z * sigmoidf_(1.5957691216057308f * (z + 0.044715f * z * z * z));
}

__device__ __forceinline__ float unit_act(int act, float g, float u, float limit, float alpha) {
  if (act == 0) return silu_(g) * u;
  if (act == 1) return gelu_tanhf_(g) * u;
  g = fminf(g, limit);
  return g * __builtin_amdgcn_rcpf(1.0f + exp2_(-1.4426950408889634f * alpha * g)) * (fminf(fmaxf(u, -limit), limit) + 1.0f);
}

}  // namespace sm
