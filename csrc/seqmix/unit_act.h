// The gated units of feed-forwards, on fp32 values: 0 silu(g) u, 1 gelu(g) u in its tanh form, 2 the clamped unit
// min(g, limit) sigmoid(alpha .) (clamp(u, +-limit) + 1)
#pragma once
#include "common.h"

namespace sm {

// tanh form of gelu: 0.5 z (1 + tanh(y)), y = sqrt(2/pi) (z + 0.044715 z^3), evaluated as
// z * sigmoid(2 y), which is the same function (1 + tanh(y) = 2 sigmoid(2 y))
__device__ __forceinline__ float gelu_arg(float z) { return 1.5957691216057308f * (z + 0.044715f * z * z * z); }
__device__ __forceinline__ float gelu_tanhf_(float z) { return z * sigmoidf_(gelu_arg(z)); }

// (one sigmoid for all three, so that an unrolled epilogue stays short.  For fp32 results it is sigmoidf_: e^-y as exp2 of a
// rounded product is off by |y| 2^-24 more, silu of gates from -20 to -5 by up to 1.0e-6 where expf and a division leave 1.7e-7)
template <bool F32>
__device__ __forceinline__ float unit_act(int act, float g, float u, float limit, float alpha) {
  if (act == 2) g = fminf(g, limit), u = fminf(fmaxf(u, -limit), limit) + 1.0f;
  const float y = act == 0 ? g : act == 1 ? gelu_arg(g) : alpha * g;
  return g * (F32 ? sigmoidf_(y) : __builtin_amdgcn_rcpf(1.0f + exp2_(-1.4426950408889634f * y))) * u;
}

// tanh, relative error about 1e-6: its series through x^7 below 1/4 (4e-7 of it are left out there), 1 - 2 / (1 + e^2x) from there
// on (1.1e-6 at 1/4, where 0.76 is taken from 1 and exp2 and the reciprocal are each off by their last bit; less beyond.  At 1/16
// it would be 4.5e-6)
__device__ __forceinline__ float tanh_(float x) {
  const float q = x * x;
  const float near = x * fmaf(q, fmaf(q, fmaf(q, -17.0f / 315.0f, 2.0f / 15.0f), -1.0f / 3.0f), 1.0f);
  const float far = 1.0f - 2.0f * __builtin_amdgcn_rcpf(1.0f + exp2_(2.8853900817779268f * x));
  return fabsf(x) < 0.25f ? near : far;
}

}  // namespace sm
