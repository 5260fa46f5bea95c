// Activations and logarithms that the recurrent mixers' kernels share.
#pragma once
#include "common.h"

#define RC_MAX_LAGS 7        // a convolution has at most 8 taps

__device__ __forceinline__ float rc_silu(float z) { return z / (1.f + expf(-z)); }
__device__ __forceinline__ float rc_softplus(float z) { return z > 20.f ? z : log1pf(expf(z)); }

// log(1 + e^-a) for a >= 0: u = 1 + e rounded, and log(u) e / (u - 1) takes that rounding back (Kahan's log1p), so the
// hardware's logarithm and exponential give the result to a few units in the last place.
__device__ __forceinline__ float softplus_of_negative(float a) {
  const float e = __builtin_amdgcn_exp2f(-a * 1.4426950408889634f);
  const float u = 1.f + e, d = u - 1.f;
  return d > 0.f ? __builtin_amdgcn_logf(u) * 0.6931471805599453f * (e * __builtin_amdgcn_rcpf(d)) : e;
}
