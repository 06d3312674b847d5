// What the delta-net layer does to a row before the recurrence, shared by the passes over
// whole rows and the kernels that do it on the way: SiLU, the four-tap convolution and the
// gates, with every bf16 rounding point of the reference
// (src/llm/layers/sequence_delta_net.cc:31-51,88-96).
#pragma once

#include "gdn.h"
#include "mfma_tile.h"

namespace pluto_hip {

// x / (1 + exp(-x)) from the hardware's exponential and reciprocal, with the correction
// and the last instruction of a division, which restores what the others make of
// infinities.  The uncorrected product rounds 5.9375, whose value lies next to a tie, to the
// wrong bf16 (0.1 % of the activations where inputs have four times unit size: states 2 %
// further from the specification); with it every bf16 argument above -87 rounds as with
// expf and a division.
__device__ inline float silu(float x) {
  const float d = 1.0f + __builtin_amdgcn_exp2f(-x * kLog2e);
  const float inverse = __builtin_amdgcn_rcpf(d), y = x * inverse;
  return __builtin_amdgcn_div_fixupf(__builtin_fmaf(__builtin_fmaf(-y, d, x), inverse, y), d, x);
}

// The same for a bf16 argument whose result is rounded to bf16 at once, without the
// correction: the 1 of the denominator is the next FP32 number above it, which moves the one
// argument whose quotient lies next to a tie (5.9375) to its right side.  All 65536 arguments
// round as silu's results do.
__device__ inline float silu_of_bf16(float x) {
  return x * __builtin_amdgcn_rcpf(0x1.000002p0f + __builtin_amdgcn_exp2f(-x * kLog2e));
}

// Two channels of a row of the convolution and its activation, packed: taps of rows t - 3 .. t.
__device__ inline uint32_t convolved_pair(const float (&x0)[4], const float (&w0)[4], const float (&x1)[4],
                                          const float (&w1)[4]) {
  float first = 0.0f, second = 0.0f;
#pragma unroll
  for (int tap = 0; tap < 4; ++tap) first += x0[tap] * w0[tap], second += x1[tap] * w1[tap];
  const uint32_t sums = pack_bf16(first, second);
  return pack_bf16(silu_of_bf16(__uint_as_float(sums << 16)), silu_of_bf16(__uint_as_float(sums & 0xffff0000u)));
}

// alpha: the token's a plus the head's dt_bias.  Stable softplus: no overflow for strongly
// positive time steps.
__device__ inline float log_decay_of(float alpha, float a_log) {
  const float softplus = fmaxf(alpha, 0.0f) + log1pf(expf(-fabsf(alpha)));
  return -expf(a_log) * softplus;
}
__device__ inline float beta_of(float b) { return 1.0f / (1.0f + expf(-b)); }

}  // namespace pluto_hip
