// Activations and recurrence steps shared by the projections' epilogues and the row kernels; all in f32.
#pragma once

#include "nv_common.cuh"

namespace nv {

__device__ __forceinline__ float sigmoid(float v) { return 1.0f / (1.0f + expf(-v)); }
__device__ __forceinline__ float softplus(float v) { return v > 20.0f ? v : log1pf(expf(v)); }

// e^x for |x| <= 89 (infinity from 88.73 on): a whole power of two and the hardware's power of the fraction, which keeps the bits that the product by log2(e)
// would lose. (expf takes some more instructions for ranges that its callers here do not need.)
__device__ __forceinline__ float exp_bounded(float x) {
  constexpr float kLog2e = 1.44269504f, kRest = 1.92596299e-8f;   // log2(e) and what its f32 leaves of it
  const float whole = rintf(x * kLog2e);
  const float fraction = fmaf(x, kRest, fmaf(x, kLog2e, -whole));
  return ldexpf(__builtin_amdgcn_exp2f(fraction), static_cast<int>(whole));
}
// v / (1 + e^(-slope v)), the quotient by a reciprocal and one correction of it that takes 1 and the exponential apart (their rounded
// sum is off by as much as the division's rounding), in less than half the instructions of expf and a division. Against 64 bits,
// largest and mean error: slope 1 over -8 .. 8 1.50e-7 and 2.6e-8 (expf and a division 1.51e-7 and 3.2e-8), over -80 .. 80 1.46e-7 and
// 1.8e-8 (1.75e-7 and 1.9e-8), over -87.3 .. -80 1.28e-7 and 2.95e-8 (1.25e-7 and 2.93e-8: the hardware's power); slope 1.702 over
// -8 .. 8 5.9e-7 and 8.5e-8 (6.1e-7 and 9.4e-8).
// The reciprocal is of a quarter of the divisor: that of one past 2^126 (gates from -87.3 to -88.7, or so much less with a slope) is no
// normal number and would come out as 0. Infinities, NaN and gates whose exponential overflows come out as with a division, by
// the plain product: the correction would be NaN.
__device__ __forceinline__ float gated(float v, float slope) {
  const float e = exp_bounded(-fminf(fmaxf(slope * v, -89.0f), 89.0f));
  const float r = __builtin_amdgcn_rcpf(fmaf(0.25f, e, 0.25f)) * 0.25f;
  const float q = v * r, exact = fmaf(fmaf(-q, e, v) - q, r, q);
  return fmaxf(v, e) < INFINITY ? exact : q;
}
// Two results as one word, rounded by the hardware's conversions (a NaN stays one; its bits may differ from enc16's).
template <uint32_t DT>
__device__ __forceinline__ uint32_t enc16_pair(float lo, float hi) {
  if constexpr (DT == kBF16) {
    typedef __bf16 pair_t __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, pair_t{static_cast<__bf16>(lo), static_cast<__bf16>(hi)});
  } else {
    return enc16<DT>(lo) | (static_cast<uint32_t>(enc16<DT>(hi)) << 16);
  }
}

// e^z - 1 - z for z <= 0: the power series where the difference would cancel, else the difference.
__device__ __forceinline__ float exp_remainder(float z) {
  float s = fmaf(z, 1.0f / 3628800.0f, 1.0f / 362880.0f);
  s = fmaf(z, s, 1.0f / 40320.0f);
  s = fmaf(z, s, 1.0f / 5040.0f);
  s = fmaf(z, s, 1.0f / 720.0f);
  s = fmaf(z, s, 1.0f / 120.0f);
  s = fmaf(z, s, 1.0f / 24.0f);
  s = fmaf(z, s, 1.0f / 6.0f);
  s = fmaf(z, s, 0.5f);
  const float far = (exp_bounded(fmaxf(z, -87.0f)) - 1.0f) - z;
  return z > -1.0f ? z * z * s : far;
}

// xIELU: with two learned numbers (p, q), above zero softplus(p) z^2 + z / 2, at and below it
// (softplus(q) + 1/2) (e^z - 1 - z) + z / 2.
struct XieluParams {
  float above, below;
};
template <uint32_t DT>
__device__ __forceinline__ XieluParams xielu_params(const uint16_t *pq) {
  return XieluParams{softplus(dec16<DT>(pq[0])), 0.5f + softplus(dec16<DT>(pq[1]))};
}
__device__ __forceinline__ float xielu(float z, const XieluParams &a) {
  const float low = fminf(z, 0.0f);
  return (z > 0.0f ? a.above * z * z : a.below * exp_remainder(low)) + 0.5f * z;
}

// Gated linear unit with bounds: the gate from above, the linear part on both sides and moved up by one.
__device__ __forceinline__ float clamped_glu(float g, float u, float limit) {
  g = fminf(g, limit);
  u = fminf(fmaxf(u, -limit), limit);
  return gated(g, 1.702f) * (u + 1.0f);
}

// minGRU: gate and candidate from the current token alone (pre-activations with their biases added).
__device__ __forceinline__ float mingru_candidate(float u) { return u >= 0.0f ? u + 0.5f : sigmoid(u); }
__device__ __forceinline__ float mingru_step(float z_pre, float u, float state) {
  const float z = sigmoid(z_pre);
  return (1.0f - z) * state + z * mingru_candidate(u);
}

}  // namespace nv
