// What becomes of a gate and its up: the unit between the two projections of a gated feed-forward, for kernels that take it
// along on the way out of the first and store it as bfloat16. The same numbers as `silu_mul` of a bfloat16 product
// (GLU_SILU_ROUNDED) and `capped_glu` of 32-bit sums (the others) store, so that a unit does not depend on which kernel made it.
#pragma once
#include "attention_mfma.h"

// GLU_SIGMOID_LIBRARY: the sigmoid by the library's exponential and a division, for what comes between two routers, where a token whose scores lie close
// takes another expert once a rounding changes.
enum { GLU_SILU_ROUNDED, GLU_SIGMOID, GLU_RELU, GLU_GELU, GLU_SIGMOID_LIBRARY };

// g / (1 + e^z). With z = t ln 2 + rest, t rounded, e^z is p + p rest, p = 2^t (the hardware's, good to its last place); the denominator is 1 + p rounded,
// and what that leaves goes into the remainder that corrects g times the hardware's reciprocal (nothing where g is infinite). Beyond z = 87 the reciprocal
// is 0 instead of what lies below 2^-126. 1.7e7 gates of size 0.5 and 3, 2-norm of the error: slope 1 4.6e-8 and 4.9e-8 by the library's exponential and
// a division, 3.7e-8 and 3.6e-8 here; gelu 4.8e-8 and 3.8e-8 by its tanh, 3.9e-8 and 3.3e-8 here, in half as many instructions (a prompt of 2,048 through eight
// gate|up products of F 8,192 3,455 -> 3,403 us).
static __device__ __forceinline__ float glu_over_one_and_exp(float g, float z) {
  z = __builtin_amdgcn_fmed3f(z, -150.f, 88.5f);
  const float t = z * 1.44269504088896340736f;
  const float rest = fmaf(t, -(float)(0.69314718055994530942 - (double)0.693147182464599609375f), fmaf(t, -0.693147182464599609375f, z));
  const float p = __builtin_amdgcn_exp2f(t), d = 1.0f + p, r = __builtin_amdgcn_rcpf(d), q = g * r;
  const float left = fmaf(p, rest, p - (d - 1.0f));
  return fmaf(__builtin_amdgcn_fmed3f(fmaf(-q, left, fmaf(-q, d, g)), -3e38f, 3e38f), r, q);
}

// What the gate passes: g sigmoid(slope g), relu, or gelu in its tanh form, 0.5 g (1 + tanh(w)) = g sigmoid(2 w), w = sqrt(2 / pi) (g + 0.044715 g^3)
static __device__ __forceinline__ float glu_gate(int act, float g, float slope) {
  if (act == GLU_RELU) return fmaxf(g, 0.f);
  if (act == GLU_SIGMOID_LIBRARY) return g / (1.0f + expf(-slope * g));
  return glu_over_one_and_exp(g, g * (act == GLU_GELU ? fmaf(-2.f * 0.7978845608028654f * 0.044715f, g * g, -2.f * 0.7978845608028654f) : -slope));
}

static __device__ __forceinline__ float glu_capped(int act, float g, float u, float limit, float slope, float up_shift) {
  if (limit > 0.f) {
    g = fminf(g, limit);
    u = fminf(fmaxf(u, -limit), limit);
  }
  return glu_gate(act, g, slope) * (u + up_shift);
}
