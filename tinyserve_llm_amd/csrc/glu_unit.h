// What becomes of a gate and its up: the unit between the two projections of a gated feed-forward, for kernels that take it
// along on the way out of the first and store it as bfloat16. The same numbers as `silu_mul` of a bfloat16 product
// (GLU_SILU_ROUNDED) and `capped_glu` of 32-bit sums (the others) store, so that a unit does not depend on which kernel made it.
#pragma once
#include "attention_mfma.h"

enum { GLU_SILU_ROUNDED, GLU_SIGMOID, GLU_RELU, GLU_GELU };

static __device__ __forceinline__ float glu_capped(int act, float g, float u, float limit, float slope, float up_shift) {
  if (limit > 0.f) {
    g = fminf(g, limit);
    u = fminf(fmaxf(u, -limit), limit);
  }
  u += up_shift;
  if (act == GLU_RELU) return fmaxf(g, 0.f) * u;
  if (act == GLU_GELU) return 0.5f * g * (1.0f + tanhf(0.7978845608028654f * (g + 0.044715f * g * g * g))) * u;
  return g / (1.0f + expf(-slope * g)) * u;
}
