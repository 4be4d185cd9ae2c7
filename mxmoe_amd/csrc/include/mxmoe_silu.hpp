// silu(gate) * up in the arithmetic that the activation quantisers and the gate_up epilogues share.
#pragma once
#include <hip/hip_runtime.h>

namespace mxmoe {

// Keeps a freshly computed fp32 value opaque to the optimiser.  Without it the compiler folds "fp32 multiply, then convert to
// fp16" into one v_fma_mixlo_f16, which rounds the exact product once; the reference arithmetic (and its CPU restatement) rounds
// to fp32 first and to fp16 second, and the two differ on ties.
__device__ __forceinline__ float keep_f32(float v) {
  asm("" : "+v"(v));  // not volatile: it may be scheduled freely, it just cannot be looked through
  return v;
}

// silu(g) = g / (1 + exp(-g)) as a fixed sequence of correctly rounded fp32 operations and exact integer ones, identical to the CPU
// restatement (every multiply-add is fused: one rounding): exp(-g) = 2^t with t = clamp(-g log2(e), +-100) split into k = rint(t) and
// f = t - k (exact), 2^f by a degree-4 Horner polynomial (relative error 3.7e-6), 2^k added to the exponent field (the result stays a
// normal number); the reciprocal of d = 1 + exp(-g) from an integer-subtraction seed (within 5.06 %) and two Newton steps (7e-6).
// silu(g) * u rounded to fp16 lies within 0.52 fp16 ulp of the exact value for every fp16 g.
__device__ __forceinline__ float silu_fixed(float g) {
  float t = g * -1.4426950408889634f;
  t = fminf(fmaxf(t, -100.0f), 100.0f);
  const float k = rintf(t);
  const float f = t - k;
  float p = 0.00967604f;
  p = __builtin_fmaf(p, f, 0.05592204f);
  p = __builtin_fmaf(p, f, 0.24022107f);
  p = __builtin_fmaf(p, f, 0.693121f);
  p = __builtin_fmaf(p, f, 1.0000001f);
  const float e = __int_as_float(__float_as_int(p) + (int)((unsigned)(int)k << 23));
  const float d = 1.0f + e;
  float r = __int_as_float(0x7EF31000 - __float_as_int(d));
  r = __builtin_fmaf(r, __builtin_fmaf(-d, r, 1.0f), r);
  r = __builtin_fmaf(r, __builtin_fmaf(-d, r, 1.0f), r);
  return g * r;
}

// round_to_half(silu(g) * u) of two values that are fp16 numbers
__device__ __forceinline__ _Float16 silu_mul_half(_Float16 g, _Float16 u) { return (_Float16)keep_f32(silu_fixed((float)g) * (float)u); }

}  // namespace mxmoe
