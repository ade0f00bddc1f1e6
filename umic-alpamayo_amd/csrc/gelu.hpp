// The GELU epilogues of the linear kernels (gemm.hip, gemm_ks.hip, gemm_mid.hip),
// one definition so that every kernel gives the same bits.
#pragma once

#include "common.hpp"

namespace umic {

// Exact-erf GELU for the linear's epilogue, formed as eager does:
// GELU(x) = 0.5 * x * (1 + erf(x / sqrt2)) in fp32.  erf(|u|) is taken as
// 1 - erfc(|u|) rounded to fp32, with erfc(z) = t * exp(-z^2 + P(t)),
// t = 1 / (1 + z/2) -- the functional form of Numerical Recipes' erfcc
// (W. H. Press et al., 2nd ed., sec. 6.2).  The coefficients of P are this
// library's own least-squares fit in float64 of log(erfc(z) / t) + z^2 on
// z in [0, 10]; evaluated in fp32 with the hardware reciprocal and exp2,
// erfc is within 1.5e-5 relative on [0, 10], so the fp32 erf matches a
// correctly rounded erff to about an ulp (tests/test_gelu_epilogue.py
// re-checks these constants).  Forming 1 + erf in fp32 keeps eager's
// behaviour for very negative x, where it cancels to 0 or to one ulp of 1
// (the more accurate x/2 * erfc(|u|) would differ from eager there by many
// bf16 ulps).  About 17 VALU operations against the library erff's branches.
__device__ __forceinline__ float gelu_erf(float x) {
  const float z = __builtin_fabsf(x) * 0.70710678118654752f;
  const float t = __builtin_amdgcn_rcpf(1.0f + 0.5f * z);
  float p = 1.449302137e-01f;
  p = __builtin_fmaf(p, t, -6.808271779e-01f);
  p = __builtin_fmaf(p, t, 1.156733757e+00f);
  p = __builtin_fmaf(p, t, -6.962518993e-01f);
  p = __builtin_fmaf(p, t, -8.028043184e-02f);
  p = __builtin_fmaf(p, t, 1.267586182e-03f);
  p = __builtin_fmaf(p, t, 3.460280007e-02f);
  p = __builtin_fmaf(p, t, 3.866404121e-01f);
  p = __builtin_fmaf(p, t, 9.986327833e-01f);
  p = __builtin_fmaf(p, t, -1.265447997e+00f);
  const float erfc_z = t * __builtin_amdgcn_exp2f((p - z * z) * 1.4426950408889634f);
  const float erf_abs = 1.0f - erfc_z;
  return 0.5f * x * (1.0f + (x < 0.0f ? -erf_abs : erf_abs));
}

// tanh-approximate GELU, as torch's gelu(approximate="tanh") (HF
// gelu_pytorch_tanh, the Qwen3-VL ViT MLP's activation) forms it in fp32:
// 0.5 x (1 + tanh(y)), y = sqrt(2/pi) (x + 0.044715 x^3) in the same
// operation order.  tanh|y| = 1 - 2 / (1 + exp(2|y|)) with the hardware exp2
// and reciprocal: the final subtraction puts it on the fp32 grid of [0.5, 1),
// as tanhf's result, so 1 + tanh(y) cancels in the negative tail exactly as
// eager's does; it is exactly 1 where exp overflows.
__device__ __forceinline__ float gelu_tanh(float x) {
  const float y = 0.7978845608028654f * (x + 0.044715f * (x * x * x));
  const float e = __builtin_amdgcn_exp2f(__builtin_fabsf(y) * 2.8853900817779268f);  // exp(2|y|)
  // 2 r is exact, so the fma rounds as 1 - 2 r does
  const float th_abs = __builtin_fmaf(-2.0f, __builtin_amdgcn_rcpf(1.0f + e), 1.0f);
  return 0.5f * x * (1.0f + __builtin_copysignf(th_abs, y));
}

}  // namespace umic
