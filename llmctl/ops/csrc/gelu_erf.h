#pragma once
#include <hip/hip_runtime.h>

namespace llmctl {
// The erf GELU of a result that is rounded to bf16: 0.5 x (1 + erf(x / sqrt 2)) = 0.5 x + 0.5 |x| (1 - 2 h), h = 0.5 erfc(z), z = |x| / sqrt 2.  erfc(z) is
// e^(-z^2) t p(t) with t = 1 / (1 + 0.33 z) and p of degree 7, a least-maximum fit of the relative error over z in [0, 10] (9.4e-8).  In fp32 it is within 2.3e-7 |x| of
// the exact value for any x (1 + erff, which rounds: 1.1e-7 |x|), and the tail keeps its digits.  Some 22 instructions where erff's two branches are 43; infinities and what is no
// number give what that form gives.
__device__ __forceinline__ float gelu_erf16(float x) {
  const float a = __builtin_fminf(__builtin_fabsf(x), 100.f);  // (e^(-z^2) is 0 from 14 on)
  const float t = __builtin_amdgcn_rcpf(__builtin_fmaf(0.33f * 0.70710678118654752440f, a, 1.f));
  float p = -0.13534443f;
  p = __builtin_fmaf(p, t, 0.460232079f);
  p = __builtin_fmaf(p, t, -0.351141359f);
  p = __builtin_fmaf(p, t, 0.408492589f);
  p = __builtin_fmaf(p, t, 0.0472244295f);
  p = __builtin_fmaf(p, t, 0.201222778f);
  p = __builtin_fmaf(p, t, 0.182956115f);
  p = __builtin_fmaf(p, t, 0.186357792f);
  const float e = __builtin_amdgcn_exp2f(a * (-0.72134752044448170f * a));
  return __builtin_fmaf(0.5f, x, 0.5f * __builtin_fabsf(x)) - 0.5f * a * t * (p * e);
}
}  // namespace llmctl
