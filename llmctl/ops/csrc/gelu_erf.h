#pragma once
#include <hip/hip_runtime.h>

namespace llmctl {
// The erf GELU 0.5 x (1 + erf(x / sqrt 2)) = 0.5 x + 0.5 |x| (1 - e), e = erfc(|x| / sqrt 2) = 2^-q(|x|), with q(a) = a r(a) and r of degree 9, a least-maximum fit over a in
// [0, 8] of the error that it leaves in the result (6e-9 |x|) or, of what is left below 2e-5, in e itself.  e is near 1 where a is small, so nothing cancels there: within
// 7.3e-8 |x| of the exact value for any x, 1.6e-8 |x| in the root mean square (1 + erff, which rounds: 1.06e-7 and 2.1e-8), and to 4e-4 of a result down to x = -8, where 1 + erff
// has no digits from -5.6 on.  q grows beyond 8, so e is 0 from 14 on.  16 instructions where erff's two branches are 43: an epilogue has 144 of them, and erff's came from
// memory (a tile of 256 rows 14.3 us longer, so 3.9; 2911 tokens through 8 experts of width 2048 96, so 85).  Infinities and what is no number give what the form with erff gives.
__device__ __forceinline__ float gelu_erf(float x) {
  const float a = __builtin_fminf(__builtin_fabsf(x), 16.f);
  float r = 1.9735479e-08f;
  r = __builtin_fmaf(r, a, -6.64567438e-07f);
  r = __builtin_fmaf(r, a, 9.31520026e-06f);
  r = __builtin_fmaf(r, a, -6.91485402e-05f);
  r = __builtin_fmaf(r, a, 0.000260956527f);
  r = __builtin_fmaf(r, a, 2.91971337e-05f);
  r = __builtin_fmaf(r, a, -0.00697499095f);
  r = __builtin_fmaf(r, a, 0.0524571799f);
  r = __builtin_fmaf(r, a, 0.459216237f);
  r = __builtin_fmaf(r, a, 1.15110469f);
  return __builtin_fmaf(-0.5f * a, __builtin_amdgcn_exp2f(-(a * r)), __builtin_fmaf(0.5f, x, 0.5f * __builtin_fabsf(x)));
}
}  // namespace llmctl
