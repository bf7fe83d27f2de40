#pragma once
#include <hip/hip_runtime.h>

namespace llmctl {
// Sums and maxima over the 64 lanes (all of them active), in the order of exchanges with the lanes 32, 16, 8, 4, 2 and 1 away: two half-wave swaps, then rotations inside a
// row of 16, after each of which the row repeats itself.  Through LDS (ds_bpermute) every exchange waited for a round trip; rows of few launches are chains of
// such waits (16 rows of 2048, norm and router: 8.2 us, so and with the router's weight asked for first 6.6; a decode step of five layers 283 us, so 276).
template <int N>
__device__ __forceinline__ float row_ror(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x120 + N, 0xf, 0xf, true));
}
template <typename F>
__device__ __forceinline__ float wave_fold(float v, F&& f) {
  const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = f(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = f(__uint_as_float(b[0]), __uint_as_float(b[1]));
  v = f(v, row_ror<8>(v));
  v = f(v, row_ror<4>(v));
  v = f(v, row_ror<2>(v));
  return f(v, row_ror<1>(v));
}
__device__ __forceinline__ float wave_sum(float v) {
  return wave_fold(v, [](float x, float y) { return x + y; });
}
__device__ __forceinline__ float wave_max(float v) {
  return wave_fold(v, [](float x, float y) { return fmaxf(x, y); });
}
}  // namespace llmctl
