// Chunked recurrences on the fp32 matrix cores (MFMA 16x16x4): the block products that memory.hip, mlstm_chunk.hip and gla_chunk.hip
// share.  All products run in fp32.  A step j of such a product takes logical index 4 g + j of a 16-wide block from lane group
// g = lane / 16 on both sides, so that a lane's A operands are 16 neighbouring bytes and a result (rows 4 g + r, column lane % 16)
// is a B operand as it stands: values, solved rows and memories stay in registers from product to product, and only K, Q and the
// score blocks go through LDS.  A wave owns 16 value columns.
#pragma once
#include "hybrid_common.h"

#include <type_traits>

namespace llmctl_hybrid {
namespace {
using f32x4 = float __attribute__((ext_vector_type(4)));

constexpr int CH = 64;            // tokens per chunk
constexpr int AS = CH + 4;        // row stride of the score blocks in LDS

__device__ __forceinline__ f32x4 mfma4(float x, float y, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(x, y, c, 0, 0, 0); }
__device__ __forceinline__ f32x4 lds4(const float* p) { return *reinterpret_cast<const f32x4*>(p); }

// acc += X Y over one 16-wide block: x4 the lane's four A operands, y its four B operands
__device__ __forceinline__ f32x4 block_product(f32x4 x4, f32x4 y, f32x4 acc) {
#pragma unroll
  for (int j = 0; j < 4; ++j) acc = mfma4(x4[j], y[j], acc);
  return acc;
}

// n rows of one head to LDS as fp32 [CH][dkp + 4]; rows past n and columns past dk become zeros
template <typename T>
__device__ __forceinline__ void stage_rows(float* dst, int stride, const T* src, int64_t st, int n, int dk, int dkp, bool vec) {
  const int nt = blockDim.x;
  if (vec) {
    const int per = dkp / 4;
    for (int e = threadIdx.x; e < CH * per; e += nt) {
      const int r = e / per, c = (e - r * per) * 4;
      float4 x = make_float4(0.f, 0.f, 0.f, 0.f);
      if (r < n && c < dk) {
        const T* p = src + (int64_t)r * st + c;
        if constexpr (sizeof(T) == 4) {
          x = *reinterpret_cast<const float4*>(p);
        } else {
          const uint2 w = *reinterpret_cast<const uint2*>(p);
          x = make_float4(__uint_as_float(w.x << 16), __uint_as_float(w.x & 0xffff0000u), __uint_as_float(w.y << 16),
                          __uint_as_float(w.y & 0xffff0000u));
        }
      }
      *reinterpret_cast<float4*>(dst + r * stride + c) = x;
    }
  } else {
    for (int e = threadIdx.x; e < CH * dkp; e += nt) {
      const int r = e / dkp, c = e - r * dkp;
      dst[r * stride + c] = (r < n && c < dk) ? ldf(src + (int64_t)r * st + c) : 0.f;
    }
  }
}

__device__ __forceinline__ void lower_tile(int i, int& ti, int& tj) {  // the ten 16 x 16 tiles on and below the diagonal
  ti = i < 1 ? 0 : (i < 3 ? 1 : (i < 6 ? 2 : 3));
  tj = i - ti * (ti + 1) / 2;
}

// one score tile: rows 16 ti .. of X against rows 16 tj .. of Y (both [CH][ks] in LDS)
template <int NKK>
__device__ __forceinline__ f32x4 score_tile(const float* X, const float* Y, int ks, int nkk, int ti, int tj, int lane) {
  const float* xr = X + (16 * ti + (lane & 15)) * ks + (lane >> 4) * 4;
  const float* yr = Y + (16 * tj + (lane & 15)) * ks + (lane >> 4) * 4;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  if constexpr (NKK > 0) {
#pragma unroll
    for (int kk = 0; kk < NKK; ++kk) acc = block_product(lds4(xr + 16 * kk), lds4(yr + 16 * kk), acc);
  } else {
    for (int kk = 0; kk < nkk; ++kk) acc = block_product(lds4(xr + 16 * kk), lds4(yr + 16 * kk), acc);
  }
  return acc;
}

int waves_for(int dv) { return dv > 64 ? 8 : 4; }

// channels that a chunk's keys take in LDS: the compile-time widths 32, 64 and 128, else filled up to 16
int staged_width(int dk) { return dk <= 32 ? 32 : (dk <= 64 ? 64 : (dk <= 128 && dk > 96 ? 128 : (dk + 15) / 16 * 16)); }
template <typename F>
void by_width(int dk, F&& f) {
  if (dk <= 32) f(std::integral_constant<int, 2>());
  else if (dk <= 64) f(std::integral_constant<int, 4>());
  else if (dk <= 128 && dk > 96) f(std::integral_constant<int, 8>());
  else f(std::integral_constant<int, 0>());
}

}  // namespace
}  // namespace llmctl_hybrid
