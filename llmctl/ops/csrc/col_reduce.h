// Column sums: the last stage, shared by the norms' weight gradients (norm.hip) and the bias gradients (col_sum.hip).
#pragma once
#include "common.h"

namespace llmctl {
namespace {

struct ColReduceArgs {
  const float* part[2];  // [P, H] fp32 partial rows of up to two sums of one launch (blockIdx.y)
  void* out[2];          // [H], bf16 or fp32
  int add[2];            // out += sum instead of out = sum
  int P, H;
};

// out[c] (+)= sum_p part[p, c].  Block: 64 columns x 16 waves; wave w takes rows w, w + 16, ... (4 independent loads in flight per
// lane), the waves meet in LDS.  Latency-bound (12 blocks at 768 columns): with 4 waves per block and one launch per sum, 256 rows x
// 768 columns took 6.9 us, twice per LayerNorm; this takes 4 for both.
template <typename T>
__global__ __launch_bounds__(1024) void col_reduce_kernel(ColReduceArgs a) {
  __shared__ float red[16][64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int c = blockIdx.x * 64 + lane, H = a.H, P = a.P;
  const float* part = a.part[blockIdx.y];
  float s0 = 0.f, s1 = 0.f, s2 = 0.f, s3 = 0.f;
  if (c < H) {
    int p = w;
    for (; p + 48 < P; p += 64) {
      s0 += part[(size_t)p * H + c];
      s1 += part[(size_t)(p + 16) * H + c];
      s2 += part[(size_t)(p + 32) * H + c];
      s3 += part[(size_t)(p + 48) * H + c];
    }
    for (; p < P; p += 16) s0 += part[(size_t)p * H + c];
  }
  red[w][lane] = (s0 + s1) + (s2 + s3);
  __syncthreads();
  if (w != 0 || c >= H) return;
  float s = 0.f;
#pragma unroll
  for (int k = 0; k < 16; ++k) s += red[k][lane];
  T* out = static_cast<T*>(a.out[blockIdx.y]) + c;
  if constexpr (sizeof(T) == 2) *out = f2bf(a.add[blockIdx.y] ? s + bf2f(*out) : s);
  else *out = a.add[blockIdx.y] ? s + *out : s;
}

// n sums (1 or 2); the outputs share a type
inline void launch_col_reduce(const ColReduceArgs& a, int n, bool f32, hipStream_t s) {
  const dim3 grid((unsigned)((a.H + 63) / 64), (unsigned)n);
  if (f32) hipLaunchKernelGGL((col_reduce_kernel<float>), grid, dim3(1024), 0, s, a);
  else hipLaunchKernelGGL((col_reduce_kernel<unsigned short>), grid, dim3(1024), 0, s, a);
}

// host: a column-sum output is a contiguous [H] vector of the parameter type or of fp32 main gradients
inline bool col_out_ok(const at::Tensor& t, int64_t H) {
  return t.is_cuda() && t.is_contiguous() && t.numel() == H && (t.scalar_type() == at::kBFloat16 || t.scalar_type() == at::kFloat);
}

}  // namespace
}  // namespace llmctl
