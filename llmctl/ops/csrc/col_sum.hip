// Bias gradients: column sums of bf16 rows, straight into the gradient vector.
//
// Bound: one pass over the rows.  Every block sums up to ``rows`` rows of 256 columns (8 rows of 512 bytes at a time, four such
// steps in flight) and writes one fp32 partial row; col_reduce_kernel adds the partial rows in a fixed order (no atomics, so the
// same bits every time) into the parameter's gradient.  Blocks are about four per CU, and no fewer than 32 rows each.
// Measured on one MI355X, 8192 rows, against the library's reduction: 768 columns
// 5.7 us (18.7), 2304 columns 8.7 (24.4), 3072 columns 11.1 (24.5: 4.5 TB/s now); 256 rows x 768 columns 3.9 (8.6).
#include "col_reduce.h"

namespace llmctl {
namespace {
constexpr int CS_COLS = 256, CS_ROWS = 32;

__global__ __launch_bounds__(256) void col_sum_kernel(const unsigned short* __restrict__ x, long stride, int T, int N, int rows,
                                                      float* __restrict__ part) {
  __shared__ __attribute__((aligned(16))) float red[8][CS_COLS];
  const int c8 = (threadIdx.x & 31) * 8, slot = threadIdx.x >> 5;
  const int col = blockIdx.x * CS_COLS + c8;
  const int r0 = blockIdx.y * rows, r1 = min(T, r0 + rows);
  float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  if (col < N) {
    int r = r0 + slot;
    for (; r + 24 < r1; r += 32) {
      bf16x8 v[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = *reinterpret_cast<const bf16x8*>(x + (long)(r + 8 * i) * stride + col);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 8; ++j) s[j] += bf2f(v[i][j]);
    }
    for (; r < r1; r += 8) {
      const bf16x8 v = *reinterpret_cast<const bf16x8*>(x + (long)r * stride + col);
#pragma unroll
      for (int j = 0; j < 8; ++j) s[j] += bf2f(v[j]);
    }
  }
  *reinterpret_cast<float4*>(&red[slot][c8]) = make_float4(s[0], s[1], s[2], s[3]);
  *reinterpret_cast<float4*>(&red[slot][c8 + 4]) = make_float4(s[4], s[5], s[6], s[7]);
  __syncthreads();
  const int c = blockIdx.x * CS_COLS + threadIdx.x;
  if (c >= N) return;
  float t = 0.f;
#pragma unroll
  for (int k = 0; k < 8; ++k) t += red[k][threadIdx.x];
  part[(size_t)blockIdx.y * N + c] = t;
}
}  // namespace

// out (+)= sum over the rows of x [T, N] (unit column stride)
void col_sum_(const at::Tensor& x, at::Tensor out, bool add) {
  LLMCTL_CHECK(x.is_cuda() && x.dim() == 2 && x.scalar_type() == at::kBFloat16 && x.size(0) > 0 && x.stride(1) == 1 && x.size(1) % 8 == 0 &&
                   x.stride(0) % 8 == 0 && (reinterpret_cast<uintptr_t>(x.data_ptr()) & 15) == 0,
               "col_sum: bf16 rows, 16-byte aligned, a multiple of 8 wide");
  LLMCTL_CHECK(x.size(0) < (1 << 30) && x.size(1) < (1 << 30), "col_sum: sizes");
  const int T = (int)x.size(0), N = (int)x.size(1);
  LLMCTL_CHECK(col_out_ok(out, N), "col_sum: the output is a contiguous bf16 or fp32 vector of the row's length");
  const c10::DeviceGuard g(x.device());
  const int cb = (N + CS_COLS - 1) / CS_COLS;
  const int want = std::max(1, std::min((T + CS_ROWS - 1) / CS_ROWS, std::max(1, 4 * num_cus() / cb)));
  const int rows = (((T + want - 1) / want + CS_ROWS - 1) / CS_ROWS) * CS_ROWS;
  const int P = (T + rows - 1) / rows;
  auto part = at::empty({P, N}, x.options().dtype(at::kFloat));
  auto s = stream();
  hipLaunchKernelGGL(col_sum_kernel, dim3((unsigned)cb, (unsigned)P), dim3(256), 0, s, bf_ptr(x), (long)x.stride(0), T, N, rows,
                     part.data_ptr<float>());
  launch_col_reduce(ColReduceArgs{{part.data_ptr<float>(), nullptr}, {out.data_ptr(), nullptr}, {add, 0}, P, N}, 1,
                    out.scalar_type() == at::kFloat, s);
}

TORCH_LIBRARY_IMPL(llmctl, CUDA, m) { m.impl("col_sum_", &col_sum_); }

}  // namespace llmctl
