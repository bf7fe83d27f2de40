// Projections of a few rows (decode steps): see ../stream_linear.h.
#include "hybrid_common.h"
#include "stream_linear_launch.h"

namespace llmctl_hybrid {

// act(x w^T + bias): x bf16 [M <= 32, K] (row-strided views allowed), w bf16 [N, K], bias bf16 [N]; act 0 none, 1 gelu, 2 gelu (tanh), 3 relu^2, on the first
// act_cols columns.
at::Tensor rows_linear(const at::Tensor& x, const at::Tensor& w, const c10::optional<at::Tensor>& bias, int64_t act, int64_t act_cols, bool f32) {
  HYB_CHECK(x.is_cuda() && w.is_cuda() && x.dim() == 2 && w.dim() == 2 && x.scalar_type() == at::kBFloat16 && w.scalar_type() == at::kBFloat16,
            "rows_linear: bf16 GPU matrices");
  const int64_t M = x.size(0), K = x.size(1), N = w.size(0);
  HYB_CHECK(M <= 32 && w.size(1) == K && K % 8 == 0 && K > 0 && x.stride(1) == 1 && w.stride(1) == 1 && x.stride(0) % 8 == 0 && w.stride(0) % 8 == 0 &&
                reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0 && reinterpret_cast<uintptr_t>(w.data_ptr()) % 16 == 0,
            "rows_linear: at most 32 rows, K a multiple of 8, rows aligned to 16 bytes");
  if (bias.has_value())
    HYB_CHECK(bias->is_cuda() && bias->scalar_type() == at::kBFloat16 && bias->is_contiguous() && bias->numel() == N, "rows_linear: bias bf16 [N]");
  HYB_CHECK(act >= 0 && act <= 3, "rows_linear: act 0 .. 3");
  c10::DeviceGuard guard(x.device());
  at::Tensor y = at::empty({M, N}, x.options().dtype(f32 ? at::kFloat : at::kBFloat16));
  if (M == 0 || N == 0) return y;
  stream_linear::Args a{reinterpret_cast<const bf16_t*>(x.data_ptr()), (long)x.stride(0), reinterpret_cast<const bf16_t*>(w.data_ptr()), (long)w.stride(0),
                        bias.has_value() ? reinterpret_cast<const bf16_t*>(bias->data_ptr()) : nullptr, y.data_ptr(), (int)M, (int)N, (int)K, (int)act,
                        (int)act_cols,
                        f32 ? 1 : 0};
  stream_linear::launch(a, cur_stream());
  return y;
}

// x w^T as fp32 sums over ``parts`` ranges of K, [parts or fewer, M, N], for norm_add_parts_f32_
at::Tensor rows_parts(const at::Tensor& x, const at::Tensor& w, int64_t parts) {
  HYB_CHECK(x.is_cuda() && w.is_cuda() && x.dim() == 2 && w.dim() == 2 && x.scalar_type() == at::kBFloat16 && w.scalar_type() == at::kBFloat16,
            "rows_parts: bf16 GPU matrices");
  const int64_t M = x.size(0), K = x.size(1), N = w.size(0);
  HYB_CHECK(M <= 32 && w.size(1) == K && K % 8 == 0 && K > 0 && x.stride(1) == 1 && w.stride(1) == 1 && x.stride(0) % 8 == 0 && w.stride(0) % 8 == 0 &&
                reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0 && reinterpret_cast<uintptr_t>(w.data_ptr()) % 16 == 0,
            "rows_parts: at most 32 rows, K a multiple of 8, rows aligned to 16 bytes");
  HYB_CHECK(parts >= 1 && parts <= 16, "rows_parts: 1 .. 16 ranges");
  c10::DeviceGuard guard(x.device());
  const int64_t part = ((K + parts - 1) / parts + 31) / 32 * 32;
  at::Tensor y = at::empty({(K + part - 1) / part, M, N}, x.options().dtype(at::kFloat));
  if (M == 0 || N == 0) return y;
  stream_linear::Args a{reinterpret_cast<const bf16_t*>(x.data_ptr()), (long)x.stride(0), reinterpret_cast<const bf16_t*>(w.data_ptr()), (long)w.stride(0),
                        nullptr, y.data_ptr(), (int)M, (int)N, (int)K, 0, 0, 1};
  stream_linear::launch_parts(a, (int)parts, cur_stream());
  return y;
}

namespace {
// y [T, N] fp32 = x [T, K] bf16 times w [N, K] fp32, T <= 32: a recurrence's gates, whose weights stay fp32.  A workgroup per output, eight columns to a thread
// and turn, all rows' loads in flight; bound by the one round trip and the launch.  16 rows 8 x 2048 in a graph: the library's fp32 product 11.4 us and a cast
// of x 5.1, so 4.9.
template <int MT>
__global__ __launch_bounds__(256) void rows_f32w_kernel(const bf16_t* __restrict__ x, long ldx, const float* __restrict__ w, float* __restrict__ y, int T, int N,
                                                        int K) {
  __shared__ float red[MT][256 + 1];
  const int n = blockIdx.x, tid = threadIdx.x;
  float acc[MT] = {};
  for (int c = tid * 8; c < K; c += 256 * 8) {
    const float4 a = *reinterpret_cast<const float4*>(w + (long)n * K + c), b = *reinterpret_cast<const float4*>(w + (long)n * K + c + 4);
    const float wv[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    uint4 v[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) v[t] = *reinterpret_cast<const uint4*>(x + min(t, T - 1) * ldx + c);
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      const unsigned u[4] = {v[t].x, v[t].y, v[t].z, v[t].w};
#pragma unroll
      for (int j = 0; j < 4; ++j)
        acc[t] = fmaf(__uint_as_float(u[j] & 0xffff0000u), wv[2 * j + 1], fmaf(__uint_as_float(u[j] << 16), wv[2 * j], acc[t]));
    }
  }
#pragma unroll
  for (int t = 0; t < MT; ++t) red[t][tid] = acc[t];
  __syncthreads();
  for (int t = tid / 16; t < MT; t += 16) {
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) s += red[t][(tid & 15) + 16 * i];
#pragma unroll
    for (int o = 8; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if ((tid & 15) == 0 && t < T) y[(long)t * N + n] = s;
  }
}
}  // namespace

at::Tensor rows_f32w(const at::Tensor& x, const at::Tensor& w) {
  HYB_CHECK(x.is_cuda() && w.is_cuda() && x.dim() == 2 && w.dim() == 2 && x.scalar_type() == at::kBFloat16 && w.scalar_type() == at::kFloat &&
                w.is_contiguous() && w.size(1) == x.size(1),
            "rows_f32w: x bf16 [T, K], w contiguous fp32 [N, K]");
  const int64_t T = x.size(0), K = x.size(1), N = w.size(0);
  HYB_CHECK(T <= 32 && K % 8 == 0 && x.stride(1) == 1 && x.stride(0) % 8 == 0 && reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0 &&
                reinterpret_cast<uintptr_t>(w.data_ptr()) % 16 == 0,
            "rows_f32w: at most 32 rows, K a multiple of 8, rows aligned to 16 bytes");
  c10::DeviceGuard guard(x.device());
  at::Tensor y = at::empty({T, N}, w.options());
  if (T == 0 || N == 0) return y;
  auto go = [&](auto kern) {
    kern<<<dim3((unsigned)N), 256, 0, cur_stream()>>>(reinterpret_cast<const bf16_t*>(x.data_ptr()), (long)x.stride(0), w.data_ptr<float>(), y.data_ptr<float>(),
                                                      (int)T, (int)N, (int)K);
  };
  if (T <= 4) go(rows_f32w_kernel<4>);
  else if (T <= 16) go(rows_f32w_kernel<16>);
  else go(rows_f32w_kernel<32>);
  return y;
}

}  // namespace llmctl_hybrid
