// Projections of a few rows with their bias and activation in the same launch: see stream_linear.h.
#include "common.h"
#include "stream_linear_launch.h"

namespace llmctl {

// act(x w^T + bias): x bf16 [M <= 32, K] (row-strided views allowed), w bf16 [N, K], bias bf16 [N]; act 0 none, 1 gelu (erf), 2 gelu (tanh),
// 3 relu^2.
at::Tensor stream_linear(const at::Tensor& x, const at::Tensor& w, const c10::optional<at::Tensor>& bias, int64_t act) {
  LLMCTL_CHECK(x.is_cuda() && w.is_cuda() && x.dim() == 2 && w.dim() == 2 && x.scalar_type() == at::kBFloat16 && w.scalar_type() == at::kBFloat16,
               "stream_linear: bf16 GPU matrices");
  const int64_t M = x.size(0), K = x.size(1), N = w.size(0);
  LLMCTL_CHECK(M <= 32 && w.size(1) == K && K % 8 == 0 && K > 0 && x.stride(1) == 1 && w.stride(1) == 1 && x.stride(0) % 8 == 0 && w.stride(0) % 8 == 0 &&
                   reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0 && reinterpret_cast<uintptr_t>(w.data_ptr()) % 16 == 0,
               "stream_linear: at most 32 rows, K a multiple of 8, rows aligned to 16 bytes");
  const bool has_bias = bias.has_value() && bias->defined();
  if (has_bias)
    LLMCTL_CHECK(bias->is_cuda() && bias->scalar_type() == at::kBFloat16 && bias->is_contiguous() && bias->numel() == N, "stream_linear: bias bf16 [N]");
  LLMCTL_CHECK(act >= 0 && act <= 3, "stream_linear: act 0 .. 3");
  const c10::DeviceGuard guard(x.device());
  at::Tensor y = at::empty({M, N}, x.options());
  if (M == 0 || N == 0) return y;
  ::stream_linear::Args a{bf_ptr(x), (long)x.stride(0), bf_ptr(w), (long)w.stride(0), has_bias ? bf_ptr(*bias) : nullptr, y.data_ptr(), (int)M, (int)N,
                          (int)K, (int)act, (int)N, 0};
  ::stream_linear::launch(a, stream());
  return y;
}

TORCH_LIBRARY_IMPL(llmctl, CUDA, m) { m.impl("stream_linear", &stream_linear); }

}  // namespace llmctl
