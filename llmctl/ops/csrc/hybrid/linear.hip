// Projections of a few rows (decode steps): see ../stream_linear.h.
#include "hybrid_common.h"
#include "stream_linear.h"

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

}  // namespace llmctl_hybrid
