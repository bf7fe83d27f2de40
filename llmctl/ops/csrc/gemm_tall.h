// Products on 256 x 128 tiles (gemm_tall.hip), for gemm64's dispatch
#pragma once
#include <ATen/ATen.h>

namespace llmctl {
int gemm_tall_splits(long M, long N, long K, long n_main, long n_tail, int splits, double* us_of = nullptr);
int64_t gemm_tall_back_splits(int64_t T, int64_t O, int64_t I, bool bias, double two_us);
void gemm_tall(const at::Tensor& a, const at::Tensor& b, at::Tensor out, bool at_, bool accumulate, int64_t splits, const c10::optional<at::Tensor>& bias = c10::nullopt,
               bool bias_add = false);
}  // namespace llmctl
