// The weighted sum of a token's chosen experts as the norm kernels that add it to the residual stream read it: the experts' results stay
// where the products left them, and no [T, W] sum is written and read between.
#pragma once

#include "hybrid_common.h"

namespace llmctl_hybrid {

struct ExpertRows {
  const void* y;  // [T * top, W], fp32 (few tokens) or bf16; rows of experts without weights are not written
  const int* idx;  // [T, top]
  const float* wgt;  // [T, top]
  const bf16_t* x;  // [T, W]: what an expert without weights (idx >= E) gives
  long ldx;
  const bf16_t* shared;  // [T, W] or null, times sigmoid(gate [T, 1]) if given
  long ld_shared;
  const bf16_t* gate;
  long ld_gate;
  int E, top;
};

// Checks the operands of a sum and describes them; ``sizes``: of the sum.
ExpertRows expert_rows_of(const at::Tensor& y, const at::Tensor& idx, const at::Tensor& wgt, const at::Tensor& x,
                          const c10::optional<at::Tensor>& shared, const c10::optional<at::Tensor>& gate, int64_t experts);

// sum_k w_k y_k (+ the shared expert) of row r: quads threadIdx.x + i * NT of it (those beyond the row repeat its last one).  The experts'
// indices are only needed once their rows are there, so nothing waits for them.
template <typename Y, int NT, int VQ>
__device__ __forceinline__ void expert_sum_quads(const ExpertRows& m, int64_t r, int W, float4 (&s)[VQ]) {
#pragma unroll
  for (int i = 0; i < VQ; ++i) s[i] = make_float4(0.f, 0.f, 0.f, 0.f);
  float4 sv[VQ];
  float gate = 0.f;
  if (m.shared != nullptr) {  // (asked for with the rest, used last)
    if (m.gate != nullptr) gate = ldf(m.gate + r * m.ld_gate);
#pragma unroll
    for (int i = 0; i < VQ; ++i) sv[i] = ld4(m.shared + r * m.ld_shared + min((int)(threadIdx.x + i * NT) * 4, W - 4));
  }
  for (int k0 = 0; k0 < m.top; k0 += 2) {
    float4 v[2][VQ];
    int id[2];
    float w[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int64_t en = r * m.top + min(k0 + u, m.top - 1);
      id[u] = m.idx[en];
      w[u] = m.wgt[en];
#pragma unroll
      for (int i = 0; i < VQ; ++i) v[u][i] = ld4(static_cast<const Y*>(m.y) + en * W + min((int)(threadIdx.x + i * NT) * 4, W - 4));
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      if (k0 + u >= m.top) break;
#pragma unroll
      for (int i = 0; i < VQ; ++i) {
        if (id[u] >= m.E) v[u][i] = ld4(m.x + r * m.ldx + min((int)(threadIdx.x + i * NT) * 4, W - 4));
        s[i].x = fmaf(w[u], v[u][i].x, s[i].x), s[i].y = fmaf(w[u], v[u][i].y, s[i].y);
        s[i].z = fmaf(w[u], v[u][i].z, s[i].z), s[i].w = fmaf(w[u], v[u][i].w, s[i].w);
      }
    }
  }
  if (m.shared != nullptr) {
    const float g = m.gate != nullptr ? 1.0f / (1.0f + expf(-gate)) : 1.0f;
#pragma unroll
    for (int i = 0; i < VQ; ++i) {
      s[i].x = fmaf(g, sv[i].x, s[i].x), s[i].y = fmaf(g, sv[i].y, s[i].y), s[i].z = fmaf(g, sv[i].z, s[i].z), s[i].w = fmaf(g, sv[i].w, s[i].w);
    }
  }
}

}  // namespace llmctl_hybrid
