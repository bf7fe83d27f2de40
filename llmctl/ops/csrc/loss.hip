// Fused softmax cross-entropy (gfx950).
//
// Forward: one 256-thread block per token row, single pass over the [V] bf16 logits with
// an online (max, sum-exp) per lane, combined across lanes/waves -> per-row loss and
// logsumexp (fp32).  No [T, V] fp32 softmax is ever materialised.
// Backward: dlogits = (softmax - onehot) * dloss, recomputed from logits + lse and written
// IN PLACE over the logits (they are dead after the loss), so the lm_head backward GEMM
// reads it directly and the [T, V] buffer is allocated once.
#include "common.h"

namespace llmctl {
namespace {

__device__ __forceinline__ void combine(float& m, float& s, float m2, float s2) {
  const float M = fmaxf(m, m2);
  if (M == -INFINITY) return;
  s = s * __expf(m - M) + s2 * __expf(m2 - M);
  m = M;
}

__global__ __launch_bounds__(256) void ce_fwd_kernel(const unsigned short* __restrict__ logits,
                                                      const int64_t* __restrict__ labels, float* __restrict__ loss,
                                                      float* __restrict__ lse_out, int V, long ignore_index) {
  __shared__ float sm[4], ss[4];
  const long row = blockIdx.x;
  const unsigned short* lr = logits + row * (long)V;
  float m = -INFINITY, s = 0.f;
  const int V8 = V & ~7;
  for (int c = threadIdx.x * 8; c < V8; c += 2048) {
    float v[8];
    load8(lr + c, v);
    float mx = v[0];
#pragma unroll
    for (int j = 1; j < 8; ++j) mx = fmaxf(mx, v[j]);
    if (mx > m) {
      s = (m == -INFINITY) ? 0.f : s * __expf(m - mx);
      m = mx;
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) s += __expf(v[j] - m);
  }
  for (int c = V8 + threadIdx.x; c < V; c += 256) {
    const float x = bf2f(lr[c]);
    if (x > m) {
      s = (m == -INFINITY) ? 0.f : s * __expf(m - x);
      m = x;
    }
    s += __expf(x - m);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const float m2 = __shfl_xor(m, o), s2 = __shfl_xor(s, o);
    combine(m, s, m2, s2);
  }
  const int w = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) {
    sm[w] = m;
    ss[w] = s;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    float M = sm[0], S = ss[0];
    for (int i = 1; i < 4; ++i) combine(M, S, sm[i], ss[i]);
    const float lse = M + __logf(S);
    lse_out[row] = lse;
    const long lab = labels[row];
    loss[row] = (lab == ignore_index || lab < 0 || lab >= V) ? 0.f : lse - bf2f(lr[lab]);
  }
}

__global__ __launch_bounds__(256) void ce_bwd_kernel(const float* __restrict__ dloss,
                                                      const unsigned short* __restrict__ logits,
                                                      const float* __restrict__ lse,
                                                      const int64_t* __restrict__ labels,
                                                      unsigned short* __restrict__ out, int V, long ignore_index, int per_row, float factor) {
  const long row = blockIdx.x;
  const long lab = labels[row];
  const bool valid = !(lab == ignore_index || lab < 0 || lab >= V);
  const float d = valid ? (per_row ? dloss[row] : dloss[0] * factor) : 0.f;  // (one gradient of the mean: no pass that spreads it over the rows)
  const float L = lse[row];
  const unsigned short* lr = logits + row * (long)V;
  unsigned short* orow = out + row * (long)V;
  const int V8 = V & ~7;
  for (int c = threadIdx.x * 8; c < V8; c += 2048) {
    float v[8];
    load8(lr + c, v);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      v[j] = __expf(v[j] - L) * d;
      if (c + j == lab) v[j] -= d;
    }
    store8(orow + c, v);
  }
  for (int c = V8 + threadIdx.x; c < V; c += 256) {
    float g = __expf(bf2f(lr[c]) - L) * d;
    if (c == lab) g -= d;
    orow[c] = f2bf(g);
  }
}

// out = sum(loss) / denom, one workgroup, summed in 64 bits: up to 32768 rows (128 KB, 5 us) one launch where the library takes two, three with the memset that it
// clears its counters with from 16384 rows on.
__global__ __launch_bounds__(1024) void loss_mean_kernel(const float* __restrict__ loss, int T, double denom, float* __restrict__ out) {
  __shared__ double part[16];
  double s = 0.0;
  for (int i = threadIdx.x; i < T; i += 1024) s += (double)loss[i];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < 16; ++w) s += part[w];
    out[0] = (float)(s / denom);
  }
}

}  // namespace

std::tuple<at::Tensor, at::Tensor> cross_entropy_fwd(const at::Tensor& logits, const at::Tensor& labels,
                                                     int64_t ignore_index) {
  LLMCTL_CHECK(logits.is_cuda() && logits.dim() == 2 && logits.is_contiguous() &&
                   logits.scalar_type() == at::kBFloat16,
               "logits must be contiguous [T, V] bf16");
  LLMCTL_CHECK(labels.numel() == logits.size(0) && labels.scalar_type() == at::kLong && labels.is_contiguous(),
               "labels must be contiguous int64 [T]");
  const c10::DeviceGuard g(logits.device());
  const long T = logits.size(0);
  const int V = logits.size(1);
  auto loss = at::empty({T}, logits.options().dtype(at::kFloat));
  auto lse = at::empty({T}, logits.options().dtype(at::kFloat));
  if (T)
    hipLaunchKernelGGL(ce_fwd_kernel, dim3(T), dim3(256), 0, stream(), bf_ptr(logits), labels.data_ptr<int64_t>(),
                       loss.data_ptr<float>(), lse.data_ptr<float>(), V, (long)ignore_index);
  return {loss, lse};
}

at::Tensor cross_entropy_bwd(const at::Tensor& dloss, const at::Tensor& logits, const at::Tensor& lse,
                             const at::Tensor& labels, int64_t ignore_index, bool inplace) {
  LLMCTL_CHECK(dloss.scalar_type() == at::kFloat && dloss.is_contiguous() && dloss.numel() == logits.size(0),
               "dloss must be contiguous fp32 [T]");
  const c10::DeviceGuard g(logits.device());
  const long T = logits.size(0);
  const int V = logits.size(1);
  at::Tensor out = inplace ? logits : at::empty_like(logits);
  if (T)
    hipLaunchKernelGGL(ce_bwd_kernel, dim3(T), dim3(256), 0, stream(), dloss.data_ptr<float>(), bf_ptr(logits),
                       lse.data_ptr<float>(), labels.data_ptr<int64_t>(), bf_mut(out), V, (long)ignore_index, 1, 1.f);
  return out;
}

// sum(loss) / denom of loss fp32 [T], T at most 32768
at::Tensor loss_mean(const at::Tensor& loss, double denom) {
  LLMCTL_CHECK(loss.is_cuda() && loss.scalar_type() == at::kFloat && loss.is_contiguous() && loss.numel() <= 32768, "loss_mean: contiguous fp32, at most 32768 rows");
  const c10::DeviceGuard g(loss.device());
  at::Tensor out = at::empty({}, loss.options());
  hipLaunchKernelGGL(loss_mean_kernel, dim3(1), dim3(1024), 0, stream(), loss.data_ptr<float>(), (int)loss.numel(), denom, out.data_ptr<float>());
  return out;
}

// cross_entropy_bwd where every row's gradient is g / denom
at::Tensor cross_entropy_bwd_mean(const at::Tensor& g, double denom, const at::Tensor& logits, const at::Tensor& lse, const at::Tensor& labels, int64_t ignore_index,
                                  bool inplace) {
  LLMCTL_CHECK(g.is_cuda() && g.scalar_type() == at::kFloat && g.numel() == 1, "cross_entropy_bwd_mean: one fp32 gradient");
  LLMCTL_CHECK(logits.is_cuda() && logits.dim() == 2 && logits.is_contiguous() && logits.scalar_type() == at::kBFloat16 && lse.is_contiguous() &&
                   lse.numel() == logits.size(0) && labels.is_contiguous() && labels.scalar_type() == at::kLong && labels.numel() == logits.size(0),
               "cross_entropy_bwd_mean: what cross_entropy_fwd took and gave");
  const c10::DeviceGuard guard(logits.device());
  const long T = logits.size(0);
  at::Tensor out = inplace ? logits : at::empty_like(logits);
  if (T)
    hipLaunchKernelGGL(ce_bwd_kernel, dim3(T), dim3(256), 0, stream(), g.data_ptr<float>(), bf_ptr(logits), lse.data_ptr<float>(), labels.data_ptr<int64_t>(),
                       bf_mut(out), (int)logits.size(1), (long)ignore_index, 0, 1.f / (float)denom);
  return out;
}

TORCH_LIBRARY_IMPL(llmctl, CUDA, m) {
  m.impl("cross_entropy_fwd", &cross_entropy_fwd);
  m.impl("cross_entropy_bwd", &cross_entropy_bwd);
  m.impl("loss_mean", &loss_mean);
  m.impl("cross_entropy_bwd_mean", &cross_entropy_bwd_mean);
}

}  // namespace llmctl
