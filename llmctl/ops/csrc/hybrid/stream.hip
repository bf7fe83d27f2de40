// The fp32 residual stream of parallel layers and the small row-wise passes around the mixers:
// LayerNorm (two-pass mean / variance), residual update fused with the next LayerNorm, RMS norm of a
// column range, sigmoid gating, SwiGLU, per-head unit-RMS with weight and gate.
#include "expert_rows.h"
#include "router_rows.h"

namespace llmctl_hybrid {

constexpr int NT = 256;
constexpr int NW = NT / 64;

// x [T, W] fp32 (updated in place when a != nullptr: x += a + b), h = LayerNorm(x) * w + bias.
template <typename T>
__global__ __launch_bounds__(NT) void add_layernorm_kernel(float* __restrict__ x, const T* __restrict__ a, int64_t a_stride,
                                                           const float* __restrict__ b, const float* __restrict__ w,
                                                           const float* __restrict__ bias, T* __restrict__ h, int W,
                                                           float eps) {
  __shared__ float red[NW];
  const int64_t r = blockIdx.x;
  float* xr = x + r * W;
  float s = 0.f;
  for (int c = threadIdx.x; c < W; c += NT) {
    float v = xr[c];
    if (a != nullptr) {
      v += ldf(a + r * a_stride + c);
      if (b != nullptr) v += b[r * W + c];
      xr[c] = v;
    }
    s += v;
  }
  if (h == nullptr) return;
  const float mean = block_sum<NW>(s, red) / (float)W;
  float q = 0.f;
  for (int c = threadIdx.x; c < W; c += NT) {
    const float d = xr[c] - mean;
    q += d * d;
  }
  const float rstd = 1.0f / sqrtf(block_sum<NW>(q, red) / (float)W + eps);
  for (int c = threadIdx.x; c < W; c += NT) stf(h + r * W + c, (xr[c] - mean) * rstd * w[c] + bias[c]);
}

// The same for rows of up to 4 * NT * VQ values in quads: all of a row's loads in flight at once, the row in registers from then on.  A decode
// step's rows are a chain of latencies (16 rows of 2048: 8.9 us as above, 8 dependent loads deep, 4.4 so; 2048 rows 14.5 and 13.3).
// ``Y``: b is the weighted sum of the routed experts' rows of that type (expert_rows.h) instead of a tensor; as a pass of its own that sum
// cost a launch and its own traffic (16 rows of 2048, two experts each: 4.7 + 4.7 us, together 5.0; 2048 rows 8.6 + 14.3, together 11.7).
// ``ROUTE``: the rows go through a router too (router_rows.h).
template <typename T, int VQ, typename Y = void, bool ROUTE = false>
__global__ __launch_bounds__(NT) void add_layernorm_quads_kernel(float* __restrict__ x, const T* __restrict__ a, int64_t a_stride,
                                                                 const float* __restrict__ b, const float* __restrict__ w,
                                                                 const float* __restrict__ bias, T* __restrict__ h, int W, float eps,
                                                                 ExpertRows m, RouteOut route) {
  __shared__ float red[2][NW];
  const int64_t r = blockIdx.x;
  float4 v[VQ], av[VQ], bv[VQ], wv[VQ], cv[VQ];
#pragma unroll
  for (int i = 0; i < VQ; ++i) {
    const int c = min((int)(threadIdx.x + i * NT) * 4, W - 4);
    v[i] = ld4(x + r * W + c);
    av[i] = a != nullptr ? ld4(a + r * a_stride + c) : make_float4(0.f, 0.f, 0.f, 0.f);
    if constexpr (std::is_void_v<Y>) bv[i] = b != nullptr ? ld4(b + r * W + c) : make_float4(0.f, 0.f, 0.f, 0.f);
    if (h != nullptr) wv[i] = ld4(w + c), cv[i] = ld4(bias + c);
  }
  RouterRows<NW, VQ> rw;
  if constexpr (ROUTE) rw.load(route.w, route.c.E, W, 0);
  if constexpr (!std::is_void_v<Y>) expert_sum_quads<Y, NT, VQ>(m, r, W, bv);
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < VQ; ++i) {
    const int c = (int)(threadIdx.x + i * NT) * 4;
    v[i].x = v[i].x + av[i].x + bv[i].x, v[i].y = v[i].y + av[i].y + bv[i].y;
    v[i].z = v[i].z + av[i].z + bv[i].z, v[i].w = v[i].w + av[i].w + bv[i].w;
    if (c < W) {
      if (a != nullptr) st4(x + r * W + c, v[i]);
      s += (v[i].x + v[i].y) + (v[i].z + v[i].w);
    }
  }
  if (h == nullptr) return;
  const float mean = block_sum<NW, true>(s, red[0]) / (float)W;
  float q = 0.f;
#pragma unroll
  for (int i = 0; i < VQ; ++i) {
    v[i].x -= mean, v[i].y -= mean, v[i].z -= mean, v[i].w -= mean;
    if ((int)(threadIdx.x + i * NT) * 4 < W) q += (v[i].x * v[i].x + v[i].y * v[i].y) + (v[i].z * v[i].z + v[i].w * v[i].w);
  }
  const float rstd = 1.0f / sqrtf(block_sum<NW, true>(q, red[1]) / (float)W + eps);
#pragma unroll
  for (int i = 0; i < VQ; ++i) {
    const int c = (int)(threadIdx.x + i * NT) * 4;
    v[i] = make_float4(v[i].x * rstd * wv[i].x + cv[i].x, v[i].y * rstd * wv[i].y + cv[i].y, v[i].z * rstd * wv[i].z + cv[i].z,
                       v[i].w * rstd * wv[i].w + cv[i].w);
    if (c < W) st4(h + r * W + c, v[i]);
  }
  if constexpr (ROUTE) route.row<NW, VQ>(v, rw, r, W);
}

// The first of a step: x = table[id] * scale, h = LayerNorm(x) * w + bias; the product in fp32, as a cast and a multiplication give it.  One
// launch for the gather, the cast, the scale and the norm (16 rows of 2048: four launches, 27.1 us -> 6.5; 2048 rows 27.4 -> 13.0).
template <typename T, int VQ, bool ROUTE>
__global__ __launch_bounds__(NT) void embed_layernorm_quads_kernel(const int64_t* __restrict__ ids, const T* __restrict__ table, int64_t rows,
                                                                   float scale, const float* __restrict__ w, const float* __restrict__ bias,
                                                                   float* __restrict__ x, T* __restrict__ h, int W, float eps, RouteOut route) {
  __shared__ float red[2][NW];
  const int64_t r = blockIdx.x, id = ids[r];
  CUDA_KERNEL_ASSERT(id >= 0 && id < rows);
  float4 v[VQ], wv[VQ], cv[VQ];
#pragma unroll
  for (int i = 0; i < VQ; ++i) {
    const int c = min((int)(threadIdx.x + i * NT) * 4, W - 4);
    v[i] = ld4(table + id * W + c);
    wv[i] = ld4(w + c);
    cv[i] = ld4(bias + c);
  }
  RouterRows<NW, VQ> rw;
  if constexpr (ROUTE) rw.load(route.w, route.c.E, W, 0);
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < VQ; ++i) {
    const int c = (int)(threadIdx.x + i * NT) * 4;
    v[i].x *= scale, v[i].y *= scale, v[i].z *= scale, v[i].w *= scale;
    if (c < W) {
      st4(x + r * W + c, v[i]);
      s += (v[i].x + v[i].y) + (v[i].z + v[i].w);
    }
  }
  const float mean = block_sum<NW, true>(s, red[0]) / (float)W;
  float q = 0.f;
#pragma unroll
  for (int i = 0; i < VQ; ++i) {
    v[i].x -= mean, v[i].y -= mean, v[i].z -= mean, v[i].w -= mean;
    if ((int)(threadIdx.x + i * NT) * 4 < W) q += (v[i].x * v[i].x + v[i].y * v[i].y) + (v[i].z * v[i].z + v[i].w * v[i].w);
  }
  const float rstd = 1.0f / sqrtf(block_sum<NW, true>(q, red[1]) / (float)W + eps);
#pragma unroll
  for (int i = 0; i < VQ; ++i) {
    const int c = (int)(threadIdx.x + i * NT) * 4;
    v[i] = make_float4(v[i].x * rstd * wv[i].x + cv[i].x, v[i].y * rstd * wv[i].y + cv[i].y, v[i].z * rstd * wv[i].z + cv[i].z,
                       v[i].w * rstd * wv[i].w + cv[i].w);
    if (c < W) st4(h + r * W + c, v[i]);
  }
  if constexpr (ROUTE) route.row<NW, VQ>(v, rw, r, W);
}

// Rows that the quads do not take: x alone, its LayerNorm by add_layernorm_kernel.
template <typename T>
__global__ __launch_bounds__(NT) void embed_scale_kernel(const int64_t* __restrict__ ids, const T* __restrict__ table, int64_t rows, float scale,
                                                         float* __restrict__ x, int W) {
  const int64_t r = blockIdx.x, id = ids[r];
  CUDA_KERNEL_ASSERT(id >= 0 && id < rows);
  for (int c = threadIdx.x; c < W; c += NT) x[r * W + c] = ldf(table + id * W + c) * scale;
}

// x [T, W] fp32 (updated in place when a != nullptr: x += a + b), then up to two RMS norms of the same
// x (one statistic): h_k = x / sqrt(mean(x^2) + eps) * (plus + w_k); ``plus`` = 1 for weights stored
// around zero.  A parallel layer's residual update and the two norms its branches read, in one pass.
template <typename T>
__global__ __launch_bounds__(NT) void add_rmsnorm2_kernel(float* __restrict__ x, const T* __restrict__ a, int64_t a_stride,
                                                          const T* __restrict__ b, int64_t b_stride, const float* __restrict__ w1,
                                                          const float* __restrict__ w2, T* __restrict__ h1, T* __restrict__ h2, int W,
                                                          float eps, float plus) {
  __shared__ float red[NW];
  constexpr int KEEP = 16;  // a thread's first KEEP values stay in registers (rows up to KEEP * NT wide are read once)
  const int64_t r = blockIdx.x;
  float* xr = x + r * W;
  float keep[KEEP];
  float q = 0.f;
#pragma unroll
  for (int i = 0; i < KEEP; ++i) {
    const int c = threadIdx.x + i * NT;
    float v = 0.f;
    if (c < W) {
      v = xr[c];
      if (a != nullptr) {
        float d = ldf(a + r * a_stride + c);
        if (b != nullptr) d += ldf(b + r * b_stride + c);
        v += d;
        xr[c] = v;
      }
    }
    keep[i] = v;
    q += v * v;
  }
  for (int c = threadIdx.x + KEEP * NT; c < W; c += NT) {
    float v = xr[c];
    if (a != nullptr) {
      float d = ldf(a + r * a_stride + c);
      if (b != nullptr) d += ldf(b + r * b_stride + c);
      v += d;
      xr[c] = v;
    }
    q += v * v;
  }
  if (h1 == nullptr) return;
  const float rstd = 1.0f / sqrtf(block_sum<NW>(q, red) / (float)W + eps);
#pragma unroll
  for (int i = 0; i < KEEP; ++i) {
    const int c = threadIdx.x + i * NT;
    if (c < W) {
      const float v = keep[i] * rstd;
      stf(h1 + r * W + c, v * (plus + w1[c]));
      if (h2 != nullptr) stf(h2 + r * W + c, v * (plus + w2[c]));
    }
  }
  for (int c = threadIdx.x + KEEP * NT; c < W; c += NT) {
    const float v = xr[c] * rstd;
    stf(h1 + r * W + c, v * (plus + w1[c]));
    if (h2 != nullptr) stf(h2 + r * W + c, v * (plus + w2[c]));
  }
}

// gu [rows, 2F] = [gate | up] -> g' = min(gate, limit), u' = clamp(up, -limit, limit),
// y = g' * sigmoid(alpha * g') * (u' + 1)
template <typename T>
__global__ void clamped_glu_kernel(const T* __restrict__ gu, T* __restrict__ y, int64_t rows, int F, float limit, float alpha) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= rows * F) return;
  const int64_t r = i / F;
  const int c = (int)(i - r * F);
  const float g = fminf(ldf(gu + r * 2 * F + c), limit);
  const float u = fminf(fmaxf(ldf(gu + r * 2 * F + F + c), -limit), limit);
  stf(y + i, g / (1.0f + expf(-alpha * g)) * (u + 1.0f));
}

// the same with 16-byte accesses (F a multiple of 8, aligned rows): one thread per 8 bf16 / 4 fp32 outputs
template <typename T>
__global__ void clamped_glu_vec_kernel(const T* __restrict__ gu, T* __restrict__ y, int64_t rows, int F, float limit, float alpha) {
  constexpr int N = Vec16<T>::N;
  const int per = F / N;
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= rows * per) return;
  const int64_t r = i / per;
  const int c = (int)(i - r * per) * N;
  float g[N], u[N], o[N];
  Vec16<T>::load(gu + r * 2 * F + c, g);
  Vec16<T>::load(gu + r * 2 * F + F + c, u);
#pragma unroll
  for (int k = 0; k < N; ++k) {
    const float gk = fminf(g[k], limit), uk = fminf(fmaxf(u[k], -limit), limit);
    o[k] = gk / (1.0f + expf(-alpha * gk)) * (uk + 1.0f);
  }
  Vec16<T>::store(y + r * F + c, o);
}

template <typename T>
__global__ __launch_bounds__(NT) void rmsnorm_cols_kernel(const T* __restrict__ x, int64_t x_stride, const float* __restrict__ w,
                                                          T* __restrict__ y, int n, float eps) {
  __shared__ float red[NW];
  const int64_t r = blockIdx.x;
  float q = 0.f;
  for (int c = threadIdx.x; c < n; c += NT) {
    const float v = ldf(x + r * x_stride + c);
    q += v * v;
  }
  const float rstd = 1.0f / sqrtf(block_sum<NW>(q, red) / (float)n + eps);
  for (int c = threadIdx.x; c < n; c += NT) stf(y + r * n + c, ldf(x + r * x_stride + c) * rstd * w[c]);
}

template <typename TO, typename TG>
__global__ void gate_mul_kernel(const TO* __restrict__ o, const TG* __restrict__ g, int64_t g_stride, TG* __restrict__ y,
                                int64_t rows, int N, int per) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= rows * N) return;
  const int64_t r = i / N;
  const int c = (int)(i - r * N);
  const float gv = ldf(g + r * g_stride + c / per);  // one gate per ``per`` neighbouring columns
  stf(y + i, ldf(o + i) * (1.0f / (1.0f + expf(-gv))));
}

// The same 16 bytes at a time: rows whose pieces share one gate (per a multiple of N) or have one each (per 1).  2048 x 2048 with a gate each 11.3 us element by
// element, 7.8 so; 2911 rows with a gate per head 16.5 and 9.3.
template <typename T>
__global__ __launch_bounds__(256) void gate_mul_vec_kernel(const T* __restrict__ o, const T* __restrict__ g, int64_t g_stride, T* __restrict__ y, int64_t rows,
                                                           int W, int per) {
  constexpr int N = Vec16<T>::N;
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * N;
  if (i >= rows * W) return;
  const int64_t r = i / W;
  const int c = (int)(i - r * W);
  float v[N], gv[N];
  Vec16<T>::load(o + i, v);
  if (per == 1) {
    Vec16<T>::load(g + r * g_stride + c, gv);
  } else {
    const float one = ldf(g + r * g_stride + c / per);
#pragma unroll
    for (int j = 0; j < N; ++j) gv[j] = one;
  }
#pragma unroll
  for (int j = 0; j < N; ++j) v[j] *= 1.0f / (1.0f + expf(-gv[j]));
  Vec16<T>::store(y + i, v);
}

// o [T, H, dv] fp32 -> y [T, H*dv]: o / rms(o over dv) * w (if given) * sigmoid(g) (silu: * g sigmoid(g)); one wave per (token, head).
template <typename T>
__global__ __launch_bounds__(NT) void headnorm_gate_kernel(const float* __restrict__ o, const float* __restrict__ w,
                                                           const T* __restrict__ g, int64_t g_stride, T* __restrict__ y,
                                                           int64_t pairs, int H, int dv, float eps, int silu) {
  const int64_t p = (int64_t)blockIdx.x * NW + (threadIdx.x >> 6);
  if (p >= pairs) return;
  const int lane = threadIdx.x & 63;
  const int64_t t = p / H;
  const int hd = (int)(p - t * H);
  const float* op = o + p * dv;
  float q = 0.f;
  for (int c = lane; c < dv; c += 64) q += op[c] * op[c];
  const float rstd = 1.0f / sqrtf(wave_sum(q) / (float)dv + eps);
  for (int c = lane; c < dv; c += 64) {
    const float gv = ldf(g + t * g_stride + hd * dv + c);
    const float gate = 1.0f / (1.0f + expf(-gv));
    stf(y + p * dv + c, op[c] * rstd * (w != nullptr ? w[hd * dv + c] : 1.0f) * (silu ? gv * gate : gate));
  }
}

// The same for heads of at most 256 values in quads: ``lg`` lanes (a power of two) own a head, four neighbouring entries each.
template <typename T>
__global__ __launch_bounds__(NT) void headnorm_gate_quads_kernel(const float* __restrict__ o, const float* __restrict__ w,
                                                                 const T* __restrict__ g, int64_t g_stride, T* __restrict__ y,
                                                                 int64_t pairs, int H, int dv, float eps, int silu, int lg) {
  const int64_t p = ((int64_t)blockIdx.x * NT + threadIdx.x) / lg;
  if (p >= pairs) return;  // (a head's lanes leave together)
  const int c = (threadIdx.x % lg) * 4;
  const bool ok = c < dv;
  const int64_t t = p / H;
  const int hd = (int)(p - t * H);
  float v[4] = {0.f, 0.f, 0.f, 0.f}, gv[4] = {0.f, 0.f, 0.f, 0.f}, wv[4] = {1.f, 1.f, 1.f, 1.f};
  if (ok) {
    Vec16<float>::load(o + p * dv + c, v);
    const T* gp = g + t * g_stride + hd * dv + c;
    if constexpr (sizeof(T) == 4) {
      Vec16<float>::load(reinterpret_cast<const float*>(gp), gv);
    } else {
      const uint2 x = *reinterpret_cast<const uint2*>(gp);
      gv[0] = __uint_as_float(x.x << 16), gv[1] = __uint_as_float(x.x & 0xffff0000u);
      gv[2] = __uint_as_float(x.y << 16), gv[3] = __uint_as_float(x.y & 0xffff0000u);
    }
    if (w != nullptr) Vec16<float>::load(w + hd * dv + c, wv);
  }
  float q = (v[0] * v[0] + v[1] * v[1]) + (v[2] * v[2] + v[3] * v[3]);
  for (int s = lg >> 1; s > 0; s >>= 1) q += __shfl_xor(q, s, 64);
  if (!ok) return;
  const float rstd = 1.0f / sqrtf(q / (float)dv + eps);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float gate = 1.0f / (1.0f + expf(-gv[i]));
    v[i] *= rstd * wv[i] * (silu ? gv[i] * gate : gate);
  }
  if constexpr (sizeof(T) == 4) {
    Vec16<float>::store(reinterpret_cast<float*>(y) + p * dv + c, v);
  } else {
    unsigned x[2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
      x[i] = (unsigned)__bfloat16_as_ushort(__float2bfloat16(v[2 * i])) | ((unsigned)__bfloat16_as_ushort(__float2bfloat16(v[2 * i + 1])) << 16);
    *reinterpret_cast<uint2*>(y + p * dv + c) = make_uint2(x[0], x[1]);
  }
}

// ------------------------------------------------------------------------------------------ host
static at::Tensor out_like(const at::Tensor& ref, at::IntArrayRef shape, bool bf16) {
  return at::empty(shape, ref.options().dtype(bf16 ? at::kBFloat16 : at::kFloat));
}

// x += a (+ b) where a is given, h = LN(x) where h is: rows in quads where widths and addresses allow
template <typename T>
static void launch_add_layernorm(float* x, const T* a, int64_t a_st, const float* b, const float* w, const float* bias, T* h, int64_t rows, int W,
                                 double eps) {
  auto go = [&](auto kern) { kern<<<dim3((unsigned)rows), NT, 0, cur_stream()>>>(x, a, a_st, b, w, bias, h, W, (float)eps, ExpertRows{}, RouteOut{}); };
  const bool quads = W <= 16 * NT && quads_ok(x, W, W) && (a == nullptr || quads_ok(a, a_st, W)) && (b == nullptr || quads_ok(b, W, W)) &&
                     (h == nullptr || (quads_ok(w, W, W) && quads_ok(bias, W, W)));
  if (quads && W <= 4 * NT) go(add_layernorm_quads_kernel<T, 1>);
  else if (quads && W <= 8 * NT) go(add_layernorm_quads_kernel<T, 2>);
  else if (quads) go(add_layernorm_quads_kernel<T, 4>);
  else add_layernorm_kernel<T><<<dim3((unsigned)rows), NT, 0, cur_stream()>>>(x, a, a_st, b, w, bias, h, W, (float)eps);
}

at::Tensor layernorm_f32(const at::Tensor& x, const at::Tensor& w, const at::Tensor& b, double eps, bool out_bf16) {
  HYB_CHECK(x.is_cuda() && x.dim() == 2 && x.is_contiguous() && x.scalar_type() == at::kFloat, "x: contiguous fp32 [T, W]");
  const int W = (int)x.size(1);
  HYB_CHECK(w.scalar_type() == at::kFloat && b.scalar_type() == at::kFloat && w.numel() == W && b.numel() == W && w.is_contiguous() && b.is_contiguous(), "norm weight / bias: fp32 [W]");
  c10::DeviceGuard guard(x.device());
  at::Tensor h = out_like(x, x.sizes(), out_bf16);
  if (x.size(0) == 0) return h;
  dispatch_act(h, [&](auto* tag) {
    using T = std::remove_pointer_t<decltype(tag)>;
    launch_add_layernorm<T>(x.data_ptr<float>(), nullptr, 0, nullptr, w.data_ptr<float>(), b.data_ptr<float>(), (T*)h.data_ptr(), x.size(0), W, eps);
  });
  return h;
}

// x and h; with a router (bf16 rows) the chosen experts of every row of h and their weights too.
std::vector<at::Tensor> embed_layernorm_f32(const at::Tensor& ids, const at::Tensor& table, double scale, const at::Tensor& w, const at::Tensor& b,
                                            double eps, const c10::optional<at::Tensor>& router, const c10::optional<at::Tensor>& rbias, int64_t top,
                                            int64_t groups, int64_t keep, bool softmax, bool renorm) {
  HYB_CHECK(table.is_cuda() && table.dim() == 2 && table.is_contiguous(), "table: contiguous [vocab, W]");
  HYB_CHECK(ids.is_cuda() && ids.is_contiguous() && ids.scalar_type() == at::kLong && ids.dim() == 1, "ids: int64 [T]");
  const int64_t T = ids.numel(), W = table.size(1);
  HYB_CHECK(w.scalar_type() == at::kFloat && b.scalar_type() == at::kFloat && w.numel() == W && b.numel() == W && w.is_contiguous() && b.is_contiguous(), "norm weight / bias: fp32 [W]");
  HYB_CHECK(!router.has_value() || table.scalar_type() == at::kBFloat16, "a router takes bf16 rows");
  c10::DeviceGuard guard(table.device());
  at::Tensor x = at::empty({T, W}, table.options().dtype(at::kFloat)), h = at::empty({T, W}, table.options());
  const float *wp = w.data_ptr<float>(), *bp = b.data_ptr<float>();
  float* xp = x.data_ptr<float>();
  const bool quads = W <= 16 * NT && W % 4 == 0 && quads_ok(wp, W, W) && quads_ok(bp, W, W) &&
                     reinterpret_cast<uintptr_t>(table.data_ptr()) % (4 * table.element_size()) == 0;
  std::vector<at::Tensor> out = {x, h};
  RouteOut route{};
  if (router.has_value() && quads) route = route_out(*router, W, rbias, top, groups, keep, softmax, renorm, T, out);
  if (T > 0)
    dispatch_act(table, [&](auto* tag) {
      using Tt = std::remove_pointer_t<decltype(tag)>;
      const Tt* tp = (const Tt*)table.data_ptr();
      auto go = [&](auto kern) {
        kern<<<dim3((unsigned)T), NT, 0, cur_stream()>>>(ids.data_ptr<int64_t>(), tp, table.size(0), (float)scale, wp, bp, xp, (Tt*)h.data_ptr(), (int)W,
                                                         (float)eps, route);
      };
      auto pick = [&](auto on) {
        constexpr bool R = decltype(on)::value;
        if (W <= 4 * NT) go(embed_layernorm_quads_kernel<Tt, 1, R>);
        else if (W <= 8 * NT) go(embed_layernorm_quads_kernel<Tt, 2, R>);
        else go(embed_layernorm_quads_kernel<Tt, 4, R>);
      };
      if (quads) {
        if constexpr (std::is_same_v<Tt, bf16_t>) {
          if (router.has_value()) return pick(std::true_type{});
        }
        pick(std::false_type{});
      } else {
        embed_scale_kernel<Tt><<<dim3((unsigned)T), NT, 0, cur_stream()>>>(ids.data_ptr<int64_t>(), tp, table.size(0), (float)scale, xp, (int)W);
        launch_add_layernorm<Tt>(xp, nullptr, 0, nullptr, wp, bp, (Tt*)h.data_ptr(), T, (int)W, eps);
      }
    });
  if (router.has_value() && !quads) add_routed(out, h, *router, rbias, top, groups, keep, softmax, renorm);
  return out;
}

static void check_add(const at::Tensor& x, const at::Tensor& a, const c10::optional<at::Tensor>& b) {
  HYB_CHECK(x.is_cuda() && x.dim() == 2 && x.is_contiguous() && x.scalar_type() == at::kFloat, "x: contiguous fp32 [T, W]");
  check_rows(a, "a");
  HYB_CHECK(a.size(0) == x.size(0) && a.size(1) == x.size(1), "a must have x's shape");
  if (b.has_value()) HYB_CHECK(b->is_cuda() && b->is_contiguous() && b->scalar_type() == at::kFloat && b->sizes() == x.sizes(), "b: contiguous fp32 of x's shape");
}

void residual_add_(at::Tensor x, const at::Tensor& a, const c10::optional<at::Tensor>& b) {
  check_add(x, a, b);
  if (x.size(0) == 0) return;
  c10::DeviceGuard guard(x.device());
  dispatch_act(a, [&](auto* tag) {
    using T = std::remove_pointer_t<decltype(tag)>;
    launch_add_layernorm<T>(x.data_ptr<float>(), (const T*)a.data_ptr(), a.stride(0), b.has_value() ? b->data_ptr<float>() : nullptr, nullptr, nullptr,
                            nullptr, x.size(0), (int)x.size(1), 0.0);
  });
}

at::Tensor add_layernorm_f32_(at::Tensor x, const at::Tensor& a, const c10::optional<at::Tensor>& b, const at::Tensor& w,
                              const at::Tensor& bias, double eps, bool out_bf16) {
  check_add(x, a, b);
  const int W = (int)x.size(1);
  HYB_CHECK(w.scalar_type() == at::kFloat && bias.scalar_type() == at::kFloat && w.numel() == W && bias.numel() == W && w.is_contiguous() && bias.is_contiguous(), "norm weight / bias: fp32 [W]");
  HYB_CHECK((a.scalar_type() == at::kBFloat16) == out_bf16, "the output has a's dtype");
  c10::DeviceGuard guard(x.device());
  at::Tensor h = out_like(x, x.sizes(), out_bf16);
  if (x.size(0) == 0) return h;
  dispatch_act(a, [&](auto* tag) {
    using T = std::remove_pointer_t<decltype(tag)>;
    launch_add_layernorm<T>(x.data_ptr<float>(), (const T*)a.data_ptr(), a.stride(0), b.has_value() ? b->data_ptr<float>() : nullptr,
                            w.data_ptr<float>(), bias.data_ptr<float>(), (T*)h.data_ptr(), x.size(0), W, eps);
  });
  return h;
}

at::Tensor moe_sum(const at::Tensor& y, const at::Tensor& idx, const at::Tensor& wgt, const at::Tensor& x, const c10::optional<at::Tensor>& shared,
                   const c10::optional<at::Tensor>& gate, int64_t experts);

// add_layernorm_f32_ with b = the weighted sum of the routed experts' rows y (moe_sum); without w: the sum alone, no norm.  With a router the chosen
// experts of every row of the result and their weights too.
std::vector<at::Tensor> add_experts_layernorm_f32_(at::Tensor x, const at::Tensor& a, const c10::optional<at::Tensor>& w, const c10::optional<at::Tensor>& bias,
                                                   double eps, const at::Tensor& y, const at::Tensor& idx, const at::Tensor& wgt, const at::Tensor& xin,
                                                   const c10::optional<at::Tensor>& shared, const c10::optional<at::Tensor>& gate, int64_t experts,
                                                   const c10::optional<at::Tensor>& router, const c10::optional<at::Tensor>& rbias, int64_t top,
                                                   int64_t groups, int64_t keep, bool softmax, bool renorm) {
  check_add(x, a, c10::nullopt);
  HYB_CHECK(a.scalar_type() == at::kBFloat16 && xin.sizes() == x.sizes() && w.has_value() == bias.has_value(), "routed experts: bf16 rows of x's shape; a norm has both vectors");
  HYB_CHECK(!router.has_value() || w.has_value(), "a router reads normed rows");
  const int64_t T = x.size(0);
  const int W = (int)x.size(1);
  if (w.has_value())
    HYB_CHECK(w->scalar_type() == at::kFloat && bias->scalar_type() == at::kFloat && w->numel() == W && bias->numel() == W && w->is_contiguous() && bias->is_contiguous(),
              "norm weight / bias: fp32 [W]");
  const ExpertRows m = expert_rows_of(y, idx, wgt, xin, shared, gate, experts);
  c10::DeviceGuard guard(x.device());
  at::Tensor h = w.has_value() ? out_like(x, x.sizes(), true) : at::empty({0}, x.options());
  const float *wp = w.has_value() ? w->data_ptr<float>() : nullptr, *bp = w.has_value() ? bias->data_ptr<float>() : nullptr;
  bf16_t* hp = w.has_value() ? (bf16_t*)h.data_ptr() : nullptr;
  const bf16_t* ap = (const bf16_t*)a.data_ptr();
  float* xp = x.data_ptr<float>();
  const bool quads = W <= 16 * NT && quads_ok(xp, W, W) && quads_ok(ap, a.stride(0), W) && (wp == nullptr || (quads_ok(wp, W, W) && quads_ok(bp, W, W)));
  std::vector<at::Tensor> out = {h};
  RouteOut route{};
  if (router.has_value() && quads) route = route_out(*router, W, rbias, top, groups, keep, softmax, renorm, T, out);
  auto go = [&](auto kern) { kern<<<dim3((unsigned)T), NT, 0, cur_stream()>>>(xp, ap, a.stride(0), nullptr, wp, bp, hp, W, (float)eps, m, route); };
  auto pick = [&](auto* tag, auto on) {
    using Y = std::remove_pointer_t<decltype(tag)>;
    constexpr bool R = decltype(on)::value;
    if (W <= 4 * NT) go(add_layernorm_quads_kernel<bf16_t, 1, Y, R>);
    else if (W <= 8 * NT) go(add_layernorm_quads_kernel<bf16_t, 2, Y, R>);
    else go(add_layernorm_quads_kernel<bf16_t, 4, Y, R>);
  };
  if (quads && T > 0) {
    const bool f32 = y.scalar_type() == at::kFloat;
    if (router.has_value()) f32 ? pick((float*)nullptr, std::true_type{}) : pick((bf16_t*)nullptr, std::true_type{});
    else f32 ? pick((float*)nullptr, std::false_type{}) : pick((bf16_t*)nullptr, std::false_type{});
  } else if (T > 0) {  // rows that the quads do not take
    const at::Tensor b = moe_sum(y, idx, wgt, xin, shared, gate, experts);
    launch_add_layernorm<bf16_t>(xp, ap, a.stride(0), b.data_ptr<float>(), wp, bp, hp, T, W, eps);
  }
  if (router.has_value() && !quads) add_routed(out, h, *router, rbias, top, groups, keep, softmax, renorm);
  return out;
}

at::Tensor rmsnorm_cols(const at::Tensor& x, const at::Tensor& w, double eps, int64_t n, bool out_bf16) {
  check_rows(x, "x");
  HYB_CHECK(n >= 1 && n <= x.size(1) && w.numel() == n && w.scalar_type() == at::kFloat && w.is_contiguous(), "w: fp32 [n], n <= columns");
  HYB_CHECK((x.scalar_type() == at::kBFloat16) == out_bf16, "the output has x's dtype");
  c10::DeviceGuard guard(x.device());
  at::Tensor y = out_like(x, {x.size(0), n}, out_bf16);
  if (x.size(0) == 0) return y;
  dispatch_act(x, [&](auto* tag) {
    using T = std::remove_pointer_t<decltype(tag)>;
    rmsnorm_cols_kernel<T><<<dim3((unsigned)x.size(0)), NT, 0, cur_stream()>>>((const T*)x.data_ptr(), x.stride(0), w.data_ptr<float>(),
                                                                            (T*)y.data_ptr(), (int)n, (float)eps);
  });
  return y;
}

at::Tensor sigmoid_gate_mul(const at::Tensor& o, const at::Tensor& g) {
  check_rows(g, "g");
  HYB_CHECK(o.is_cuda() && o.is_contiguous() && o.dim() == 2 && o.size(0) == g.size(0) && g.size(1) >= 1 && o.size(1) % g.size(1) == 0,
            "o: contiguous [T, C]; g [T, C] or [T, H] with H dividing C");
  HYB_CHECK(o.scalar_type() == g.scalar_type(), "o and g share a dtype");
  c10::DeviceGuard guard(g.device());
  at::Tensor y = at::empty(o.sizes(), g.options());
  const int64_t n = o.numel();
  if (n == 0) return y;
  dispatch_act(g, [&](auto* tag) {
    using T = std::remove_pointer_t<decltype(tag)>;
    constexpr int N = Vec16<T>::N;
    const T *op = (const T*)o.data_ptr(), *gp = (const T*)g.data_ptr();
    const int W = (int)o.size(1), per = (int)(o.size(1) / g.size(1));
    auto at16 = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
    // (up to 2^17 elements a thread each covers the latency better: 16 rows of 4096 1.94 us, in sixteen-byte pieces 2.14)
    if (n > 1 << 17 && W % N == 0 && at16(op) && at16(y.data_ptr()) && (per % N == 0 || (per == 1 && at16(gp) && g.stride(0) % N == 0)))
      gate_mul_vec_kernel<T><<<dim3((unsigned)((n / N + 255) / 256)), 256, 0, cur_stream()>>>(op, gp, g.stride(0), (T*)y.data_ptr(), o.size(0), W, per);
    else
      gate_mul_kernel<T, T><<<dim3((unsigned)((n + 255) / 256)), 256, 0, cur_stream()>>>(op, gp, g.stride(0), (T*)y.data_ptr(), o.size(0), W, per);
  });
  return y;
}

std::tuple<at::Tensor, at::Tensor> add_rmsnorm2_f32_(at::Tensor x, const c10::optional<at::Tensor>& a, const c10::optional<at::Tensor>& b,
                                                     const at::Tensor& w1, const c10::optional<at::Tensor>& w2, double eps, bool one_plus,
                                                     bool out_bf16) {
  HYB_CHECK(x.is_cuda() && x.dim() == 2 && x.is_contiguous() && x.scalar_type() == at::kFloat, "x: contiguous fp32 [T, W]");
  const int W = (int)x.size(1);
  auto okw = [&](const at::Tensor& w) { return w.is_cuda() && w.scalar_type() == at::kFloat && w.numel() == W && w.is_contiguous(); };
  HYB_CHECK(okw(w1) && (!w2.has_value() || okw(*w2)), "norm weights: fp32 [W]");
  const at::ScalarType act = out_bf16 ? at::kBFloat16 : at::kFloat;
  if (a.has_value()) {
    check_rows(*a, "a");
    HYB_CHECK(a->sizes() == x.sizes() && a->scalar_type() == act, "a: x's shape, the output dtype");
    if (b.has_value()) {
      check_rows(*b, "b");
      HYB_CHECK(b->sizes() == x.sizes() && b->scalar_type() == act, "b: x's shape, the output dtype");
    }
  } else {
    HYB_CHECK(!b.has_value(), "b without a");
  }
  c10::DeviceGuard guard(x.device());
  at::Tensor h1 = out_like(x, x.sizes(), out_bf16);
  at::Tensor h2 = w2.has_value() ? out_like(x, x.sizes(), out_bf16) : at::Tensor();
  if (x.size(0) == 0) return {h1, w2.has_value() ? h2 : h1};
  dispatch_act(h1, [&](auto* tag) {
    using T = std::remove_pointer_t<decltype(tag)>;
    add_rmsnorm2_kernel<T><<<dim3((unsigned)x.size(0)), NT, 0, cur_stream()>>>(
        x.data_ptr<float>(), a.has_value() ? (const T*)a->data_ptr() : nullptr, a.has_value() ? a->stride(0) : 0,
        b.has_value() ? (const T*)b->data_ptr() : nullptr, b.has_value() ? b->stride(0) : 0, w1.data_ptr<float>(),
        w2.has_value() ? w2->data_ptr<float>() : nullptr, (T*)h1.data_ptr(), w2.has_value() ? (T*)h2.data_ptr() : nullptr, W, (float)eps,
        one_plus ? 1.0f : 0.0f);
  });
  return {h1, w2.has_value() ? h2 : h1};
}

void residual_add_act_(at::Tensor x, const at::Tensor& a, const c10::optional<at::Tensor>& b) {
  HYB_CHECK(x.is_cuda() && x.dim() == 2 && x.is_contiguous() && x.scalar_type() == at::kFloat, "x: contiguous fp32 [T, W]");
  check_rows(a, "a");
  HYB_CHECK(a.sizes() == x.sizes(), "a must have x's shape");
  if (b.has_value()) {
    check_rows(*b, "b");
    HYB_CHECK(b->sizes() == x.sizes() && b->scalar_type() == a.scalar_type(), "b: x's shape, a's dtype");
  }
  if (x.size(0) == 0) return;
  c10::DeviceGuard guard(x.device());
  dispatch_act(a, [&](auto* tag) {
    using T = std::remove_pointer_t<decltype(tag)>;
    add_rmsnorm2_kernel<T><<<dim3((unsigned)x.size(0)), NT, 0, cur_stream()>>>(
        x.data_ptr<float>(), (const T*)a.data_ptr(), a.stride(0), b.has_value() ? (const T*)b->data_ptr() : nullptr,
        b.has_value() ? b->stride(0) : 0, nullptr, nullptr, (T*)nullptr, (T*)nullptr, (int)x.size(1), 0.f, 0.f);
  });
}

at::Tensor clamped_glu(const at::Tensor& gu, double limit, double alpha) {
  HYB_CHECK(gu.is_cuda() && gu.is_contiguous() && gu.dim() == 2 && gu.size(1) % 2 == 0, "gu: contiguous [T, 2F]");
  c10::DeviceGuard guard(gu.device());
  const int F = (int)(gu.size(1) / 2);
  at::Tensor y = at::empty({gu.size(0), F}, gu.options());
  const int64_t n = y.numel();
  if (n == 0) return y;
  dispatch_act(gu, [&](auto* tag) {
    using T = std::remove_pointer_t<decltype(tag)>;
    if (F % 8 == 0 && aligned16<T>(gu)) {
      const int64_t nv = n / Vec16<T>::N;
      clamped_glu_vec_kernel<T><<<dim3((unsigned)((nv + 255) / 256)), 256, 0, cur_stream()>>>((const T*)gu.data_ptr(), (T*)y.data_ptr(), gu.size(0),
                                                                                            F, (float)limit, (float)alpha);
    } else {
      clamped_glu_kernel<T><<<dim3((unsigned)((n + 255) / 256)), 256, 0, cur_stream()>>>((const T*)gu.data_ptr(), (T*)y.data_ptr(), gu.size(0), F,
                                                                                       (float)limit, (float)alpha);
    }
  });
  return y;
}

at::Tensor headnorm_gate(const at::Tensor& o, const c10::optional<at::Tensor>& w, const at::Tensor& g, double eps, bool out_bf16, bool silu) {
  HYB_CHECK(o.is_cuda() && o.is_contiguous() && o.dim() == 3 && o.scalar_type() == at::kFloat, "o: contiguous fp32 [T, H, dv]");
  check_rows(g, "g");
  const int64_t T = o.size(0);
  const int H = (int)o.size(1), dv = (int)o.size(2);
  HYB_CHECK(g.size(0) == T && g.size(1) == (int64_t)H * dv && (!w.has_value() || (w->numel() == (int64_t)H * dv && w->scalar_type() == at::kFloat && w->is_contiguous())), "g [T, H*dv], w fp32 [H*dv]");
  HYB_CHECK((g.scalar_type() == at::kBFloat16) == out_bf16, "the output has g's dtype");
  c10::DeviceGuard guard(o.device());
  at::Tensor y = out_like(o, {T, (int64_t)H * dv}, out_bf16);
  if (T == 0) return y;
  const int64_t pairs = T * H;
  dispatch_act(g, [&](auto* tag) {
    using Tt = std::remove_pointer_t<decltype(tag)>;
    const bool quads = dv % 4 == 0 && dv <= 256 && g.stride(0) % 4 == 0 && reinterpret_cast<uintptr_t>(g.data_ptr()) % (4 * sizeof(Tt)) == 0 &&
                       reinterpret_cast<uintptr_t>(o.data_ptr()) % 16 == 0 && (!w.has_value() || reinterpret_cast<uintptr_t>(w->data_ptr()) % 16 == 0);
    if (quads) {
      int lg = 1;
      while (lg * 4 < dv) lg *= 2;
      headnorm_gate_quads_kernel<Tt><<<dim3((unsigned)((pairs * lg + NT - 1) / NT)), NT, 0, cur_stream()>>>(
          o.data_ptr<float>(), w.has_value() ? w->data_ptr<float>() : nullptr, (const Tt*)g.data_ptr(), g.stride(0), (Tt*)y.data_ptr(), pairs, H, dv,
          (float)eps, silu ? 1 : 0, lg);
      return;
    }
    headnorm_gate_kernel<Tt><<<dim3((unsigned)((pairs + NW - 1) / NW)), NT, 0, cur_stream()>>>(
        o.data_ptr<float>(), w.has_value() ? w->data_ptr<float>() : nullptr, (const Tt*)g.data_ptr(), g.stride(0), (Tt*)y.data_ptr(), pairs, H, dv, (float)eps, silu ? 1 : 0);
  });
  return y;
}

}  // namespace llmctl_hybrid
