// A decode step's LayerNorm and the projection behind it in one launch: y = act(LN(x (+ res)) W^T + bias) for up to 16 rows, and for the
// QKV projection its split: q rows out, K and V rows to the paged cache.
//
// Bound: at these sizes a launch (3.5 us and the gap before it) and one round trip to HBM for the weights.  The norm of a few short rows
// costs less than its launch did, so every workgroup repeats it: its first weights are requested first, the rows are
// normalised while they arrive, and go through LDS as the product's bf16 operand (the same numbers as the separate kernels').  The
// first workgroup stores the new residual.  Split of the product as in stream_linear.h: 16 weight rows per workgroup, K over four waves.
// Measured in a graph, one MI355X, against LayerNorm + stream_linear: 1 row, K 768, N 3072 4.8 us (6.7), N 2304 with the split 4.7 (9.2); 8
// rows 6.3 (7.2).  A decode step of gpt2-125m: 1 row 466 -> 375 us, 4 rows 498 -> 412, 16 rows 551 -> 520.
#include "common.h"
#include "stream_linear.h"

namespace llmctl {
namespace {
using stream_linear::acc_t;
using stream_linear::frag_t;
using stream_linear::load_or_zero;

struct NLArgs {
  const unsigned short* x;    // [M, K]
  const unsigned short* res;  // [M, K] or null
  unsigned short* res_out;    // [M, K] (res given)
  const unsigned short* nw;
  const unsigned short* nb;
  float eps;
  const unsigned short* w;  // [N, K]
  long ldw;
  const unsigned short* bias;  // [N] or null
  unsigned short* y;           // [M, N]; with a cache: [M, q_cols]
  int M, N, K, act;
  // QKV: columns from q_cols on go to the cache rows of ``slots`` (-1: nowhere)
  void* kc;
  void* vc;
  const int64_t* slots;
  int q_cols, kv_cols, fp8;
};

constexpr int U = 8;

template <int NV, bool CACHE>  // NV: 512-column pieces of a row
__global__ __launch_bounds__(256) void norm_linear_kernel(NLArgs g) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  __shared__ acc_t red[4][64];
  unsigned short* const xs = reinterpret_cast<unsigned short*>(smem);  // [M][K + 8]
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r = lane & 15, kg = lane >> 4, K = g.K, ldx = K + 8;
  const int n0 = blockIdx.x * 16;
  const unsigned short* wp = g.w + (long)min(n0 + r, g.N - 1) * g.ldw + 8 * kg;
  const int steps = (K + 31) / 32, per = (steps + 3) / 4, s0 = wave * per, s1 = min(s0 + per, steps);
  uint4 wv[U];
  auto load_weights = [&](int s) {
#pragma unroll
    for (int u = 0; u < U; ++u) wv[u] = load_or_zero(wp + (s + u) * 32, s + u < s1 && (s + u) * 32 + 8 * kg < K);
  };
  load_weights(s0);
  __builtin_amdgcn_sched_barrier(0);
  // a wave's rows (wave, wave + 4, ..) in batches of RB, their loads in flight together
  constexpr int RB = NV <= 2 ? 4 : 2;
  bf16x8 wn[NV], bn[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int col = min(i * 512 + lane * 8, K - 8);
    wn[i] = *reinterpret_cast<const bf16x8*>(g.nw + col);
    bn[i] = *reinterpret_cast<const bf16x8*>(g.nb + col);
  }
  const float inv_k = 1.f / (float)K;
  const unsigned short* second = g.res != nullptr ? g.res : g.x;
  for (int row0 = wave; row0 < g.M; row0 += 4 * RB) {
    bf16x8 xv[RB][NV], qv[RB][NV];
#pragma unroll
    for (int k = 0; k < RB; ++k)
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        const long at = (long)min(row0 + 4 * k, g.M - 1) * K + min(i * 512 + lane * 8, K - 8);
        xv[k][i] = *reinterpret_cast<const bf16x8*>(g.x + at);
        qv[k][i] = *reinterpret_cast<const bf16x8*>(second + at);
      }
#pragma unroll
    for (int k = 0; k < RB; ++k) {
      const int row = row0 + 4 * k;
      if (row >= g.M) break;
      float v[NV][8];
      float s = 0.f;
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        const int col = i * 512 + lane * 8;
#pragma unroll
        for (int j = 0; j < 8; ++j) v[i][j] = col < K ? bf2f(xv[k][i][j]) : 0.f;
        if (g.res != nullptr && col < K) {
          bf16x8 o;
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            o[j] = f2bf(v[i][j] + bf2f(qv[k][i][j]));
            v[i][j] = bf2f(o[j]);  // normalise the rounded residual
          }
          if (blockIdx.x == 0) *reinterpret_cast<bf16x8*>(g.res_out + (long)row * K + col) = o;
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) s += v[i][j];
      }
      const float mean = wave_sum(s) * inv_k;
      float ss = 0.f;
#pragma unroll
      for (int i = 0; i < NV; ++i)
        if (i * 512 + lane * 8 < K)
#pragma unroll
          for (int j = 0; j < 8; ++j) ss += (v[i][j] - mean) * (v[i][j] - mean);
      const float rs = rsqrtf(wave_sum(ss) * inv_k + g.eps);
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        const int col = i * 512 + lane * 8;
        if (col < K) {
          float o[8];
#pragma unroll
          for (int j = 0; j < 8; ++j) o[j] = (v[i][j] - mean) * rs * bf2f(wn[i][j]) + bf2f(bn[i][j]);
          store8(xs + row * ldx + col, o);
        }
      }
    }
  }
  __syncthreads();
  const unsigned short* xr = xs + min(r, g.M - 1) * ldx + 8 * kg;
  acc_t acc = {0.f, 0.f, 0.f, 0.f};
  for (int s = s0; s < s1; s += U) {
    if (s > s0) load_weights(s);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint4 xv = load_or_zero(xr + (s + u) * 32, s + u < s1 && (s + u) * 32 + 8 * kg < K);
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(frag_t, wv[u]), __builtin_bit_cast(frag_t, xv), acc, 0, 0, 0);
    }
  }
  red[wave][lane] = acc;
  __syncthreads();
  if (wave != 0) return;
  const int row = r, c = n0 + 4 * kg;  // four neighbouring outputs of one row
  if (row >= g.M || c >= g.N) return;
  acc_t sum = red[0][lane];
#pragma unroll
  for (int k = 1; k < 4; ++k) sum += red[k][lane];
  unsigned short h[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float b = g.bias != nullptr ? bf2f(g.bias[c + j]) : 0.f;  // N is a multiple of 4
    h[j] = f2bf(stream_linear::activate(g.act, sum[j] + b));
  }
  const uint2 packed = make_uint2(h[0] | ((unsigned)h[1] << 16), h[2] | ((unsigned)h[3] << 16));
  if (!CACHE) {
    *reinterpret_cast<uint2*>(g.y + (long)row * g.N + c) = packed;
    return;
  }
  if (c < g.q_cols) {
    *reinterpret_cast<uint2*>(g.y + (long)row * g.q_cols + c) = packed;
    return;
  }
  const long slot = g.slots[row];
  if (slot < 0) return;
  const bool is_v = c >= g.q_cols + g.kv_cols;
  const long at = slot * g.kv_cols + c - g.q_cols - (is_v ? g.kv_cols : 0);
  void* cache = is_v ? g.vc : g.kc;
  if (g.fp8) {
    int q8 = __builtin_amdgcn_cvt_pk_fp8_f32(sat_fp8(bf2f(h[0])), sat_fp8(bf2f(h[1])), 0, false);
    q8 = __builtin_amdgcn_cvt_pk_fp8_f32(sat_fp8(bf2f(h[2])), sat_fp8(bf2f(h[3])), q8, true);
    *reinterpret_cast<int*>(static_cast<unsigned char*>(cache) + at) = q8;
  } else {
    *reinterpret_cast<uint2*>(static_cast<unsigned short*>(cache) + at) = packed;
  }
}

bool vec_ok(const at::Tensor& t, int64_t n) {
  return t.is_cuda() && t.is_contiguous() && t.scalar_type() == at::kBFloat16 && t.numel() == n;
}
bool aligned16(const at::Tensor& t) { return (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0; }

NLArgs nl_args(const at::Tensor& x, const c10::optional<at::Tensor>& res, const at::Tensor& nw, const at::Tensor& nb, double eps,
               const at::Tensor& w, const c10::optional<at::Tensor>& bias, at::Tensor& res_out) {
  LLMCTL_CHECK(x.is_cuda() && x.dim() == 2 && x.is_contiguous() && x.scalar_type() == at::kBFloat16 && aligned16(x), "norm_linear: x bf16 [M, K]");
  const int64_t M = x.size(0), K = x.size(1);
  LLMCTL_CHECK(M >= 1 && M <= 16 && K >= 8 && K % 8 == 0 && K <= 2048 && M * K <= 24576, "norm_linear: up to 16 rows, K a multiple of 8 up to 2048");
  LLMCTL_CHECK(w.is_cuda() && w.dim() == 2 && w.size(1) == K && w.stride(1) == 1 && w.scalar_type() == at::kBFloat16 && w.stride(0) % 8 == 0 &&
                   aligned16(w) && w.size(0) % 4 == 0 && w.size(0) >= 4,
               "norm_linear: w bf16 [N, K], 16-byte aligned rows, N a multiple of 4");
  LLMCTL_CHECK(vec_ok(nw, K) && vec_ok(nb, K) && aligned16(nw) && aligned16(nb), "norm_linear: norm weight and bias bf16 [K]");
  const bool has_b = bias.has_value() && bias->defined(), has_res = res.has_value() && res->defined();
  if (has_b) LLMCTL_CHECK(vec_ok(*bias, w.size(0)), "norm_linear: bias bf16 [N]");
  if (has_res) LLMCTL_CHECK(res->sizes() == x.sizes() && vec_ok(*res, M * K) && aligned16(*res), "norm_linear: residual like x");
  res_out = has_res ? at::empty_like(x) : at::empty({0}, x.options());
  NLArgs a = {};
  a.x = bf_ptr(x), a.res = has_res ? bf_ptr(*res) : nullptr, a.res_out = has_res ? bf_mut(res_out) : nullptr;
  a.nw = bf_ptr(nw), a.nb = bf_ptr(nb), a.eps = (float)eps;
  a.w = bf_ptr(w), a.ldw = w.stride(0), a.bias = has_b ? bf_ptr(*bias) : nullptr;
  a.M = (int)M, a.N = (int)w.size(0), a.K = (int)K;
  return a;
}

template <bool CACHE>
void nl_launch(const NLArgs& a) {
  const dim3 grid((unsigned)((a.N + 15) / 16));
  const size_t lds = (size_t)a.M * (a.K + 8) * 2;
  auto s = stream();
  if (a.K <= 512) hipLaunchKernelGGL((norm_linear_kernel<1, CACHE>), grid, dim3(256), lds, s, a);
  else if (a.K <= 1024) hipLaunchKernelGGL((norm_linear_kernel<2, CACHE>), grid, dim3(256), lds, s, a);
  else hipLaunchKernelGGL((norm_linear_kernel<4, CACHE>), grid, dim3(256), lds, s, a);
}
}  // namespace

// (act(LN(x + res) w^T + bias), x + res); without res the second is empty
std::tuple<at::Tensor, at::Tensor> norm_linear(const at::Tensor& x, const c10::optional<at::Tensor>& res, const at::Tensor& nw, const at::Tensor& nb,
                                               double eps, const at::Tensor& w, const c10::optional<at::Tensor>& bias, int64_t act) {
  at::Tensor res_out;
  const c10::DeviceGuard guard(x.device());
  NLArgs a = nl_args(x, res, nw, nb, eps, w, bias, res_out);
  LLMCTL_CHECK(act >= 0 && act <= 3, "norm_linear: activation");
  at::Tensor y = at::empty({x.size(0), w.size(0)}, x.options());
  a.y = bf_mut(y), a.act = (int)act;
  nl_launch<false>(a);
  return {y, res_out};
}

// (q [M, nq, D], x + res); the K and V rows go to the caches [slots, nkv, D] (bf16 or fp8)
std::tuple<at::Tensor, at::Tensor> norm_qkv_cache(const at::Tensor& x, const c10::optional<at::Tensor>& res, const at::Tensor& nw,
                                                  const at::Tensor& nb, double eps, const at::Tensor& w, const c10::optional<at::Tensor>& bias,
                                                  int64_t nq, int64_t nkv, at::Tensor k_cache, at::Tensor v_cache, const at::Tensor& slots) {
  at::Tensor res_out;
  const c10::DeviceGuard guard(x.device());
  NLArgs a = nl_args(x, res, nw, nb, eps, w, bias, res_out);
  LLMCTL_CHECK(nq >= 1 && nkv >= 1 && w.size(0) % (nq + 2 * nkv) == 0, "norm_qkv_cache: heads");
  const int64_t D = w.size(0) / (nq + 2 * nkv);
  LLMCTL_CHECK(D % 8 == 0, "norm_qkv_cache: head size a multiple of 8");
  for (const at::Tensor* c : {&k_cache, &v_cache})
    LLMCTL_CHECK(c->is_cuda() && c->is_contiguous() && kv_cache_ok(*c) && c->dim() == 4 && c->size(2) == nkv && c->size(3) == D,
                 "norm_qkv_cache: cache [blocks, block_size, nkv, D], bf16 or fp8");
  LLMCTL_CHECK(k_cache.scalar_type() == v_cache.scalar_type() && slots.is_cuda() && slots.is_contiguous() && slots.scalar_type() == at::kLong &&
                   slots.numel() == x.size(0),
               "norm_qkv_cache: slots int64 [M]");
  at::Tensor q = at::empty({x.size(0), nq, D}, x.options());
  a.y = bf_mut(q), a.kc = k_cache.data_ptr(), a.vc = v_cache.data_ptr(), a.slots = slots.data_ptr<int64_t>();
  a.q_cols = (int)(nq * D), a.kv_cols = (int)(nkv * D), a.fp8 = kv_fp8(k_cache);
  nl_launch<true>(a);
  return {q, res_out};
}

TORCH_LIBRARY_IMPL(llmctl, CUDA, m) {
  m.impl("norm_linear", &norm_linear);
  m.impl("norm_qkv_cache", &norm_qkv_cache);
}

}  // namespace llmctl
