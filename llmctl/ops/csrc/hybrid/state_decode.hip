// One token per sequence through a head's memory and all that hangs on it, in one launch each:
//   gla_decode    S = diag(a) S + k v^T with a = sigmoid(W_a2 z_a + b)^(1/tau), o = S^T q, then the head norm and its silu gate
//   mlstm_decode  the gates (two rows of an fp32 weight a head), S, n and m of mlstm.hip, o, then the head norm and its sigmoid gate
//
// A decode step has one token for a head's 32 KB of memory: the bound is that read and write (16 sequences of 16 heads of 64 x 128: 16.8 MB, 3.2 us) and, as
// separate launches, the launches: the decay's product, the scan (64 lanes a workgroup, a column each) and the head norm, or the gates' product, the gates, the scan
// and the norm.  Here a workgroup owns a head: 16 groups of lanes share its rows, a lane has four neighbouring columns of every 16th row, all of them asked for before
// anything else, and the sums over the rows meet in LDS once.  The arithmetic is that of the scans, in fp32.  In a graph, us, before / here, 16 heads of 64 x 128, width 2048:
//   sequences       1            16           64           256
//   gla        13.0 /  5.1  14.2 / 6.2   21.2 / 12.5  64.3 / 47.7
//   mlstm      16.7 /  6.1  18.8 / 7.2   31.1 / 17.0  79.4 / 59.4   (the gates' product apart: 7.9, 9.9, 26.1, 61.2)
// Keys of 256: 16 sequences 40 / 20 and 32 / 16, 64 of them 77 / 71 and 86 / 55, but 256 341 / 364 and 313 / 299: beyond 128 channels for at most 64 sequences (state_decode_ok).
#include "hybrid_common.h"

namespace llmctl_hybrid {

namespace {
__device__ __forceinline__ float log_sigmoid(float x) { return fminf(x, 0.f) - log1pf(expf(-fabsf(x))); }

struct StateArgs {
  const bf16_t* q;
  const bf16_t* k;
  const bf16_t* v;
  int64_t q_st, q_sh, k_st, k_sh, v_st, v_sh;  // token and head strides (elements)
  float* S;  // [slots, H, dk, dv]
  const int* slots;
  const int* start;
  const float* hn_w;   // [H * dv]
  const bf16_t* hn_g;  // [T, H * dv]
  int64_t hn_st;
  float hn_eps, qscale;
  bf16_t* y;  // [T, H * dv]
  int H, dk, dv;
};
struct GlaGates {
  const bf16_t* a;  // [T, rank]
  int64_t a_st;
  const bf16_t* w;  // [H * dk, rank]
  const float* b;   // [H * dk]
  float inv_tau;
  int rank;
};
struct MlstmGates {
  const float* raw;  // [T, 2 H], or null: h w^T
  const bf16_t* h;   // [T, W]
  int64_t h_st;
  const float* w;  // [2 H, W]
  const float* b_i;
  const float* b_f;
  float* n;  // [slots, H, dk]
  float* m;  // [slots, H]
  float cap;
  int W;
};

// 16 groups of CL lanes; a lane has the columns 4 cl .. of rows rg + 16 i
template <int NR, int CL>
struct HeadRows {
  static constexpr int NT = 16 * CL, NWV = NT / 64;
  int n, h, cl, rg, col;
  bool cok;
  float* Sb;
  float S[NR][4], kr[NR], qr[NR], v[4];

  __device__ __forceinline__ void load(const StateArgs& a, bool fresh, int64_t slot) {
    const int tid = threadIdx.x;
    n = blockIdx.x, h = blockIdx.y, cl = tid % CL, rg = tid / CL, col = 4 * cl;
    cok = col < a.dv;  // (quads divide dv)
    const int colc = cok ? col : 0;
    Sb = a.S + (slot * a.H + h) * (int64_t)a.dk * a.dv + colc;
    const bf16_t *kp = a.k + n * a.k_st + h * a.k_sh, *qp = a.q + n * a.q_st + h * a.q_sh, *vp = a.v + n * a.v_st + h * a.v_sh + colc;
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const int d = rg + 16 * i;
      const bool ok = d < a.dk;
#pragma unroll
      for (int c = 0; c < 4; ++c) S[i][c] = 0.f;
      if (ok && !fresh) Vec16<float>::load(Sb + (int64_t)d * a.dv, S[i]);
      kr[i] = ok ? ldf(kp + d) : 0.f;
      qr[i] = ok ? ldf(qp + d) * a.qscale : 0.f;
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) v[c] = ldf(vp + c);
  }
  // row i becomes f S + k u and is stored; o += its part of S^T q
  __device__ __forceinline__ void step(const StateArgs& a, int i, float f, const float (&u)[4], float (&o)[4]) {
    const int d = rg + 16 * i;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      S[i][c] = f * S[i][c] + kr[i] * u[c];
      o[c] += S[i][c] * qr[i];
    }
    if (cok && d < a.dk) Vec16<float>::store(Sb + (int64_t)d * a.dv, S[i]);
  }
  // the sums over the groups of N values to the lanes of the first one
  template <int N>
  __device__ __forceinline__ void sum(float (&o)[N], float (&red)[NWV][CL][N]) {
#pragma unroll
    for (int c = 0; c < N; ++c)
#pragma unroll
      for (int x = CL; x < 64; x <<= 1) o[c] += __shfl_xor(o[c], x, 64);
    if ((threadIdx.x & 63) < CL) {
#pragma unroll
      for (int c = 0; c < N; ++c) red[threadIdx.x >> 6][cl][c] = o[c];
    }
    __syncthreads();
    if (threadIdx.x >= CL) return;
#pragma unroll
    for (int c = 0; c < N; ++c) {
      o[c] = red[0][cl][c];
#pragma unroll
      for (int w = 1; w < NWV; ++w) o[c] += red[w][cl][c];
    }
  }
  // y = o / rms(o) * w * sigmoid(g), times g where SILU: the first group's lanes
  template <bool SILU>
  __device__ __forceinline__ void finish(const StateArgs& a, const float (&o)[4], const float (&g)[4], const float (&w)[4]) {
    float q = cok ? (o[0] * o[0] + o[1] * o[1]) + (o[2] * o[2] + o[3] * o[3]) : 0.f;
#pragma unroll
    for (int x = CL / 2; x > 0; x >>= 1) q += __shfl_xor(q, x, 64);
    if (!cok) return;
    const float rstd = 1.0f / sqrtf(q / (float)a.dv + a.hn_eps);
    bf16_t* yp = a.y + ((int64_t)n * a.H + h) * a.dv + col;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const float gate = 1.0f / (1.0f + expf(-g[c]));
      stf(yp + c, o[c] * (rstd * w[c] * (SILU ? g[c] * gate : gate)));
    }
  }
  __device__ __forceinline__ void load_gate(const StateArgs& a, float (&g)[4], float (&w)[4]) const {
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const bool on = threadIdx.x < CL && cok;
      g[c] = on ? ldf(a.hn_g + n * a.hn_st + h * a.dv + col + c) : 0.f;
      w[c] = on ? a.hn_w[h * a.dv + col + c] : 0.f;
    }
  }
};

template <int NR, int CL>
__global__ __launch_bounds__(16 * CL) void gla_decode_kernel(StateArgs a, GlaGates z) {
  using R = HeadRows<NR, CL>;
  __shared__ float decay[16 * NR];
  __shared__ float red[R::NWV][CL][4];
  R r;
  r.load(a, a.start[blockIdx.x] == 0, a.slots[blockIdx.x]);
  float g[4], w[4];
  r.load_gate(a, g, w);
  // eight lanes a key channel
  for (int e = threadIdx.x; e < 16 * NR * 8; e += R::NT) {
    const int d = e >> 3, row = r.h * a.dk + min(d, a.dk - 1);
    float s = 0.f;
    for (int c = e & 7; c < z.rank; c += 8) s += ldf(z.a + r.n * z.a_st + c) * ldf(z.w + (int64_t)row * z.rank + c);
#pragma unroll
    for (int x = 4; x > 0; x >>= 1) s += __shfl_xor(s, x, 64);
    if ((e & 7) == 0) decay[d] = expf(log_sigmoid(s + z.b[row]) * z.inv_tau);
  }
  __syncthreads();
  float o[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < NR; ++i) r.step(a, i, decay[r.rg + 16 * i], r.v, o);
  r.sum(o, red);
  if (threadIdx.x < CL) r.template finish<true>(a, o, g, w);
}

template <int NR, int CL>
__global__ __launch_bounds__(16 * CL) void mlstm_decode_kernel(StateArgs a, MlstmGates z) {
  using R = HeadRows<NR, CL>;
  __shared__ float red[R::NWV][CL][5];
  __shared__ float part[R::NWV][2];
  R r;
  const bool fresh = a.start[blockIdx.x] == 0;
  const int64_t slot = a.slots[blockIdx.x];
  r.load(a, fresh, slot);
  float g[4], w[4];
  r.load_gate(a, g, w);
  float* nb = z.n + (slot * a.H + r.h) * (int64_t)a.dk;
  float nr[NR];  // the normaliser's rows: the first lane of every group reads and rewrites them
#pragma unroll
  for (int i = 0; i < NR; ++i) nr[i] = r.cl == 0 && !fresh && r.rg + 16 * i < a.dk ? nb[r.rg + 16 * i] : 0.f;
  const float m = fresh ? 0.f : z.m[slot * a.H + r.h];
  float zi, zf;
  if (z.raw != nullptr) {
    zi = z.raw[(int64_t)r.n * 2 * a.H + r.h];
    zf = z.raw[(int64_t)r.n * 2 * a.H + a.H + r.h];
  } else {
    zi = 0.f, zf = 0.f;
    for (int c = threadIdx.x * 4; c < z.W; c += R::NT * 4) {
      const float4 x = ld4(z.h + r.n * z.h_st + c), wi = ld4(z.w + (int64_t)r.h * z.W + c), wf = ld4(z.w + (int64_t)(a.H + r.h) * z.W + c);
      zi = fmaf(x.x, wi.x, fmaf(x.y, wi.y, fmaf(x.z, wi.z, fmaf(x.w, wi.w, zi))));
      zf = fmaf(x.x, wf.x, fmaf(x.y, wf.y, fmaf(x.z, wf.z, fmaf(x.w, wf.w, zf))));
    }
    zi = wave_sum(zi), zf = wave_sum(zf);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6][0] = zi, part[threadIdx.x >> 6][1] = zf;
    __syncthreads();
    zi = part[0][0], zf = part[0][1];
#pragma unroll
    for (int x = 1; x < R::NWV; ++x) zi += part[x][0], zf += part[x][1];
  }
  const float ig = z.cap * tanhf((zi + z.b_i[r.h]) / z.cap), fg = log_sigmoid(z.cap * tanhf((zf + z.b_f[r.h]) / z.cap));
  const float mn = fmaxf(fg + m, ig), da = __expf(fg + m - mn), db = __expf(ig - mn);
  float o[5] = {0.f, 0.f, 0.f, 0.f, 0.f}, o4[4] = {0.f, 0.f, 0.f, 0.f}, u[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) u[c] = db * r.v[c];
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    r.step(a, i, da, u, o4);
    const int d = r.rg + 16 * i;
    if (r.cl == 0 && d < a.dk) {
      nr[i] = da * nr[i] + db * r.kr[i];
      o[4] += nr[i] * r.qr[i];
      nb[d] = nr[i];
    }
  }
#pragma unroll
  for (int c = 0; c < 4; ++c) o[c] = o4[c];
  r.sum(o, red);
  if (threadIdx.x >= CL) return;
  if (threadIdx.x == 0) z.m[slot * a.H + r.h] = mn;  // (every wave has used the old one: the sum's barrier)
  const float den = fmaxf(fabsf(__shfl(o[4], 0, 64)), __expf(-mn)) + 1e-6f;
#pragma unroll
  for (int c = 0; c < 4; ++c) o4[c] = o[c] / den;
  r.template finish<false>(a, o4, g, w);
}

bool f32of(const at::Tensor& t, int64_t n) { return t.is_cuda() && t.is_contiguous() && t.scalar_type() == at::kFloat && t.numel() == n; }

StateArgs state_args(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, double qscale, const at::Tensor& S, const at::Tensor& slots,
                     const at::Tensor& start, const at::Tensor& hn_w, const at::Tensor& hn_g, double eps) {
  for (const at::Tensor* t : {&q, &k, &v})
    HYB_CHECK(t->is_cuda() && t->dim() == 3 && (t->size(2) == 1 || t->stride(2) == 1) && t->scalar_type() == at::kBFloat16, "q, k, v: bf16 [T, H, d] with unit last stride");
  const int64_t T = q.size(0), H = q.size(1), dk = q.size(2), dv = v.size(2);
  HYB_CHECK(k.sizes() == q.sizes() && v.size(0) == T && v.size(1) == H, "q, k, v: one number of rows and heads");
  HYB_CHECK(dk >= 1 && dk <= 256 && dv >= 4 && dv <= 128 && dv % 4 == 0 && H <= 65535, "key size 1 .. 256, value size up to 128 in quads");
  HYB_CHECK(S.is_cuda() && S.is_contiguous() && S.scalar_type() == at::kFloat && S.dim() == 4 && S.size(1) == H && S.size(2) == dk && S.size(3) == dv &&
                reinterpret_cast<uintptr_t>(S.data_ptr()) % 16 == 0,
            "state: contiguous fp32 [slots, H, dk, dv]");
  for (const at::Tensor* t : {&slots, &start}) HYB_CHECK(t->is_cuda() && t->is_contiguous() && t->scalar_type() == at::kInt && t->numel() == T, "slots, start: int32 [T]");
  HYB_CHECK(f32of(hn_w, H * dv), "norm weight: fp32 [H * dv]");
  check_rows(hn_g, "gate");
  HYB_CHECK(hn_g.size(0) == T && hn_g.size(1) == H * dv && hn_g.scalar_type() == at::kBFloat16, "gate: bf16 [T, H * dv]");
  auto bf = [](const at::Tensor& t) { return reinterpret_cast<const bf16_t*>(t.data_ptr()); };
  return {bf(q), bf(k), bf(v), q.stride(0), q.stride(1), k.stride(0), k.stride(1), v.stride(0), v.stride(1), S.data_ptr<float>(), slots.data_ptr<int>(),
          start.data_ptr<int>(), hn_w.data_ptr<float>(), bf(hn_g), hn_g.stride(0), (float)eps, (float)qscale, nullptr, (int)H, (int)dk, (int)dv};
}

template <typename F>
void by_rows(const StateArgs& a, F&& go) {
  auto lanes = [&](auto cl) {
    if (a.dk <= 16) go(std::integral_constant<int, 1>{}, cl);
    else if (a.dk <= 32) go(std::integral_constant<int, 2>{}, cl);
    else if (a.dk <= 64) go(std::integral_constant<int, 4>{}, cl);
    else if (a.dk <= 128) go(std::integral_constant<int, 8>{}, cl);
    else go(std::integral_constant<int, 16>{}, cl);
  };
  if (a.dv <= 64) lanes(std::integral_constant<int, 16>{});
  else lanes(std::integral_constant<int, 32>{});
}
}  // namespace

// a [T, rank], w [H * dk, rank] bf16, b fp32 [H * dk] -> y [T, H * dv]; S at slots in place
at::Tensor gla_decode(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, const at::Tensor& a, const at::Tensor& w, const at::Tensor& b, double tau,
                      double qscale, at::Tensor S, const at::Tensor& slots, const at::Tensor& start, const at::Tensor& hn_w, const at::Tensor& hn_g, double eps) {
  StateArgs s = state_args(q, k, v, qscale, S, slots, start, hn_w, hn_g, eps);
  const int64_t T = q.size(0), rows = (int64_t)s.H * s.dk, rank = w.dim() == 2 ? w.size(1) : 0;
  check_rows(a, "a");
  HYB_CHECK(a.size(0) == T && a.size(1) == rank && rank >= 1 && a.scalar_type() == at::kBFloat16, "a: bf16 [T, rank]");
  HYB_CHECK(w.is_cuda() && w.is_contiguous() && w.size(0) == rows && w.scalar_type() == at::kBFloat16 && f32of(b, rows) && tau > 0.0,
            "w: bf16 [H * dk, rank], b: fp32 [H * dk], tau > 0");
  c10::DeviceGuard guard(q.device());
  at::Tensor y = at::empty({T, (int64_t)s.H * s.dv}, q.options());
  if (T == 0) return y;
  s.y = reinterpret_cast<bf16_t*>(y.data_ptr());
  const GlaGates z{reinterpret_cast<const bf16_t*>(a.data_ptr()), a.stride(0), reinterpret_cast<const bf16_t*>(w.data_ptr()), b.data_ptr<float>(), (float)(1.0 / tau), (int)rank};
  by_rows(s, [&](auto nr, auto cl) {
    gla_decode_kernel<decltype(nr)::value, decltype(cl)::value><<<dim3((unsigned)T, (unsigned)s.H), 16 * decltype(cl)::value, 0, cur_stream()>>>(s, z);
  });
  return y;
}

// raw: fp32 [T, 2 H], or None: h [T, W] bf16 times w [2 H, W] fp32
at::Tensor mlstm_decode(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, const c10::optional<at::Tensor>& raw, const at::Tensor& h, const at::Tensor& w,
                        const at::Tensor& b_i, const at::Tensor& b_f, double cap, double qscale, at::Tensor S, at::Tensor n, at::Tensor m, const at::Tensor& slots,
                        const at::Tensor& start, const at::Tensor& hn_w, const at::Tensor& hn_g, double eps) {
  StateArgs s = state_args(q, k, v, qscale, S, slots, start, hn_w, hn_g, eps);
  const int64_t T = q.size(0), H = s.H, W = h.dim() == 2 ? h.size(1) : 0;
  HYB_CHECK(f32of(n, S.size(0) * H * s.dk) && f32of(m, S.size(0) * H) && f32of(b_i, H) && f32of(b_f, H), "n: fp32 [slots, H, dk], m: [slots, H], b_i, b_f: [H]");
  if (raw.has_value()) {
    HYB_CHECK(f32of(*raw, T * 2 * H), "gates: fp32 [T, 2 H]");
  } else {
    check_rows(h, "h");
    HYB_CHECK(h.size(0) == T && h.scalar_type() == at::kBFloat16 && f32of(w, 2 * H * W) && quads_ok(reinterpret_cast<const bf16_t*>(h.data_ptr()), h.stride(0), W) &&
                  quads_ok(w.data_ptr<float>(), W, W),
              "h: bf16 [T, W], w: fp32 [2 H, W], rows in quads");
  }
  c10::DeviceGuard guard(q.device());
  at::Tensor y = at::empty({T, H * s.dv}, q.options());
  if (T == 0) return y;
  s.y = reinterpret_cast<bf16_t*>(y.data_ptr());
  const MlstmGates z{raw.has_value() ? raw->data_ptr<float>() : nullptr, reinterpret_cast<const bf16_t*>(h.data_ptr()), h.stride(0), w.data_ptr<float>(),
                     b_i.data_ptr<float>(), b_f.data_ptr<float>(), n.data_ptr<float>(), m.data_ptr<float>(), (float)cap, (int)W};
  by_rows(s, [&](auto nr, auto cl) {
    mlstm_decode_kernel<decltype(nr)::value, decltype(cl)::value><<<dim3((unsigned)T, (unsigned)H), 16 * decltype(cl)::value, 0, cur_stream()>>>(s, z);
  });
  return y;
}

}  // namespace llmctl_hybrid
