// Gated linear attention over long portions: the recurrence of gla.hip in chunks of 64 tokens, as fp32 matrix products (chunk_mfma.h).
//
// With a_t[d] = sigmoid(z + bias)^(1/tau) and G(s, t)[d] the product of a over the tokens s + 1 .. t,
//   o_t = qscale (sum_(s <= t) (sum_d q_t[d] k_s[d] G(s, t)[d]) v_s + S_0^T (q_t G(start, t))),
//   S_n = diag(G(start, n)) S_0 + sum_s (k_s G(s, n)) v_s^T.
// G is split per 16-token block, and every factor is a product of decays (never a quotient), so that none exceeds one or loses digits
// however fast the memory decays: a pair of different blocks has (product up to t in its block) * (products of the blocks between) *
// (product after s in its block), the outer two folded into Q and K.  Pairs within a block are summed channel by channel with the
// running product, as the token-by-token form does.
//   gla_chunk_local   every chunk from a zero memory: its contribution and total log decay
//   gla_chunk_out     every chunk's outputs from the memory at its first token (gla_chunk_combine, gla.hip)
//
// Bound: the chain of a chunk's phases (stage, decays, pairs within a block, folding, tiles, values).  16 heads of 64 x 128, us: a pass of
// the token-by-token scan over 2911 tokens in five portions took 97, twice; these take 34 and 58 (whole call 228 -> 132, 8192
// tokens 447 -> 270, keys of 128 at 2048 tokens 447 -> 158).
#include "chunk_mfma.h"

namespace llmctl_hybrid {
namespace {

struct GCArgs {
  const void* q;
  const void* k;
  const void* v;
  int64_t q_st, q_sh, k_st, k_sh, v_st, v_sh;  // token and head strides (elements)
  const float* z;                              // [T, H * dk] decay logits
  int64_t z_st;
  const float* zb;  // [H * dk]
  float inv_tau, qscale;
  const int* cu;    // [P + 1] chunk row offsets
  float* loc;       // [P, H, dk, dv]
  float* logd;      // [P, H, dk]
  const float* init;
  float* out;       // [T, H, dv]
  int H, dk, dv, vec;
};

// G [CH][ks] <- the decays; E [4][dkp] <- their products over every 16-token block (rows past n and channels past dk: one);
// L [4][dkp] (if given) <- the sums of their logarithms
__device__ __forceinline__ void block_decays(const GCArgs& a, float* G, float* E, float* L, int h, int t0, int n, int dkp, int ks) {
  const int nt = blockDim.x;
  const float* zp = a.z + (int64_t)t0 * a.z_st + (int64_t)h * a.dk;
  for (int e = threadIdx.x; e < 4 * dkp; e += nt) {
    const int b = e / dkp, d = e - b * dkp;
    float z[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int t = 16 * b + i;
      z[i] = (t < n && d < a.dk) ? zp[t * a.z_st + d] : 0.f;
    }
    const float bias = d < a.dk ? a.zb[h * a.dk + d] : 0.f;
    float s = 0.f, f = 1.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      float g = 1.f;
      if (16 * b + i < n && d < a.dk) {
        const float x = z[i] + bias, la = (fminf(x, 0.f) - log1pf(expf(-fabsf(x)))) * a.inv_tau;
        s += la;
        g = expf(la);
      }
      G[(16 * b + i) * ks + d] = g;
      f *= g;
    }
    E[e] = f;
    if (L != nullptr) L[e] = s;
  }
}

// LDS: K [CH][ks] | G [CH][ks] | E [4][dkp] | L [4][dkp].  A wave takes 16 value columns.
template <typename T, int NKK>
__global__ __launch_bounds__(512, 4) void gla_chunk_local_kernel(GCArgs a) {
  extern __shared__ __attribute__((aligned(16))) float smem[];
  const int p = blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6, nw = blockDim.x >> 6;
  const int t0 = a.cu[p], n = a.cu[p + 1] - t0;
  const int dk = a.dk, dv = a.dv, nkk = NKK > 0 ? NKK : (dk + 15) / 16, dkp = 16 * nkk, ks = dkp + 4;
  float* Ks = smem;
  float* G = Ks + CH * ks;
  float* E = G + CH * ks;
  float* L = E + 4 * dkp;
  const int col = (blockIdx.z * nw + wave) * 16 + (lane & 15), g4 = (lane >> 4) * 4;
  const bool cok = col < dv;
  const T* vp = reinterpret_cast<const T*>(a.v) + t0 * a.v_st + h * a.v_sh;
  f32x4 y[4];
#pragma unroll
  for (int m = 0; m < 4; ++m)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int t = 16 * m + g4 + r;
      y[m][r] = (cok && t < n) ? ldf(vp + t * a.v_st + col) : 0.f;
    }
  stage_rows(Ks, ks, reinterpret_cast<const T*>(a.k) + t0 * a.k_st + h * a.k_sh, a.k_st, n, dk, dkp, a.vec != 0);
  block_decays(a, G, E, L, h, t0, n, dkp, ks);
  __syncthreads();
  for (int e = tid; e < 4 * dkp; e += blockDim.x) {  // K <- K G(s, n)
    const int b = e / dkp, d = e - b * dkp;
    float f = 1.f;
    for (int bb = b + 1; bb < 4; ++bb) f *= E[bb * dkp + d];
#pragma unroll
    for (int i = 15; i >= 0; --i) {
      const int at = (16 * b + i) * ks + d;
      Ks[at] *= f;
      f *= G[at];
    }
  }
  if (blockIdx.z == 0)
    for (int d = tid; d < dk; d += blockDim.x)
      a.logd[((int64_t)p * a.H + h) * dk + d] = (L[d] + L[dkp + d]) + (L[2 * dkp + d] + L[3 * dkp + d]);
  __syncthreads();
  for (int dt = 0; dt < nkk; ++dt) {
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc = mfma4(Ks[(16 * m + g4 + j) * ks + 16 * dt + (lane & 15)], y[m][j], acc);
    float* o = a.loc + (((int64_t)p * a.H + h) * dk + 16 * dt + g4) * dv + col;
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (cok && 16 * dt + g4 + r < dk) o[(int64_t)r * dv] = acc[r];
  }
}

// LDS: K [CH][ks] | Q [CH][ks] | G [CH][ks] | scores [CH][AS] | E [4][dkp] | pre [4][dkp]
template <typename T, int NKK>
__global__ __launch_bounds__(512, 4) void gla_chunk_out_kernel(GCArgs a) {
  extern __shared__ __attribute__((aligned(16))) float smem[];
  const int p = blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6, nw = blockDim.x >> 6;
  const int t0 = a.cu[p], n = a.cu[p + 1] - t0;
  const int dk = a.dk, dv = a.dv, nkk = NKK > 0 ? NKK : (dk + 15) / 16, dkp = 16 * nkk, ks = dkp + 4;
  float* Ks = smem;
  float* Qs = Ks + CH * ks;
  float* G = Qs + CH * ks;
  float* P = G + CH * ks;
  float* E = P + CH * AS;
  float* pre = E + 4 * dkp;  // the product over the blocks before
  const int col = (blockIdx.z * nw + wave) * 16 + (lane & 15), g4 = (lane >> 4) * 4;
  const bool cok = col < dv;
  const T* vp = reinterpret_cast<const T*>(a.v) + t0 * a.v_st + h * a.v_sh;
  f32x4 y[4];
#pragma unroll
  for (int m = 0; m < 4; ++m)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int t = 16 * m + g4 + r;
      y[m][r] = (cok && t < n) ? ldf(vp + t * a.v_st + col) : 0.f;
    }
  const float* S0 = a.init + ((int64_t)p * a.H + h) * dk * dv + (cok ? col : dv - 1);
  auto load_state = [&](int kk) {
    f32x4 s;
#pragma unroll
    for (int j = 0; j < 4; ++j) s[j] = 16 * kk + g4 + j < dk ? S0[(int64_t)(16 * kk + g4 + j) * dv] : 0.f;
    return s;
  };
  f32x4 s0[NKK > 0 && NKK < 8 ? NKK : 1];  // (128 channels: no registers to spare for them ahead of the scores)
  if constexpr (NKK > 0 && NKK < 8) {
#pragma unroll
    for (int kk = 0; kk < NKK; ++kk) s0[kk] = load_state(kk);
  }
  stage_rows(Ks, ks, reinterpret_cast<const T*>(a.k) + t0 * a.k_st + h * a.k_sh, a.k_st, n, dk, dkp, a.vec != 0);
  stage_rows(Qs, ks, reinterpret_cast<const T*>(a.q) + t0 * a.q_st + h * a.q_sh, a.q_st, n, dk, dkp, a.vec != 0);
  block_decays(a, G, E, nullptr, h, t0, n, dkp, ks);
  __syncthreads();
  // pairs within a block: eight threads per t share the channels and go back from s = t with the running product
  for (int e = tid; e < CH * 8; e += blockDim.x) {
    const int t = e >> 3, b16 = t & ~15;
    constexpr int NQ = NKK > 0 ? (NKK + 1) / 2 : 4;  // quads of channels per thread: 4 (part + 8 i) ..
    f32x4 qf[NQ];
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
      const int d = 4 * ((e & 7) + 8 * i);
      qf[i] = d < dkp ? lds4(Qs + t * ks + d) : f32x4{0.f, 0.f, 0.f, 0.f};
    }
    for (int s = b16 + 15; s > t; --s)
      if ((e & 7) == 0) P[t * AS + s] = 0.f;
    for (int s = t; s >= b16; --s) {
      float w = 0.f;
#pragma unroll
      for (int i = 0; i < NQ; ++i) {
        const int d = min(4 * ((e & 7) + 8 * i), dkp - 4);
        const f32x4 k4 = lds4(Ks + s * ks + d), g4_ = lds4(G + s * ks + d);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          w += qf[i][j] * k4[j];
          qf[i][j] *= g4_[j];
        }
      }
      w += __shfl_xor(w, 1, 64);
      w += __shfl_xor(w, 2, 64);
      w += __shfl_xor(w, 4, 64);
      if ((e & 7) == 0) P[t * AS + s] = w;
    }
  }
  __syncthreads();
  // Q <- Q (product up to t in its block), K <- K (product after s in its block), and the products up to every block
  for (int e = tid; e < 4 * dkp; e += blockDim.x) {
    const int b = e / dkp, d = e - b * dkp;
    float g[16], f = 1.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int at = (16 * b + i) * ks + d;
      g[i] = G[at];
      f *= g[i];
      Qs[at] *= f;
    }
    f = 1.f;
#pragma unroll
    for (int i = 15; i >= 0; --i) {
      Ks[(16 * b + i) * ks + d] *= f;
      f *= g[i];
    }
    f = 1.f;
    for (int bb = 0; bb < b; ++bb) f *= E[bb * dkp + d];
    pre[e] = f;
  }
  __syncthreads();
  // pairs of different blocks: the six tiles below the diagonal
  for (int i = wave; i < 6; i += nw) {
    const int ti = i < 1 ? 1 : (i < 3 ? 2 : 3), tj = i - ti * (ti - 1) / 2;
    const float* xr = Qs + (16 * ti + (lane & 15)) * ks + g4;
    const float* yr = Ks + (16 * tj + (lane & 15)) * ks + g4;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int kk = 0; kk < nkk; ++kk) {
      f32x4 x = lds4(xr + 16 * kk);
      if (tj + 1 < ti) {  // the blocks between
        x *= lds4(E + (tj + 1) * dkp + 16 * kk + g4);
        if (tj + 2 < ti) x *= lds4(E + (tj + 2) * dkp + 16 * kk + g4);
      }
      acc = block_product(x, lds4(yr + 16 * kk), acc);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) P[(16 * ti + g4 + r) * AS + 16 * tj + (lane & 15)] = acc[r];
  }
  f32x4 o[4];
#pragma unroll
  for (int m = 0; m < 4; ++m) o[m] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto read_out = [&](int kk, f32x4 s) {
#pragma unroll
    for (int m = 0; m < 4; ++m)
      o[m] = block_product(lds4(Qs + (16 * m + (lane & 15)) * ks + 16 * kk + g4) * lds4(pre + m * dkp + 16 * kk + g4), s, o[m]);
  };
  if constexpr (NKK > 0 && NKK < 8) {
#pragma unroll
    for (int kk = 0; kk < NKK; ++kk) read_out(kk, s0[kk]);
  } else {
    for (int kk = 0; kk < nkk; ++kk) read_out(kk, load_state(kk));
  }
  __syncthreads();
#pragma unroll
  for (int m = 0; m < 4; ++m) {
#pragma unroll
    for (int c = 0; c <= m; ++c) o[m] = block_product(lds4(P + (16 * m + (lane & 15)) * AS + 16 * c + g4), y[c], o[m]);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int t = 16 * m + g4 + r;
      if (cok && t < n) a.out[((int64_t)(t0 + t) * a.H + h) * dv + col] = o[m][r] * a.qscale;
    }
  }
}

GCArgs gc_args(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, const at::Tensor& z, const at::Tensor& z_bias, double tau,
               double qscale, const at::Tensor& cu) {
  HYB_CHECK(q.dim() == 3 && v.dim() == 3, "q, k [T, H, dk], v [T, H, dv]");
  const int64_t T = q.size(0), H = q.size(1), dk = q.size(2), dv = v.size(2);
  for (const at::Tensor* t : {&q, &k, &v})
    HYB_CHECK(t->is_cuda() && t->dim() == 3 && t->size(0) == T && t->size(1) == H && t->size(2) == (t == &v ? dv : dk) &&
                  (t->size(2) == 1 || t->stride(2) == 1) && t->scalar_type() == q.scalar_type(),
              "q, k, v: [T, H, d] with unit last stride, one dtype");
  HYB_CHECK(dk >= 1 && dk <= 128 && dv >= 1 && H <= 65535, "key size 1 .. 128");
  HYB_CHECK(z.is_cuda() && z.dim() == 2 && z.size(0) == T && z.size(1) == H * dk && z.scalar_type() == at::kFloat && (z.size(1) == 1 || z.stride(1) == 1),
            "decay logits: fp32 [T, H * dk]");
  HYB_CHECK(z_bias.is_cuda() && z_bias.scalar_type() == at::kFloat && z_bias.is_contiguous() && z_bias.numel() == H * dk, "decay bias: fp32 [H * dk]");
  HYB_CHECK(cu.is_cuda() && cu.is_contiguous() && cu.scalar_type() == at::kInt && cu.numel() >= 1, "cu: int32 [chunks + 1]");
  HYB_CHECK(tau > 0.0, "tau > 0");
  GCArgs a = {};
  a.q = q.data_ptr(), a.k = k.data_ptr(), a.v = v.data_ptr();
  a.q_st = q.stride(0), a.q_sh = q.stride(1), a.k_st = k.stride(0), a.k_sh = k.stride(1), a.v_st = v.stride(0), a.v_sh = v.stride(1);
  a.z = z.data_ptr<float>(), a.z_st = z.stride(0), a.zb = z_bias.data_ptr<float>();
  a.inv_tau = (float)(1.0 / tau), a.qscale = (float)qscale;
  a.cu = cu.data_ptr<int>();
  a.H = (int)H, a.dk = (int)dk, a.dv = (int)dv;
  const size_t quad = 4 * q.element_size();
  auto rows4 = [&](const at::Tensor& t) {
    return reinterpret_cast<uintptr_t>(t.data_ptr()) % quad == 0 && t.stride(0) % 4 == 0 && t.stride(1) % 4 == 0;
  };
  a.vec = dk % 4 == 0 && rows4(q) && rows4(k);
  return a;
}

template <typename K>
void gc_launch(K kern, int64_t P, size_t lds, const GCArgs& a) {
  const int nw = waves_for(a.dv);
  if (lds > 64 * 1024)
    HYB_CHECK(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) == hipSuccess, "LDS size");
  kern<<<dim3((unsigned)P, (unsigned)a.H, (unsigned)(((a.dv + 15) / 16 + nw - 1) / nw)), 64 * nw, lds, cur_stream()>>>(a);
}
bool gc_f32(const at::Tensor& t, int64_t n) { return t.is_cuda() && t.is_contiguous() && t.scalar_type() == at::kFloat && t.numel() == n; }
}  // namespace

// chunks [cu[p], cu[p + 1]) of at most 64 rows, from zeros: loc [P, H, dk, dv] and the total log decays logd [P, H, dk]
void gla_chunk_local(const at::Tensor& k, const at::Tensor& v, const at::Tensor& z, const at::Tensor& z_bias, double tau, const at::Tensor& cu,
                     at::Tensor loc, at::Tensor logd) {
  GCArgs a = gc_args(k, k, v, z, z_bias, tau, 1.0, cu);
  const int64_t P = cu.numel() - 1;
  HYB_CHECK(gc_f32(loc, P * a.H * a.dk * a.dv) && gc_f32(logd, P * a.H * a.dk), "loc: fp32 [chunks, H, dk, dv], logd: fp32 [chunks, H, dk]");
  if (P == 0) return;
  c10::DeviceGuard guard(k.device());
  a.loc = loc.data_ptr<float>(), a.logd = logd.data_ptr<float>();
  const int w = staged_width(a.dk);
  const size_t lds = sizeof(float) * (size_t)(2 * CH * (w + 4) + 8 * w);
  dispatch_act(k, [&](auto* tag) {
    using Tt = std::remove_pointer_t<decltype(tag)>;
    by_width(a.dk, [&](auto nkk) { gc_launch(gla_chunk_local_kernel<Tt, decltype(nkk)::value>, P, lds, a); });
  });
}

// outputs fp32 [T, H, dv] of the chunks from the memories init [P, H, dk, dv] at their first tokens
at::Tensor gla_chunk_out(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, const at::Tensor& z, const at::Tensor& z_bias, double tau,
                         double qscale, const at::Tensor& cu, const at::Tensor& init) {
  GCArgs a = gc_args(q, k, v, z, z_bias, tau, qscale, cu);
  const int64_t P = cu.numel() - 1;
  HYB_CHECK(gc_f32(init, P * a.H * a.dk * a.dv), "chunk-start memories: fp32 [chunks, H, dk, dv]");
  c10::DeviceGuard guard(q.device());
  at::Tensor out = at::empty({q.size(0), q.size(1), v.size(2)}, q.options().dtype(at::kFloat));
  if (P == 0) return out;
  a.init = init.data_ptr<float>(), a.out = out.data_ptr<float>();
  const int w = staged_width(a.dk);
  const size_t lds = sizeof(float) * (size_t)(3 * CH * (w + 4) + CH * AS + 8 * w);
  dispatch_act(q, [&](auto* tag) {
    using Tt = std::remove_pointer_t<decltype(tag)>;
    by_width(a.dk, [&](auto nkk) { gc_launch(gla_chunk_out_kernel<Tt, decltype(nkk)::value>, P, lds, a); });
  });
  return out;
}

}  // namespace llmctl_hybrid
