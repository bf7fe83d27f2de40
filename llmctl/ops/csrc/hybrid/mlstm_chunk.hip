// mLSTM over long portions: the recurrence of mlstm.hip in chunks of 64 tokens, as fp32 matrix products (chunk_mfma.h).
//
// With L_t the running sum of the log forget gates inside a chunk, A_s = i_s - L_s and N_t = max(m_0, max_(s <= t) A_s), the
// sequential form's stabiliser is m_t = L_t + N_t and
//   num_t = sum_(s <= t) e^(A_s - N_t) (q_t . k_s) v_s + e^(m_0 - N_t) S_0^T q_t,   o_t = num_t / (max(|nq_t|, e^(-m_t)) + 1e-6),
// nq_t the same sum with 1 for v_s and n_0 for S_0.  All exponents are <= 0.  L, A and N are formed in double and kept as pairs of
// floats (differences of large sums stay exact).
//   mlstm_chunk_local   every chunk from a zero state with m = -inf: its contribution (S_loc, n_loc, m_loc) and L_n
//   mlstm_chunk_combine the state at every chunk's first token in order, and the sequence's new carried state:
//                       m' = max(L_n + m, m_loc), S' = e^(L_n + m - m') S + e^(m_loc - m') S_loc
//   mlstm_chunk_out     every chunk's outputs from the state at its first token
//
// Bound: the chain of loads, scores and products of a chunk; a token-by-token scan of the same chunks spends 64 dependent
// steps of 32 LDS reads each.  16 heads of 64 x 128, one portion of 2048 tokens: 192 us per pass of the scan, two passes, before; 18 + 13 +
// 27 us now (whole call, us, before / now: 2048 tokens 426 / 83, 8192 490 / 197, keys of 128 at 2048 825 / 117).
#include "chunk_mfma.h"

namespace llmctl_hybrid {
namespace {

struct MLArgs {
  const void* q;
  const void* k;
  const void* v;
  int64_t st;         // row stride of q, k, v (elements); heads back to back
  const float* raw;   // [T, 2H] gate pre-activations, input gates first
  const float* b_i;
  const float* b_f;
  float cap, qscale;
  const int* cu;      // [P + 1] chunk row offsets
  const int* seq;     // [P] sequence of a chunk
  const int* base;    // [ns + 1] first chunk of a sequence
  const int* slots;
  const int* start;
  const float* m;     // [slots, H]
  float* locS;        // [P, H, dk, dv]
  float* locn;        // [P, H, dk]
  float* locm;        // [P, H]
  float* fsum;        // [P, H]
  float* m0;          // [ns, H]: the carried log-scale before this step
  const float* iS;    // the state at every chunk's first token
  const float* in_;
  const float* im;
  float* out;         // [T, H, dv]
  int H, dk, dv, vec;
};

__device__ __forceinline__ float log_sig(float x) { return fminf(x, 0.f) - log1pf(expf(-fabsf(x))); }

// lane t of the first wave: L_t and the running maximum M_t of A_s = i_s - L_s (tokens past n: no decay, no write)
struct Gate {
  double L, A, M;
};
__device__ __forceinline__ Gate chunk_gates(const MLArgs& a, float zi, float zf, int h, int n) {
  const int t = threadIdx.x;
  float ig = -INFINITY, fg = 0.f;
  if (t < n) {
    ig = a.cap * tanhf((zi + a.b_i[h]) / a.cap);
    fg = log_sig(a.cap * tanhf((zf + a.b_f[h]) / a.cap));
  }
  Gate g;
  g.L = (double)fg;
#pragma unroll
  for (int o = 1; o < CH; o <<= 1) {
    const double up = __shfl_up(g.L, o, 64);
    if (t >= o) g.L += up;
  }
  g.A = (double)ig - g.L;
  g.M = g.A;
#pragma unroll
  for (int o = 1; o < CH; o <<= 1) {
    const double up = __shfl_up(g.M, o, 64);
    if (t >= o) g.M = fmax(g.M, up);
  }
  return g;
}

// A wave takes 16 value columns: its V rows in registers, K and the gates through LDS.
template <typename T, int NKK>
__global__ __launch_bounds__(512, 4) void mlstm_chunk_local_kernel(MLArgs a) {
  extern __shared__ __attribute__((aligned(16))) float smem[];
  const int p = blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6, nw = blockDim.x >> 6;
  const int t0 = a.cu[p], n = a.cu[p + 1] - t0;
  const int dk = a.dk, dv = a.dv, nkk = NKK > 0 ? NKK : (dk + 15) / 16, dkp = 16 * nkk, ks = dkp + 4;
  float* Ks = smem;
  float* w = Ks + CH * ks;
  const int col = (blockIdx.z * nw + wave) * 16 + (lane & 15), g4 = (lane >> 4) * 4;
  const bool cok = col < dv;
  const T* kp = reinterpret_cast<const T*>(a.k) + t0 * a.st + (int64_t)h * dk;
  const T* vp = reinterpret_cast<const T*>(a.v) + t0 * a.st + (int64_t)h * dv;
  float zi = 0.f, zf = 0.f;
  if (tid < n) {  // (n <= 64: the first wave)
    zi = a.raw[(int64_t)(t0 + tid) * 2 * a.H + h];
    zf = a.raw[(int64_t)(t0 + tid) * 2 * a.H + a.H + h];
  }
  f32x4 y[4];
#pragma unroll
  for (int m = 0; m < 4; ++m)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int t = 16 * m + g4 + r;
      y[m][r] = (cok && t < n) ? ldf(vp + t * a.st + col) : 0.f;
    }
  stage_rows(Ks, ks, kp, a.st, n, dk, dkp, a.vec != 0);
  if (tid < CH) {
    const Gate g = chunk_gates(a, zi, zf, h, n);
    const double Mn = __shfl(g.M, CH - 1, 64);
    w[tid] = tid < n ? expf((float)(g.A - Mn)) : 0.f;
    if (blockIdx.z == 0 && tid == CH - 1) {
      a.fsum[(int64_t)p * a.H + h] = (float)g.L;
      a.locm[(int64_t)p * a.H + h] = (float)(g.L + Mn);
      const int s = a.seq[p];
      if (p == a.base[s]) a.m0[(int64_t)s * a.H + h] = a.start[s] == 0 ? 0.f : a.m[(int64_t)a.slots[s] * a.H + h];
    }
  }
  __syncthreads();
#pragma unroll
  for (int m = 0; m < 4; ++m)
#pragma unroll
    for (int r = 0; r < 4; ++r) y[m][r] *= w[16 * m + g4 + r];
  for (int dt = 0; dt < nkk; ++dt) {
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc = mfma4(Ks[(16 * m + g4 + j) * ks + 16 * dt + (lane & 15)], y[m][j], acc);
    float* o = a.locS + (((int64_t)p * a.H + h) * dk + 16 * dt + g4) * dv + col;
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (cok && 16 * dt + g4 + r < dk) o[(int64_t)r * dv] = acc[r];
  }
  if (blockIdx.z == 0) {
    for (int d = tid; d < dk; d += blockDim.x) {
      float s = 0.f;
#pragma unroll 8
      for (int t = 0; t < CH; ++t) s += w[t] * Ks[t * ks + d];
      a.locn[((int64_t)p * a.H + h) * dk + d] = s;
    }
  }
}

// LDS: K [CH][ks] | Q [CH][ks] | scores [CH][AS] | gate arrays
template <typename T, int NKK>
__global__ __launch_bounds__(512, 4) void mlstm_chunk_out_kernel(MLArgs a) {
  extern __shared__ __attribute__((aligned(16))) float smem[];
  const int p = blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6, nw = blockDim.x >> 6;
  const int t0 = a.cu[p], n = a.cu[p + 1] - t0;
  const int dk = a.dk, dv = a.dv, nkk = NKK > 0 ? NKK : (dk + 15) / 16, dkp = 16 * nkk, ks = dkp + 4;
  float* Ks = smem;
  float* Qs = Ks + CH * ks;
  float* P = Qs + CH * ks;
  float* Ahi = P + CH * AS;
  float *Alo = Ahi + CH, *Nhi = Alo + CH, *Nlo = Nhi + CH, *grow = Nlo + CH, *floor_ = grow + CH, *inv = floor_ + CH;
  const int col = (blockIdx.z * nw + wave) * 16 + (lane & 15), g4 = (lane >> 4) * 4;
  const bool cok = col < dv;
  const int64_t ph = (int64_t)p * a.H + h;
  const T* qp = reinterpret_cast<const T*>(a.q) + t0 * a.st + (int64_t)h * dk;
  const T* kp = reinterpret_cast<const T*>(a.k) + t0 * a.st + (int64_t)h * dk;
  const T* vp = reinterpret_cast<const T*>(a.v) + t0 * a.st + (int64_t)h * dv;
  float zi = 0.f, zf = 0.f;
  if (tid < n) {
    zi = a.raw[(int64_t)(t0 + tid) * 2 * a.H + h];
    zf = a.raw[(int64_t)(t0 + tid) * 2 * a.H + a.H + h];
  }
  const float m0 = a.im[ph];
  f32x4 y[4];
#pragma unroll
  for (int m = 0; m < 4; ++m)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int t = 16 * m + g4 + r;
      y[m][r] = (cok && t < n) ? ldf(vp + t * a.st + col) : 0.f;
    }
  const float* S0 = a.iS + ph * dk * dv + (cok ? col : dv - 1);
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
  stage_rows(Ks, ks, kp, a.st, n, dk, dkp, a.vec != 0);
  stage_rows(Qs, ks, qp, a.st, n, dk, dkp, a.vec != 0);
  if (tid < CH) {
    const Gate g = chunk_gates(a, zi, zf, h, n);
    const double N = fmax((double)m0, g.M);
    Ahi[tid] = (float)g.A;
    Alo[tid] = tid < n ? (float)(g.A - (double)(float)g.A) : 0.f;
    Nhi[tid] = (float)N;
    Nlo[tid] = (float)(N - (double)(float)N);
    grow[tid] = expf((float)((double)m0 - N)) * a.qscale;
    floor_[tid] = expf(-(float)(g.L + N));
  }
  __syncthreads();
  for (int i = wave; i < 10; i += nw) {
    int ti, tj;
    lower_tile(i, ti, tj);
    const f32x4 acc = score_tile<NKK>(Qs, Ks, ks, nkk, ti, tj, lane);
    const int s = 16 * tj + (lane & 15);
    const float shi = Ahi[s], slo = Alo[s];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int t = 16 * ti + g4 + r;
      P[t * AS + s] = s <= t ? acc[r] * a.qscale * expf((shi - Nhi[t]) + (slo - Nlo[t])) : 0.f;
    }
  }
  f32x4 o[4];
#pragma unroll
  for (int m = 0; m < 4; ++m) o[m] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto read_out = [&](int kk, f32x4 s) {
#pragma unroll
    for (int m = 0; m < 4; ++m) o[m] = block_product(lds4(Qs + (16 * m + (lane & 15)) * ks + 16 * kk + g4), s, o[m]);
  };
  if constexpr (NKK > 0 && NKK < 8) {
#pragma unroll
    for (int kk = 0; kk < NKK; ++kk) read_out(kk, s0[kk]);
  } else {
    for (int kk = 0; kk < nkk; ++kk) read_out(kk, load_state(kk));
  }
  __syncthreads();
  // the normaliser: four threads per token sum a quarter of its weights and of q . n_0 each
  if (tid < 4 * CH) {
    const int t = tid >> 2, part = tid & 3, last = min(16 * part + 15, t);
    float nq = 0.f, qn = 0.f;
    for (int s = 16 * part; s <= last; ++s) nq += P[t * AS + s];
    for (int d = part * 4; d < dk; d += 16)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (d + j < dk) qn += Qs[t * ks + d + j] * a.in_[ph * dk + d + j];
    nq += grow[t] * qn;
    nq += __shfl_xor(nq, 1, 64);
    nq += __shfl_xor(nq, 2, 64);
    if (part == 0) inv[t] = 1.0f / (fmaxf(fabsf(nq), floor_[t]) + 1e-6f);
  }
#pragma unroll
  for (int m = 0; m < 4; ++m) {
#pragma unroll
    for (int r = 0; r < 4; ++r) o[m][r] *= grow[16 * m + g4 + r];
#pragma unroll
    for (int c = 0; c <= m; ++c) o[m] = block_product(lds4(P + (16 * m + (lane & 15)) * AS + 16 * c + g4), y[c], o[m]);
  }
  __syncthreads();
#pragma unroll
  for (int m = 0; m < 4; ++m)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int t = 16 * m + g4 + r;
      if (cok && t < n) a.out[((int64_t)(t0 + t) * a.H + h) * dv + col] = o[m][r] * inv[t];
    }
}

// One thread per state entry (S, then n), chunks in order.  The log-scales come from copies (m0, locm, fsum), so the thread that
// stores the sequence's new one races with nobody.
__global__ __launch_bounds__(256) void mlstm_chunk_combine_kernel(float* __restrict__ Sp, float* __restrict__ np, float* __restrict__ mp,
                                                                  const int* __restrict__ slots, const int* __restrict__ start,
                                                                  const int* __restrict__ base, const float* __restrict__ locS,
                                                                  const float* __restrict__ locn, const float* __restrict__ locm,
                                                                  const float* __restrict__ fsum, const float* __restrict__ m0,
                                                                  float* __restrict__ iS, float* __restrict__ in_, float* __restrict__ im,
                                                                  int H, int dk, int dv) {
  constexpr int CB = 8;  // chunks fetched ahead as one batch
  const int s = blockIdx.x, h = blockIdx.y;
  const int64_t nS = (int64_t)dk * dv, e = (int64_t)blockIdx.z * 256 + threadIdx.x;
  const int lo = base[s], hi = base[s + 1];
  if (e >= nS + dk || lo == hi) return;
  const bool isn = e >= nS;
  const int64_t eo = isn ? e - nS : e, stride = isn ? dk : nS;
  const float* loc = isn ? locn : locS;
  float* init = isn ? in_ : iS;
  const int64_t at = (int64_t)slots[s] * H + h;
  float* real = (isn ? np : Sp) + at * stride + eo;
  float val = start[s] == 0 ? 0.f : *real, m = m0[(int64_t)s * H + h];
  float l[CB], F[CB], ml[CB];
  for (int p0 = lo; p0 < hi; p0 += CB) {
#pragma unroll
    for (int i = 0; i < CB; ++i) {
      const int64_t ph = (int64_t)min(p0 + i, hi - 1) * H + h;
      l[i] = loc[ph * stride + eo], F[i] = fsum[ph], ml[i] = locm[ph];
    }
#pragma unroll
    for (int i = 0; i < CB; ++i) {
      if (p0 + i < hi) {
        const int64_t ph = (int64_t)(p0 + i) * H + h;
        init[ph * stride + eo] = val;
        if (e == 0) im[ph] = m;
        const float mn = fmaxf(F[i] + m, ml[i]);
        val = expf(F[i] + m - mn) * val + expf(ml[i] - mn) * l[i];
        m = mn;
      }
    }
  }
  *real = val;
  if (e == 0) mp[at] = m;
}

bool f32c(const at::Tensor& t, int64_t n) { return t.is_cuda() && t.is_contiguous() && t.scalar_type() == at::kFloat && t.numel() == n; }
bool i32c(const at::Tensor& t, int64_t n) { return t.is_cuda() && t.is_contiguous() && t.scalar_type() == at::kInt && t.numel() == n; }
}  // namespace

// The whole step: chunks [cu[p], cu[p + 1]) of at most 64 rows, sequence s owning chunks [base[s], base[s + 1]).
at::Tensor mlstm_chunked(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, const at::Tensor& raw, const at::Tensor& b_i,
                         const at::Tensor& b_f, double cap, double qscale, at::Tensor S, at::Tensor n, at::Tensor m, const at::Tensor& slots,
                         const at::Tensor& start, const at::Tensor& cu, const at::Tensor& seq, const at::Tensor& base) {
  HYB_CHECK(q.is_cuda() && q.dim() == 3 && v.dim() == 3, "q, k [T, H, dk], v [T, H, dv]");
  const int64_t T = q.size(0), H = q.size(1), dk = q.size(2), dv = v.size(2), P = seq.numel(), ns = slots.numel();
  const int64_t st = T > 1 ? q.stride(0) : H * std::max(dk, dv);
  for (const at::Tensor* t : {&q, &k, &v}) {
    const int64_t d = t == &v ? dv : dk;
    HYB_CHECK(t->is_cuda() && t->dim() == 3 && t->size(0) == T && t->size(1) == H && t->size(2) == d && (d == 1 || t->stride(2) == 1) &&
                  (H == 1 || t->stride(1) == d) && (T <= 1 || t->stride(0) == st) && t->scalar_type() == q.scalar_type(),
              "q, k, v: [T, H, d] rows of one projection output");
  }
  HYB_CHECK(dk >= 1 && dk <= 128 && dv >= 1 && H <= 65535, "key size 1 .. 128");
  HYB_CHECK(f32c(raw, T * 2 * H) && f32c(b_i, H) && f32c(b_f, H), "gates: fp32 [T, 2H], biases [H]");
  HYB_CHECK(S.dim() == 4 && f32c(S, S.size(0) * H * dk * dv) && S.size(1) == H && S.size(2) == dk && f32c(n, S.size(0) * H * dk) && f32c(m, S.size(0) * H),
            "state pools: contiguous fp32 [slots, H, dk, dv], [slots, H, dk], [slots, H]");
  HYB_CHECK(i32c(slots, ns) && i32c(start, ns) && i32c(cu, P + 1) && i32c(seq, P) && i32c(base, ns + 1), "slots, start [n], cu [P + 1], seq [P], base [n + 1]: int32");
  c10::DeviceGuard guard(q.device());
  const auto f32 = q.options().dtype(at::kFloat);
  at::Tensor out = at::empty({T, H, dv}, f32);
  if (T == 0 || P == 0) return out;
  HYB_CHECK((dk * dv + dk + 255) / 256 <= 65535, "grid too large");
  at::Tensor locS = at::empty({P, H, dk, dv}, f32), iS = at::empty_like(locS);
  at::Tensor locn = at::empty({P, H, dk}, f32), in_ = at::empty_like(locn);
  at::Tensor locm = at::empty({P, H}, f32), fsum = at::empty_like(locm), im = at::empty_like(locm), m0 = at::empty({ns, H}, f32);
  MLArgs a;
  a.q = q.data_ptr(), a.k = k.data_ptr(), a.v = v.data_ptr(), a.st = st;
  a.raw = raw.data_ptr<float>(), a.b_i = b_i.data_ptr<float>(), a.b_f = b_f.data_ptr<float>(), a.cap = (float)cap, a.qscale = (float)qscale;
  a.cu = cu.data_ptr<int>(), a.seq = seq.data_ptr<int>(), a.base = base.data_ptr<int>(), a.slots = slots.data_ptr<int>(), a.start = start.data_ptr<int>();
  a.m = m.data_ptr<float>();
  a.locS = locS.data_ptr<float>(), a.locn = locn.data_ptr<float>(), a.locm = locm.data_ptr<float>(), a.fsum = fsum.data_ptr<float>(), a.m0 = m0.data_ptr<float>();
  a.iS = iS.data_ptr<float>(), a.in_ = in_.data_ptr<float>(), a.im = im.data_ptr<float>();
  a.out = out.data_ptr<float>();
  a.H = (int)H, a.dk = (int)dk, a.dv = (int)dv;
  const size_t quad = 4 * q.element_size();
  auto rows4 = [&](const at::Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % quad == 0; };
  a.vec = dk % 4 == 0 && st % 4 == 0 && rows4(q) && rows4(k);
  const int nw = waves_for((int)dv), ks = staged_width((int)dk) + 4;
  const dim3 grid((unsigned)P, (unsigned)H, (unsigned)(((dv + 15) / 16 + nw - 1) / nw));
  const size_t lds_local = sizeof(float) * (size_t)(CH * ks + CH), lds_out = sizeof(float) * (size_t)(2 * CH * ks + CH * AS + 7 * CH);
  const hipStream_t stream = cur_stream();
  auto launch = [&](auto kern, size_t lds) {
    if (lds > 64 * 1024)
      HYB_CHECK(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) == hipSuccess, "LDS size");
    kern<<<grid, 64 * nw, lds, stream>>>(a);
  };
  dispatch_act(q, [&](auto* tag) {
    using Tt = std::remove_pointer_t<decltype(tag)>;
    by_width((int)dk, [&](auto nkk) { launch(mlstm_chunk_local_kernel<Tt, decltype(nkk)::value>, lds_local); });
    mlstm_chunk_combine_kernel<<<dim3((unsigned)ns, (unsigned)H, (unsigned)((dk * dv + dk + 255) / 256)), 256, 0, stream>>>(
        S.data_ptr<float>(), n.data_ptr<float>(), m.data_ptr<float>(), a.slots, a.start, a.base, a.locS, a.locn, a.locm, a.fsum, a.m0,
        iS.data_ptr<float>(), in_.data_ptr<float>(), im.data_ptr<float>(), (int)H, (int)dk, (int)dv);
    by_width((int)dk, [&](auto nkk) { launch(mlstm_chunk_out_kernel<Tt, decltype(nkk)::value>, lds_out); });
  });
  return out;
}

}  // namespace llmctl_hybrid
