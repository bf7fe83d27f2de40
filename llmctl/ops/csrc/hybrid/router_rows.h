// The router's choice for one token, and the router of rows that a norm kernel has just made.
#pragma once

#include "hybrid_common.h"

#include <type_traits>

namespace llmctl_hybrid {

constexpr int MAX_ROUTED = 128;  // router outputs

struct RouterChoice {
  const float* bias;  // [E] or null: added to the scores for the choice alone
  int E, top, G, keep, softmax, renorm;
};

RouterChoice router_choice(const at::Tensor& w, int64_t W, const c10::optional<at::Tensor>& bias, int64_t top, int64_t groups, int64_t keep, bool softmax,
                           bool renorm);

// Over the wave, or (not ``wide``) over its first 16 lanes, where alone the result then is.
__device__ __forceinline__ float wave_max_of(float v, bool wide) {
  if (wide) return wave_max(v);
  v = fmaxf(v, row_ror<8>(v)), v = fmaxf(v, row_ror<4>(v)), v = fmaxf(v, row_ror<2>(v));
  return fmaxf(v, row_ror<1>(v));
}
__device__ __forceinline__ float wave_sum_of(float v, bool wide) {
  if (wide) return wave_sum(v);
  v += row_ror<8>(v), v += row_ror<4>(v), v += row_ror<2>(v);
  return v + row_ror<1>(v);
}

// The lowest index of the largest of up to 128 values, two per lane (indices lane and lane + 64), among those with ``in``; the
// lowest index with ``in`` where no value compares (NaN).  At least one must have it.
__device__ __forceinline__ int wave_argmax2(const float (&v)[2], const bool (&in)[2], bool wide) {
  const float m = wave_max_of(fmaxf(in[0] ? v[0] : -INFINITY, in[1] ? v[1] : -INFINITY), wide);
  unsigned long long m0 = __ballot(in[0] && v[0] == m), m1 = __ballot(in[1] && v[1] == m);
  if (!(m0 | m1)) m0 = __ballot(in[0]), m1 = __ballot(in[1]);
  return m0 ? __ffsll(m0) - 1 : 63 + __ffsll(m1);
}

// Choose for one token by its logits ``lg`` [E] in LDS (overwritten), one wave.
__device__ __forceinline__ void choose_experts(float* lg, int lane, const RouterChoice& c, int* __restrict__ idx, float* __restrict__ wgt) {
  const bool wide = c.E > 16;
      // lane holds router outputs lane and lane + 64
  float p[2], s[2];
  bool in[2];  // may still be chosen
  float mx = 0.f, inv = 1.f;
#pragma unroll
  for (int h = 0; h < 2; ++h) p[h] = lane + 64 * h < c.E ? lg[lane + 64 * h] : -INFINITY;
  if (c.softmax) {
    mx = wave_max_of(fmaxf(p[0], p[1]), wide);
    inv = 1.0f / wave_sum_of(expf(p[0] - mx) + expf(p[1] - mx), wide);
  }
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int e = lane + 64 * h;
    in[h] = e < c.E;
    p[h] = c.softmax ? expf(p[h] - mx) * inv : 1.0f / (1.0f + expf(-p[h]));
    s[h] = p[h] + (c.bias != nullptr && in[h] ? c.bias[e] : 0.f);
    if (in[h]) lg[e] = s[h];
  }
  if (c.G > 1) {
    // a group's score: the sum of its two best (sigmoid router) or its best choice score; the ``keep`` best groups stay open
    const int per = c.E / c.G;
    float gs[2];
    bool gin[2];
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int gi = lane + 64 * h;
      gin[h] = gi < c.G;
      float a = -INFINITY, b = -INFINITY;
      if (gin[h])
        for (int e = gi * per; e < (gi + 1) * per; ++e) {
          const float v = lg[e];
          b = fmaxf(b, fminf(a, v));
          a = fmaxf(a, v);
        }
      gs[h] = c.softmax || per == 1 ? a : a + b;
    }
    unsigned long long open[2] = {0ull, 0ull};
    for (int kk = 0; kk < c.keep; ++kk) {
      const int best = wave_argmax2(gs, gin, wide);
      if (best < 64) open[0] |= 1ull << best;
      else open[1] |= 1ull << (best - 64);
#pragma unroll
      for (int h = 0; h < 2; ++h) gin[h] = gin[h] && best != lane + 64 * h;
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int gi = min((lane + 64 * h) / per, c.G - 1);
      in[h] = in[h] && (((gi < 64 ? open[0] >> gi : open[1] >> (gi - 64)) & 1ull) != 0ull);
    }
  }
  float sum = 0.f, minew = 0.f;
  int mine = 0;
  for (int kk = 0; kk < c.top; ++kk) {  // top <= 64: lane kk keeps choice kk
    const int best = wave_argmax2(s, in, wide);
    const float pw = __shfl(best < 64 ? p[0] : p[1], best & 63);
    sum += pw;
    if (lane == kk) mine = best, minew = pw;
#pragma unroll
    for (int h = 0; h < 2; ++h) in[h] = in[h] && best != lane + 64 * h;
  }
  if (lane < c.top) {
    idx[lane] = mine;
    wgt[lane] = c.renorm ? minew * (1.0f / (sum + 1e-20f)) : minew;
  }
}

// The router weight's rows e0 .. e0 + 7, as a workgroup of NW waves multiplies them: quads threadIdx.x + i * 64 * NW.
template <int NW, int VQ>
struct RouterRows {
  float4 v[8][VQ];
  __device__ __forceinline__ void load(const float* __restrict__ w, int E, int W, int e0) {
#pragma unroll
    for (int j = 0; j < 8; ++j)
#pragma unroll
      for (int i = 0; i < VQ; ++i) v[j][i] = ld4(w + (int64_t)min(e0 + j, E - 1) * W + min(((int)threadIdx.x + i * 64 * NW) * 4, W - 4));
  }
};

// Logits of one row under the fp32 router weight w [E, W], and the choice; a workgroup of NW waves holds the row (as it rounds to bf16) in
// quads threadIdx.x + i * 64 * NW.  ``wv``: the first eight rows of the weight, asked for with the row itself.  ``part`` [NW][8] and
// ``lg`` [MAX_ROUTED] in LDS.  For steps of few rows: a row reads all of the weight, from L2, and the row's kernel is on the chip anyway
// (a launch of its own: 10 us for 16 rows; here 2).
template <int NW, int VQ>
__device__ __forceinline__ void route_row(const float* __restrict__ w, const RouterChoice& c, const float4 (&h)[VQ], RouterRows<NW, VQ>& wv, int W, float (*part)[8],
                                          float* lg, int* __restrict__ idx, float* __restrict__ wgt) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (int e0 = 0; e0 < c.E; e0 += 8) {
    if (e0 > 0) wv.load(w, c.E, W, e0);
    float a[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      a[j] = 0.f;
#pragma unroll
      for (int i = 0; i < VQ; ++i)
        if ((tid + i * 64 * NW) * 4 < W)
          a[j] = fmaf(h[i].x, wv.v[j][i].x, fmaf(h[i].y, wv.v[j][i].y, fmaf(h[i].z, wv.v[j][i].z, fmaf(h[i].w, wv.v[j][i].w, a[j]))));
    }
    // eight sums over the wave: every exchange, with the lanes 32, 16 and 8 away, halves what a lane keeps, so lane 8 v ends with sum v
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a[j]), __float_as_uint(a[j + 4]), false, false);
      a[j] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a[j]), __float_as_uint(a[j + 2]), false, false);
      a[j] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    }
    const bool high = (lane & 8) != 0;
    float t = (high ? a[1] : a[0]) + row_ror<8>(high ? a[0] : a[1]);
    auto dpp = [](float v, auto ctrl) { return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), decltype(ctrl)::value, 0xf, 0xf, true)); };
    t += dpp(dpp(t, std::integral_constant<int, 0x1b>{}), std::integral_constant<int, 0x141>{});  // quads and then eights mirrored: the lane 4 away
    t += dpp(t, std::integral_constant<int, 0x4e>{});
    t += dpp(t, std::integral_constant<int, 0xb1>{});
    if ((lane & 7) == 0) part[wave][lane >> 3] = t;
    __syncthreads();
    if (tid < 8 && e0 + tid < c.E) {
      float s = part[0][tid];
#pragma unroll
      for (int v = 1; v < NW; ++v) s += part[v][tid];
      lg[e0 + tid] = s;
    }
    __syncthreads();
  }
  if (wave == 0) choose_experts(lg, lane, c, idx, wgt);
}

// What a norm kernel needs to route its rows: ``row`` takes row r as the kernel stores it.
struct RouteOut {
  const float* w;
  RouterChoice c;
  int* idx;  // [T, top]
  float* wgt;

  template <int NW, int VQ>
  __device__ __forceinline__ void row(float4 (&h)[VQ], RouterRows<NW, VQ>& wv, int64_t r, int W) const {
    __shared__ float part[NW][8], lg[MAX_ROUTED];
    auto bf = [](float v) { return __bfloat162float(__float2bfloat16(v)); };
#pragma unroll
    for (int i = 0; i < VQ; ++i) h[i] = make_float4(bf(h[i].x), bf(h[i].y), bf(h[i].z), bf(h[i].w));
    route_row<NW, VQ>(w, c, h, wv, W, part, lg, idx + r * c.top, wgt + r * c.top);
  }
};

std::tuple<at::Tensor, at::Tensor> moe_route(const at::Tensor& x, const at::Tensor& w, const c10::optional<at::Tensor>& bias, int64_t top,
                                             int64_t groups, int64_t keep, bool softmax, bool renorm);

// The router's results for T rows, appended to ``out`` and written by a norm kernel, or by moe_route from the rows h.
inline RouteOut route_out(const at::Tensor& router, int64_t W, const c10::optional<at::Tensor>& bias, int64_t top, int64_t groups, int64_t keep,
                          bool softmax, bool renorm, int64_t T, std::vector<at::Tensor>& out) {
  const RouterChoice c = router_choice(router, W, bias, top, groups, keep, softmax, renorm);
  out.push_back(at::empty({T, top}, router.options().dtype(at::kInt)));
  out.push_back(at::empty({T, top}, router.options()));
  return RouteOut{router.data_ptr<float>(), c, out[out.size() - 2].data_ptr<int>(), out.back().data_ptr<float>()};
}
inline void add_routed(std::vector<at::Tensor>& out, const at::Tensor& h, const at::Tensor& router, const c10::optional<at::Tensor>& bias, int64_t top,
                       int64_t groups, int64_t keep, bool softmax, bool renorm) {
  auto [idx, wgt] = moe_route(h, router, bias, top, groups, keep, softmax, renorm);
  out.push_back(idx);
  out.push_back(wgt);
}

}  // namespace llmctl_hybrid
