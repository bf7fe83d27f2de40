// y[M, N] = act(x[M, K] W[N, K]^T + bias) for few rows (M <= 32): a stream of W over the matrix cores, in one launch.
//
// The bound is the weight stream and, below some 20 MB of weights, the latency of one round trip to HBM plus the launch
// (3.5 us in a graph).  Measured beside the library's product (one MI355X, weights from HBM, 16 rows, us):
//   N x K        768 x 768  768 x 3072  2048 x 2048  2048 x 4096  4240 x 2048  8256 x 2048  9248 x 2048  10496 x 2048  32000 x 2048
//   library          5.1         9.3         8.4         14.8         12.2         14.2         14.5         15.1          34
//   whole tiles      4.1         8.0         6.3         10.2         10.4         15.0         15.5         16.0          29
//   here             4.0         6.7         5.8          9.1          7.9         11.1         11.8         12.7          30
// A workgroup owns whole outputs (no partial sums between workgroups) and draws some 30 GB/s, so all 256 CUs must have the same number of them:
// it owns N / 256 outputs (or an even part, see launch), whatever that is, and the MFMA tiles' other rows repeat its last one (``whole tiles``:
// 16 or 32 outputs each, which left CUs idle below 4096 outputs and made two uneven rounds above 8192).  With K beyond 4096 a
// workgroup's own read of x weighs as much as its weights: 2048 x 8192 takes 16 us against the library's 13.7, which splits K over the
// chip.  The callers' rules (llmctl/ops/functional.py: stream_pays, decode_form) leave such shapes.
#pragma once

#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>

#include <cstdint>

namespace stream_linear {

using frag_t = __attribute__((ext_vector_type(8))) __bf16;
using acc_t = __attribute__((ext_vector_type(4))) float;

struct Args {
  const unsigned short* x;
  long ldx;
  const unsigned short* w;
  long ldw;
  const unsigned short* bias;  // bf16 [N] or null
  void* y;                     // [M, N], bf16 or fp32
  int M, N, K;
  int act;       // 0 none, 1 gelu (erf), 2 gelu (tanh), 3 relu^2
  int act_cols;  // of the first that many columns
  int f32;  // y is fp32
  int rows = 0;  // outputs of a workgroup, at most 16 NT
  int part = 0;  // > 0: blockIdx.y takes that much of K (a multiple of 32) and writes its own fp32 y [M, N]; no bias, no activation
};

__device__ __forceinline__ uint4 load_or_zero(const unsigned short* p, bool in) {
  uint4 v = make_uint4(0, 0, 0, 0);
  if (in) v = *reinterpret_cast<const uint4*>(p);
  return v;
}

__device__ __forceinline__ float activate(int act, float v) {
  if (act == 1) return 0.5f * v * (1.0f + erff(v * 0.70710678118654752440f));
  if (act == 2) {
    const float u = 0.7978845608028654f * (v + 0.044715f * v * v * v);
    return 0.5f * v * (1.0f + tanhf(u));
  }
  if (act == 3) {
    const float r = fmaxf(v, 0.f);
    return r * r;
  }
  return v;
}

// A workgroup of NW waves owns ``rows`` weight rows, at most 16 NT; the waves split K.  A lane streams 16 bytes of its weight row per 32-deep step,
// U steps in flight before the first MFMA; the weight fragment is the MFMA row operand, so a lane ends up with four
// neighbouring outputs of one token.  K is a multiple of 8 (the last step is filled up with zeros), N any.
// Workgroup (bx, by); red: LDS for the waves' sums.
template <int NT, int MT, int NW, int U>
__device__ __forceinline__ void workgroup(Args g, unsigned bx, unsigned by, acc_t (*red)[NT * MT][64]) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r = lane & 15, kg = lane >> 4;
  if (g.part > 0) {
    const int k0 = by * g.part;
    g.x += k0;
    g.w += k0;
    g.K = min(g.part, g.K - k0);
    g.y = static_cast<float*>(g.y) + (long)by * g.M * g.N;
  }
  const int n0 = bx * g.rows, n1 = min(n0 + g.rows, g.N);
  const unsigned short* wp[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) wp[n] = g.w + (long)min(n0 + n * 16 + r, n1 - 1) * g.ldw + 8 * kg;
  const unsigned short* xp[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) xp[m] = g.x + (long)min(m * 16 + r, g.M - 1) * g.ldx + 8 * kg;
  acc_t acc[NT][MT];
#pragma unroll
  for (int n = 0; n < NT; ++n)
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[n][m] = acc_t{0.f, 0.f, 0.f, 0.f};
  const int steps = (g.K + 31) / 32, per = (steps + NW - 1) / NW;
  const int s0 = wave * per, s1 = min(s0 + per, steps), whole = min(s1, g.K / 32);
  for (int s = s0; s < s1; s += U) {
    uint4 wv[U][NT], xv[U][MT];
    if (s + U <= whole) {
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int n = 0; n < NT; ++n) wv[u][n] = *reinterpret_cast<const uint4*>(wp[n] + (s + u) * 32);
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int m = 0; m < MT; ++m) xv[u][m] = *reinterpret_cast<const uint4*>(xp[m] + (s + u) * 32);
    } else {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const bool in = s + u < s1 && (s + u) * 32 + 8 * kg < g.K;
#pragma unroll
        for (int n = 0; n < NT; ++n) wv[u][n] = load_or_zero(wp[n] + (s + u) * 32, in);
#pragma unroll
        for (int m = 0; m < MT; ++m) xv[u][m] = load_or_zero(xp[m] + (s + u) * 32, in);
      }
    }
    __builtin_amdgcn_sched_barrier(0);  // the whole batch in flight before the first MFMA
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int m = 0; m < MT; ++m)
          acc[n][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(frag_t, wv[u][n]), __builtin_bit_cast(frag_t, xv[u][m]),
                                                              acc[n][m], 0, 0, 0);
  }
#pragma unroll
  for (int n = 0; n < NT; ++n)
#pragma unroll
    for (int m = 0; m < MT; ++m) red[wave][n * MT + m][lane] = acc[n][m];
  __syncthreads();
  for (int i = tid; i < NT * MT * 64; i += NW * 64) {
    const int t = i >> 6, l = i & 63, row = (t % MT) * 16 + (l & 15), c = n0 + (t / MT) * 16 + 4 * (l >> 4);
    if (row >= g.M || c >= n1) continue;
    acc_t s = red[0][t][l];
#pragma unroll
    for (int v = 1; v < NW; ++v) s += red[v][t][l];
    const long o = (long)row * g.N + c;
    const int left = min(4, n1 - c);
    float v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float b = g.bias != nullptr && j < left ? __uint_as_float((unsigned)g.bias[c + j] << 16) : 0.f;
      v[j] = activate(c + j < g.act_cols ? g.act : 0, s[j] + b);
    }
    if (g.f32) {
      float* y = static_cast<float*>(g.y) + o;
      if (left == 4 && (reinterpret_cast<uintptr_t>(y) & 15) == 0) *reinterpret_cast<float4*>(y) = make_float4(v[0], v[1], v[2], v[3]);
      else
#pragma unroll  // (a loop of ``left`` turns would index the values by a register: through LDS, 8256 x 2048 24 us for 11.5)
        for (int j = 0; j < 4; ++j)
          if (j < left) y[j] = v[j];
    } else {
      unsigned short* y = static_cast<unsigned short*>(g.y) + o;
      unsigned short h[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) h[j] = __bfloat16_as_ushort(__float2bfloat16(v[j]));
      if (left == 4 && (reinterpret_cast<uintptr_t>(y) & 7) == 0) *reinterpret_cast<uint2*>(y) = make_uint2(h[0] | ((unsigned)h[1] << 16), h[2] | ((unsigned)h[3] << 16));
      else
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (j < left) y[j] = h[j];
    }
  }
}

// Weight rows per workgroup: one round of 256 workgroups where they own at most 64 rows each, else even rounds.  Up to four rows of x cost next to nothing, and
// from 6144 outputs on smaller workgroups in more rounds hide the latency better (one row, one round / rounds of at most 16 weight rows: 8192 x 2048 9.9 / 8.5 us,
// 12288 x 2048 13.0 / 12.0, 8192 x 2304 11.3 / 9.9; four rows from K 3072 on the other way: 9248 x 4096 17.7 / 18.3, so rounds of 32 there).  Half as many rows where those
// of W lie a multiple of 8192 entries apart and crowd the same channels (16384 x 8192: four rows of x 64.8 / 53.9, five 72.9 / 57.6), and for more than 12288 short
// ones (five rows 15360 x 1024 9.7 / 8.9).  Below K 512 a workgroup of its own for a few outputs costs more than idle CUs: whole tiles (768 x 256
// 3.3 / 2.9).  The waves and so the order of a sum depend on M, N and K alone, not on who owns an output (8 waves of 4 steps instead of 4 of 8: N 2048 6.00 / 6.06
// us, N 4096 7.16 / 7.26, not worth other results).
struct Form {
  int nt, mt, nw, u, rows;
};
inline Form form_of(int M, int N, int K) {
  const bool few = M <= 4 && N >= 6144;
  int rows;
  if (K < 512) {
    rows = few || N < 5120 ? 16 : M > 16 || N < 24576 ? 32 : 64;
  } else {
    int tall = !few ? 64 : N > 16384 || K <= 2048 || (M <= 3 && N <= 8192 && K <= 3072) ? 16 : 32;  // rows of a workgroup at most
    if (M <= 16 && N <= 16384) {
      if (K % 8192 == 0 && N > (few ? 8192 : 12288)) tall /= 2;
      else if (!few && K <= 1024 && N > 12288) tall = 32;
    }
    const int rounds = (N + 256 * tall - 1) / (256 * tall);  // of 256 workgroups
    rows = (N + 256 * rounds - 1) / (256 * rounds);
    if (N > 16384) rows = few ? 16 : (rows + 3) / 4 * 4;  // (whole quads are stored at once)
  }
  const int nt = rows <= 16 ? 1 : rows <= 32 ? 2 : rows <= 48 ? 3 : 4;
  if (M > 16) return {nt, 2, 4, nt == 1 ? 8 : 4, rows};
  if (nt == 1) return {1, 1, few ? 2 : 4, 8, rows};
  if (nt == 2) return {2, 1, 4, few ? 4 : 8, rows};
  return {nt, 1, 4, 4, rows};
}

}  // namespace stream_linear
