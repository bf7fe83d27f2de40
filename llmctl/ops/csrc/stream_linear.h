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
// Workgroup (bx, by) of a launch that does other things too; red: LDS for the waves' sums.
template <int NT, int MT, int NW, int U>
__device__ __forceinline__ void workgroup(Args g, unsigned bx, unsigned by, acc_t (*red)[NT * MT][64]) {
#include "stream_linear_body.inc"
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
