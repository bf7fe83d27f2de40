// Products of a prompt's rows, y = act(x w^T (+ bias)) in bf16, on the tiles of wide_tiles.h: any number of rows, outputs in 8s, K in 128s from 256 on.
//
// A few hundred rows are 16 to 128 tiles, and a tile's K-tiles from HBM take a workgroup 0.5 to 0.8 us each whatever the others do (the lines that one CU can have on
// their way): such products are cut into ranges of K, one workgroup each, whose fp32 sums gemm_rows_sum adds in the order of K.
// us, one range / the best: 128 x 4096 x 11008 124 / 46 (2 TB/s), 200 x 2048 x 2048 19.0 / 13.7 (the adding pass and its launch are 6 of them), 200 x 2048 x 8192 68.7 / 22.9.
// GELUs in the epilogue: 3.9 us a tile of 256 rows, which nothing overlaps, so large products leave them to a pass (3379 x 8192: 21 us).
//
// y's columns may lie in groups apart (a latent prompt's keys and values beside a shared rotary key: the copy into place took 9.4 us for 2048 tokens of 16 heads).
// Tiles of 256 rows, the last one 33 to 288 (a few rows more are no tile of their own), or of 128; which, and whether at all, rows_form of exec/linear.py says.
#include "gelu_erf.h"
#include "wide_tiles.h"

namespace llmctl {
namespace {
using namespace wide;

struct RowsArgs {
  const unsigned short* a;
  const unsigned short* b;
  const unsigned short* bias;
  unsigned short* c;
  long lda, ldb;
  int M, N, K;
  int tiles_m, tiles_n;
  long ldc;
  int gw, gstep;  // y's columns lie in groups of gw (8s), gstep apart
  float* parts;   // [splits, M, N]: the sums of ranges of K
  int splits;
};
constexpr int BAND = 4;  // tile rows that walk the columns together

// ACT as in stream_linear.h (1 erf GELU, 2 tanh GELU), of the fp32 sum and the bias
template <int ACT>
__device__ __forceinline__ float act_of(float v) {
  if constexpr (ACT == 1) return gelu_erf(v);
  if constexpr (ACT == 2) return v / (1.0f + __expf(-1.5957691216057308f * (v + 0.044715f * v * v * v)));  // v sigmoid(2 z) = 0.5 v (1 + tanh z)
  return v;
}

// Where a row of y holds column c
__device__ __forceinline__ int col_at(const RowsArgs& g, int c) { return c + (g.gw < g.N ? c / g.gw : 0) * (g.gstep - g.gw); }

template <bool HALVES, int ACT, bool PARTS>
__global__ __launch_bounds__(NT4, 1) __attribute__((amdgpu_waves_per_eu(1, 1))) void gemm_rows_kernel(RowsArgs g) {
  __shared__ __attribute__((aligned(1024))) unsigned char smem[3 * SLOT];
  static_assert(4 * SLOT_H <= 3 * SLOT, "LDS");
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), wr = wave >> 1, wc = wave & 1;
  // a run of neighbouring tiles (of one range of K) to each XCD
  const int n = gridDim.x, q8 = n >> 3, r8 = n & 7, xcd = blockIdx.x & 7, item = xcd * q8 + min(xcd, r8) + ((int)blockIdx.x >> 3);
  const int sp = PARTS ? __builtin_amdgcn_readfirstlane(item / (g.tiles_m * g.tiles_n)) : 0, tile = item - sp * (g.tiles_m * g.tiles_n);
  const int k0 = PARTS ? __builtin_amdgcn_readfirstlane(sp * (g.K / 128) / g.splits * 128) : 0;
  const int K = PARTS ? __builtin_amdgcn_readfirstlane((sp + 1) * (g.K / 128) / g.splits * 128) - k0 : g.K;
  const int first = tile / (BAND * g.tiles_n) * BAND, in = tile - first * g.tiles_n, high = min(BAND, g.tiles_m - first);
  const int tn = in / high, tm = first + in - tn * high;
  const int row0 = tm * (HALVES ? 128 : 256), rows = HALVES ? min(128, g.M - row0) : tm == g.tiles_m - 1 ? g.M - row0 : 256, col0 = tn * COLS;
  // DMA offsets: piece i of an image holds its rows 32 i + tid / 8, chunk tid % 8 of a K-tile's eight at its swizzled place; rows past the end are the last one's
  unsigned va[9], vb[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int ir = 32 * i + (tid >> 3);
    vb[i] = (unsigned)min(ir, g.N - 1 - col0) * (unsigned)(g.ldb * 2) + (unsigned)(((tid & 7) ^ swr(ir)) << 4);
  }
  const Tile t{g.a + (long)row0 * g.lda + k0, g.b + (long)col0 * g.ldb + k0, K};
  first_b<HALVES ? 2 : 3>(t, vb, smem, HALVES ? SLOT_H : SLOT, HALVES ? HALF : B_H0 * HALF);
#pragma unroll
  for (int i = 0; i < 9; ++i) {
    const int ir = 32 * (i & 3) + (tid >> 3);
    const int r = i == 8 ? 256 + (tid >> 3) : HALVES ? ir : i < 4 ? tile_pos<A_LO>(ir) : tile_pos<A_HI>(ir);
    va[i] = (unsigned)min(r, rows - 1) * (unsigned)(g.lda * 2) + (unsigned)(((tid & 7) ^ swr(i == 8 ? tid >> 3 : ir)) << 4);
  }
  // lane holds [16 i + (l & 15)][16 j + 4 (l >> 4) + r] of its wave's part; 16 bytes to a lane: lanes of neighbouring groups swap halves of two column tiles
  const int kg = lane >> 4, i16 = lane & 15, c0 = col0 + wc * 64 + 16 * (kg & 1) + 8 * (kg >> 1);
  auto out = [&](auto mb_c) __attribute__((always_inline)) {
    constexpr int MB = decltype(mb_c)::value;
    f32x4_t acc[9][4];
    if constexpr (MB == 4) run_half(t, va, vb, smem, acc);
    else run<MB>(t, va, vb, smem, acc);
    if constexpr (PARTS) {
      float* out = g.parts + ((long)sp * g.M + row0) * g.N;
#pragma unroll
      for (int i = 0; i < MB; ++i) {
        const int r = i == 8 ? 256 + wr * 16 + i16 : wr * (HALVES ? 64 : 128) + 16 * i + i16;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int c = col0 + wc * 64 + 16 * j + 4 * kg;
          if (r < rows && c < g.N) *reinterpret_cast<f32x4_t*>(out + (long)r * g.N + c) = acc[i][j];
        }
      }
      return;
    }
    float bias[2][8];
    int at[2];  // where in a row of y the lane's columns are
#pragma unroll
    for (int jp = 0; jp < 2; ++jp) {
      at[jp] = col_at(g, c0 + 32 * jp);
#pragma unroll
      for (int e = 0; e < 8; ++e) bias[jp][e] = 0.f;
      if (g.bias != nullptr && c0 + 32 * jp < g.N) load8(g.bias + c0 + 32 * jp, bias[jp]);
    }
#pragma unroll
    for (int i = 0; i < MB; ++i) {
      const int r = i == 8 ? 256 + wr * 16 + i16 : wr * (HALVES ? 64 : 128) + 16 * i + i16;
#pragma unroll
      for (int jp = 0; jp < 2; ++jp) {
        float v[8];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const auto s = __builtin_amdgcn_permlane16_swap(__float_as_uint(acc[i][2 * jp][e]), __float_as_uint(acc[i][2 * jp + 1][e]), false, false);
          v[e] = __uint_as_float(s[0]);
          v[4 + e] = __uint_as_float(s[1]);
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = act_of<ACT>(v[e] + bias[jp][e]);
        if (r < rows && c0 + 32 * jp < g.N) store8(g.c + (long)(row0 + r) * g.ldc + at[jp], v);
      }
    }
  };
  if constexpr (HALVES) {
    out(K_<4>{});
  } else {
    if (rows <= 256) out(K_<8>{});
    else out(K_<9>{});
  }
}

// y = act(sum of the ranges (+ bias)): 8 outputs a thread, the loads of four ranges at once; at the copy rate out of L2 and the last-level cache.
template <int ACT>
__global__ __launch_bounds__(256) void gemm_rows_sum(RowsArgs g) {
  const unsigned i = blockIdx.x * 256 + threadIdx.x, per = (unsigned)g.N / 8;
  const unsigned r = i / per, c = (i - r * per) * 8;
  if (r >= (unsigned)g.M) return;
  const long step = (long)g.M * g.N;
  const float* p = g.parts + (long)r * g.N + c;
  float v[8] = {};
  if (g.bias != nullptr) load8(g.bias + c, v);
  f32x4_t lo = {0.f, 0.f, 0.f, 0.f}, hi = lo;
#pragma unroll 4
  for (int s = 0; s < g.splits; ++s) {
    lo += *reinterpret_cast<const f32x4_t*>(p + s * step);
    hi += *reinterpret_cast<const f32x4_t*>(p + s * step + 4);
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    v[e] = act_of<ACT>(lo[e] + v[e]);
    v[4 + e] = act_of<ACT>(hi[e] + v[4 + e]);
  }
  store8(g.c + (long)r * g.ldc + col_at(g, (int)c), v);
}

int row_tiles(int64_t M) { return M <= ROWS ? 1 : (int)((M - 33) / 256 + 1); }

// y [M, N], or [M, groups, N / groups] whose rows and groups may lie apart; undefined: made here
void rows_product(const at::Tensor& x, const at::Tensor& w, const c10::optional<at::Tensor>& bias, int64_t form, at::Tensor& y, int64_t splits, int64_t act) {
  LLMCTL_CHECK(x.dim() == 2 && w.dim() == 2 && x.is_cuda() && w.is_cuda() && x.scalar_type() == at::kBFloat16 && w.scalar_type() == at::kBFloat16 && x.stride(1) == 1 &&
                   w.stride(1) == 1,
               "gemm_rows: bf16 GPU x [M, K] and w [N, K] with unit inner strides");
  const int64_t M = x.size(0), K = x.size(1), N = w.size(0);
  LLMCTL_CHECK(w.size(1) == K && K % 128 == 0 && K >= 256 && N % 8 == 0 && (form == 1 || form == 2), "gemm_rows: K in 128s from 256 on, N in 8s, form 1 or 2");
  LLMCTL_CHECK(splits >= 1 && splits <= K / 256 && act >= 0 && act <= 2 && splits * M * N < (1L << 34) && M * N / 8 < (1L << 31) - 256,
               "gemm_rows: ranges of K of at least 256, activation 0 to 2");
  LLMCTL_CHECK(x.stride(0) % 8 == 0 && w.stride(0) % 8 == 0 && (reinterpret_cast<uintptr_t>(x.data_ptr()) & 15) == 0 && (reinterpret_cast<uintptr_t>(w.data_ptr()) & 15) == 0,
               "gemm_rows: 16-byte aligned rows");
  const bool has_bias = bias.has_value() && bias->defined();
  if (has_bias)
    LLMCTL_CHECK(bias->is_cuda() && bias->scalar_type() == at::kBFloat16 && bias->is_contiguous() && bias->numel() == N && (reinterpret_cast<uintptr_t>(bias->data_ptr()) & 15) == 0,
                 "gemm_rows: bias bf16 [N], aligned to 16 bytes");
  LLMCTL_CHECK(ROWS * x.stride(0) < (1L << 30) && COLS * w.stride(0) < (1L << 30) && x.stride(0) >= 0 && w.stride(0) >= 0 && M < (1L << 31) && N < (1L << 31),
               "gemm_rows: operand too large for 32-bit offsets");
  const bool into = y.defined();
  if (into)
    LLMCTL_CHECK(y.is_cuda() && y.scalar_type() == at::kBFloat16 && y.dim() == 3 && y.size(0) == M && y.size(1) * y.size(2) == N && y.size(2) % 8 == 0 &&
                     (y.size(2) <= 1 || y.stride(2) == 1) && y.stride(0) % 8 == 0 && y.stride(1) % 8 == 0 && y.stride(1) >= y.size(2) &&
                     y.stride(0) >= y.size(1) * y.stride(1) - (y.stride(1) - y.size(2)) && y.size(1) * y.stride(1) < (1L << 31) &&
                     (reinterpret_cast<uintptr_t>(y.data_ptr()) & 15) == 0,
                 "gemm_rows: out bf16 [M, groups, N / groups], rows and groups apart, in 8s");
  const c10::DeviceGuard guard(x.device());
  if (!into) y = at::empty({M, N}, x.options());
  if (M == 0 || N == 0) return;
  RowsArgs g{bf_ptr(x), bf_ptr(w), has_bias ? bf_ptr(*bias) : nullptr, reinterpret_cast<unsigned short*>(y.data_ptr()), (long)x.stride(0), (long)w.stride(0),
             (int)M, (int)N, (int)K, form == 1 ? row_tiles(M) : (int)((M + 127) / 128), (int)((N + COLS - 1) / COLS), into ? (long)y.stride(0) : (long)N,
             into ? (int)y.size(2) : (int)N, into ? (int)y.stride(1) : (int)N, nullptr, (int)splits};
  const dim3 grid((unsigned)(g.tiles_m * g.tiles_n * splits));
  auto go = [&](auto act_c) {
    constexpr int ACT = decltype(act_c)::value;
    if (splits > 1) gemm_rows_sum<ACT><<<dim3((unsigned)((M * N / 8 + 255) / 256)), 256, 0, stream()>>>(g);
    else if (form == 1) gemm_rows_kernel<false, ACT, false><<<grid, NT4, 0, stream()>>>(g);
    else gemm_rows_kernel<true, ACT, false><<<grid, NT4, 0, stream()>>>(g);
  };
  at::Tensor parts;
  if (splits > 1) {
    parts = at::empty({splits, M, N}, x.options().dtype(at::kFloat));
    g.parts = parts.data_ptr<float>();
    if (form == 1) gemm_rows_kernel<false, 0, true><<<grid, NT4, 0, stream()>>>(g);
    else gemm_rows_kernel<true, 0, true><<<grid, NT4, 0, stream()>>>(g);
  }
  switch (act) {
    case 0: go(K_<0>{}); break;
    case 1: go(K_<1>{}); break;
    default: go(K_<2>{}); break;
  }
}
}  // namespace

// act(x w^T (+ bias)); form: 1 = tiles of 256 rows, 2 = of 128; splits: ranges of K; act as in stream_linear.h
at::Tensor gemm_rows(const at::Tensor& x, const at::Tensor& w, const c10::optional<at::Tensor>& bias, int64_t form, int64_t splits, int64_t act) {
  at::Tensor y;
  rows_product(x, w, bias, form, y, splits, act);
  return y;
}
void gemm_rows_into(const at::Tensor& x, const at::Tensor& w, const c10::optional<at::Tensor>& bias, int64_t form, at::Tensor out, int64_t splits) {
  rows_product(x, w, bias, form, out, splits, 0);
}

TORCH_LIBRARY_IMPL(llmctl, CUDA, m) {
  m.impl("gemm_rows", &gemm_rows);
  m.impl("gemm_rows_into", &gemm_rows_into);
}

}  // namespace llmctl
