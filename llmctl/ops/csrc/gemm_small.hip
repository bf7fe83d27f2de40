// Products of few entries for training steps of a few hundred tokens: out[M, N] (+)= A B, bf16 in, fp32 sums, bf16 or fp32 out, in one launch.
//
// Bound: latency.  The operands (some 100 KB to 10 MB) lie in L2 or near it; what counts is that enough CUs ask for them at once and that a product is one
// launch.  Tiles of 128 and 256 rows leave 1 to 8 workgroups here, and a partial-sum pass behind them where they are cut in K.
//
// Split: a workgroup owns 16 F x 16 F outputs, its NW waves a part of K each, added up through LDS at the end (in the order of the waves, whatever the tile).
// Four waves where rows run along K; eight shorten the chain through the panels (weight gradients 768 x 256 of 1024 tokens 7.6 / 6.5 us, data gradients
// from K 1024 on 256 x 256 x 1408 8.6 / 8.0); sixteen gain nothing.
// A wave asks for U steps of 32 at once: fragments of an operand whose rows run along K come straight from memory, 16 bytes a lane; one that is stored along the
// other axis ([K, rows]: W of a data gradient, both operands of a weight gradient) goes through the wave's own LDS panel in 16-byte pieces and is read back by
// ds_read_b64_tr_b16.  No barrier before the end.  A panel's 32-byte segments are permuted by the row of K so that a half wave's eight of them hit eight different
// sets of banks.
// Measured on one MI355X in a graph, us, the library or the 256-row tiles / here: 256 tokens, forward 256 x 256 12.0 / 4.0, 256 x 704 17.6 / 6.1, 768 x 256 4.6 / 4.0;
// data gradients 768 x 256 12.6 / 6.4, 256 x 256 7.9 / 4.1, 1408 x 256 12.8 / 8.0; weight gradients 256 x 256 8.1 / 4.1, 768 x 256 8.3 / 4.8, 768 x 768 8.8 / 6.1.
// The error against 64 bits is that of the output's rounding, as before.
#include "common.h"
#include "attn_common.h"
#include "stream_linear.h"

namespace llmctl {
using namespace attn;
namespace {

using f32x4_t = __attribute__((ext_vector_type(4))) float;

struct SmallGemm {
  const unsigned short* a;     // [M, K], or [K, M] where TA
  const unsigned short* b;     // [N, K], or [K, N] where TB
  void* c;                     // [M, N]
  const unsigned short* bias;  // not TA: nullptr or [N], added to every row
  void* sums;                  // TA: nullptr or [M] (+)= the sums of A over K, of c's type
  long lda, ldb, ldc;
  int M, N, K, f32, add, add_sums, tiles_n, act, tile;  // act (not TA): as in stream_linear.h, of the sum and the bias
};

__device__ __forceinline__ uint4 zero_or(const unsigned short* p, bool in) {
  uint4 v = make_uint4(0, 0, 0, 0);
  if (in) v = *reinterpret_cast<const uint4*>(p);
  return v;
}

// 32-byte segment ``seg`` of row k of a panel of F segments a row
template <int F>
__device__ __forceinline__ int panel_off(int k, int seg) {
  const int turn = F == 2 ? (k >> 3) & 1 : ((k >> 1) & 1) | ((k >> 3) & 1) << 1;
  return k * 32 * F + ((seg ^ turn) << 5);
}

// One operand of a wave: R positions (rows of the tile) over the wave's steps.
template <bool T, int F, int U>
struct Operand {
  const unsigned short* p[F];
  long ld;
  int k[F];  // T: row of K of a piece within its step
  uint4 v[U][F];

  __device__ __forceinline__ void init(const unsigned short* base, long ld_, int p0, int R, int lane) {
    ld = ld_;
#pragma unroll
    for (int f = 0; f < F; ++f) {
      if constexpr (T) {
        const int i = f * 64 + lane;
        k[f] = i / (2 * F);
        p[f] = base + (long)k[f] * ld + min(p0 + (i % (2 * F)) * 8, R - 8);  // R is a multiple of 8: pieces past it repeat the last one and are not stored
      } else {
        k[f] = 8 * (lane >> 4);
        p[f] = base + (long)min(p0 + 16 * f + (lane & 15), R - 1) * ld + k[f];
      }
    }
  }
  __device__ __forceinline__ const unsigned short* at(int f, int s) const { return p[f] + (T ? (long)s * 32 * ld : (long)s * 32); }
  __device__ __forceinline__ void fetch(int s, int s1, int K, bool whole) {
    if (whole) {
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int f = 0; f < F; ++f) v[u][f] = *reinterpret_cast<const uint4*>(at(f, s + u));
    } else {
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int f = 0; f < F; ++f) v[u][f] = zero_or(at(f, s + u), s + u < s1 && (s + u) * 32 + k[f] < K);
    }
  }
  // T: into the wave's panels
  __device__ __forceinline__ void place(unsigned char* panel, int lane) {
    if constexpr (T) {
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int f = 0; f < F; ++f) {
          const int pc = (f * 64 + lane) % (2 * F);
          *reinterpret_cast<uint4*>(panel + u * 1024 * F + panel_off<F>(k[f], pc >> 1) + (pc & 1) * 16) = v[u][f];
        }
    }
  }
  __device__ __forceinline__ bf16x8_t frag(const unsigned char* panel, int u, int f, int lane) const {
    if constexpr (!T) {
      return __builtin_bit_cast(bf16x8_t, v[u][f]);
    } else {
      const int i16 = lane & 15, kr = 8 * (lane >> 4) + (i16 >> 2);
      const unsigned char* q = panel + u * 1024 * F + panel_off<F>(kr, f) + (i16 & 3) * 8;
      const s4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)q), hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(q + 4 * 32 * F));
      const s8_t w = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      return __builtin_bit_cast(bf16x8_t, w);
    }
  }
};

template <bool TA, bool TB, int F, int U, int NW>
struct Lds {
  static constexpr int PANEL = U * 1024 * F, PANELS = PANEL * ((TA ? 1 : 0) + (TB ? 1 : 0));  // bytes of a wave
  static constexpr int RED = NW * F * F * 64 * 16;
  static constexpr int BYTES = NW * PANELS > RED ? NW * PANELS : RED;
  static constexpr int ROWS = TA ? NW * 16 * F : 1;  // sums of A over K, by wave
};

// Tile ``tile`` of g; lds, rows: Lds's BYTES and ROWS
template <bool TA, bool TB, int F, int U, int NW>
__device__ __forceinline__ void workgroup(const SmallGemm& g, int tile, unsigned char* lds, float* rows) {
  constexpr int PANEL = Lds<TA, TB, F, U, NW>::PANEL, PANELS = Lds<TA, TB, F, U, NW>::PANELS;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int m0 = tile / g.tiles_n * 16 * F, n0 = tile % g.tiles_n * 16 * F;
  unsigned char* pa = lds + wave * PANELS;
  unsigned char* pb = pa + (TA ? PANEL : 0);
  Operand<TA, F, U> a;
  Operand<TB, F, U> b;
  a.init(g.a, g.lda, m0, g.M, lane);
  b.init(g.b, g.ldb, n0, g.N, lane);
  const bool sums = TA && g.sums != nullptr && n0 == 0;
  f32x4_t acc[F][F], rs[F];  // [n][m]
#pragma unroll
  for (int n = 0; n < F; ++n) {
    rs[n] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int m = 0; m < F; ++m) acc[n][m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }
  const s8_t one8 = {0x3f80, 0x3f80, 0x3f80, 0x3f80, 0x3f80, 0x3f80, 0x3f80, 0x3f80};
  const bf16x8_t ones = __builtin_bit_cast(bf16x8_t, one8);
  const int steps = (g.K + 31) / 32, per = (steps + NW - 1) / NW;
  const int s0 = wave * per, s1 = min(s0 + per, steps), full = min(s1, g.K / 32);
  for (int s = s0; s < s1; s += U) {
    const bool whole = s + U <= full;
    a.fetch(s, s1, g.K, whole);
    b.fetch(s, s1, g.K, whole);
    __builtin_amdgcn_sched_barrier(0);  // the whole batch in flight before the first use
    a.place(pa, lane);
    b.place(pb, lane);
    if constexpr (TA || TB) asm volatile("" ::: "memory");  // (a wave's LDS accesses keep their order; the lanes read what others wrote)
#pragma unroll
    for (int u = 0; u < U; ++u) {
      bf16x8_t fa[F], fb[F];
#pragma unroll
      for (int f = 0; f < F; ++f) fa[f] = a.frag(pa, u, f, lane), fb[f] = b.frag(pb, u, f, lane);
#pragma unroll
      for (int n = 0; n < F; ++n)
#pragma unroll
        for (int m = 0; m < F; ++m) acc[n][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[n], fa[m], acc[n][m], 0, 0, 0);
      if constexpr (TA) {
        if (sums) {
#pragma unroll
          for (int m = 0; m < F; ++m) rs[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, fa[m], rs[m], 0, 0, 0);
        }
      }
    }
    if constexpr (TA || TB) asm volatile("" ::: "memory");
  }
  __syncthreads();  // the panels are read
  f32x4_t* red = reinterpret_cast<f32x4_t*>(lds);  // [wave][n][m][lane]
#pragma unroll
  for (int n = 0; n < F; ++n)
#pragma unroll
    for (int m = 0; m < F; ++m) red[((wave * F + n) * F + m) * 64 + lane] = acc[n][m];
  if constexpr (TA) {
    if (sums && lane < 16) {
#pragma unroll
      for (int m = 0; m < F; ++m) rows[wave * 16 * F + 16 * m + lane] = rs[m][0];
    }
  }
  __syncthreads();
  for (int i = tid; i < F * F * 64; i += 64 * NW) {
    const int t = i >> 6, l = i & 63, row = m0 + 16 * (t % F) + (l & 15), col = n0 + 16 * (t / F) + 4 * (l >> 4);
    if (row >= g.M || col >= g.N) continue;  // (N is a multiple of 8)
    f32x4_t v = red[i];
#pragma unroll
    for (int w = 1; w < NW; ++w) v += red[w * F * F * 64 + i];
    if (!TA && g.bias != nullptr) {
      const uint2 x = *reinterpret_cast<const uint2*>(g.bias + col);
      v[0] += __uint_as_float(x.x << 16), v[1] += __uint_as_float(x.x & 0xffff0000u);
      v[2] += __uint_as_float(x.y << 16), v[3] += __uint_as_float(x.y & 0xffff0000u);
    }
    if (!TA && g.act != 0) {
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = stream_linear::activate(g.act, v[j]);
    }
    if (g.f32) {
      f32x4_t* o = reinterpret_cast<f32x4_t*>(static_cast<float*>(g.c) + (long)row * g.ldc + col);
      *o = g.add ? *o + v : v;
    } else {
      uint2* o = reinterpret_cast<uint2*>(static_cast<unsigned short*>(g.c) + (long)row * g.ldc + col);
      if (g.add) {
        const uint2 x = *o;
        v[0] += __uint_as_float(x.x << 16), v[1] += __uint_as_float(x.x & 0xffff0000u);
        v[2] += __uint_as_float(x.y << 16), v[3] += __uint_as_float(x.y & 0xffff0000u);
      }
      *o = make_uint2(f2bf(v[0]) | (unsigned)f2bf(v[1]) << 16, f2bf(v[2]) | (unsigned)f2bf(v[3]) << 16);
    }
  }
  if constexpr (TA) {
    if (sums && tid < 16 * F && m0 + tid < g.M) {
      float v = rows[tid];
#pragma unroll
      for (int w = 1; w < NW; ++w) v += rows[w * 16 * F + tid];
      if (g.f32) {
        float* o = static_cast<float*>(g.sums) + m0 + tid;
        *o = g.add_sums ? *o + v : v;
      } else {
        unsigned short* o = static_cast<unsigned short*>(g.sums) + m0 + tid;
        *o = f2bf(g.add_sums ? __uint_as_float((unsigned)*o << 16) + v : v);
      }
    }
  }
}

template <bool TA, bool TB, int F, int U, int NW>
__global__ __launch_bounds__(64 * NW) void gemm_small_kernel(SmallGemm g) {
  using L = Lds<TA, TB, F, U, NW>;
  __shared__ __attribute__((aligned(16))) unsigned char lds[L::BYTES];
  __shared__ float rows[L::ROWS];
  workgroup<TA, TB, F, U, NW>(g, (int)blockIdx.x, lds, rows);
}

// A layer's data gradient d and its weight gradient g in one launch: they read the same dY and wait for nothing of one another.  The one with the longer
// sums first (its workgroups: the first ``first``).  Nine such pairs in a step of the tiny model at 256 tokens: 306 us, so 279.
__global__ __launch_bounds__(512) void gemm_small_back_kernel(SmallGemm d, SmallGemm g, int first, int d_first) {
  using D = Lds<false, true, 2, 4, 8>;
  using W = Lds<true, true, 2, 2, 8>;
  __shared__ __attribute__((aligned(16))) unsigned char lds[D::BYTES > W::BYTES ? D::BYTES : W::BYTES];
  __shared__ float rows[W::ROWS];
  const int i = (int)blockIdx.x, rest = i - first;
  if ((i < first) == (d_first != 0)) workgroup<false, true, 2, 4, 8>(d, i < first ? i : rest, lds, rows);
  else workgroup<true, true, 2, 2, 8>(g, i < first ? i : rest, lds, rows);
}

}  // namespace

namespace {
// The operands of one product, checked; ``act`` and the layouts as of gemm_small
SmallGemm operands(const at::Tensor& a, const at::Tensor& b, const at::Tensor& out, bool at_, bool bt, bool accumulate, const c10::optional<at::Tensor>& bias,
                const c10::optional<at::Tensor>& sums, bool add_sums, int64_t act) {
  LLMCTL_CHECK(a.dim() == 2 && b.dim() == 2 && out.dim() == 2 && a.is_cuda() && b.is_cuda() && out.is_cuda(), "gemm_small: 2-D GPU operands");
  const bool f32 = out.scalar_type() == at::kFloat;
  LLMCTL_CHECK(a.scalar_type() == at::kBFloat16 && b.scalar_type() == at::kBFloat16 && (f32 || out.scalar_type() == at::kBFloat16),
               "gemm_small: bf16 operands, bf16 or fp32 out");
  LLMCTL_CHECK((!at_ || bt) && act >= 0 && act <= 3 && (act == 0 || (!at_ && !accumulate)),
               "gemm_small: a transposed A goes with a transposed B, an activation (0 .. 3) with neither of A transposed and a sum");
  const long M = at_ ? a.size(1) : a.size(0), K = at_ ? a.size(0) : a.size(1), N = bt ? b.size(1) : b.size(0);
  LLMCTL_CHECK((bt ? b.size(0) : b.size(1)) == K && out.size(0) == M && out.size(1) == N, "gemm_small: shapes");
  LLMCTL_CHECK(N % 8 == 0 && (!at_ || M % 8 == 0) && (at_ || K % 8 == 0) && M < (1l << 24) && N < (1l << 24) && K < (1l << 24), "gemm_small: sizes in 8s");
  auto rows16 = [](const at::Tensor& t, int per) {
    return t.stride(1) == 1 && t.stride(0) % per == 0 && t.stride(0) >= t.size(1) && (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0;
  };
  LLMCTL_CHECK(rows16(a, 8) && rows16(b, 8) && rows16(out, f32 ? 4 : 8), "gemm_small: 16-byte aligned rows, unit column stride");
  if (bias.has_value())
    LLMCTL_CHECK(!at_ && bias->is_cuda() && bias->scalar_type() == at::kBFloat16 && bias->is_contiguous() && bias->numel() == N &&
                     (reinterpret_cast<uintptr_t>(bias->data_ptr()) & 7) == 0,
                 "gemm_small: bias bf16 [N]");
  if (sums.has_value())
    LLMCTL_CHECK(at_ && sums->is_cuda() && sums->scalar_type() == out.scalar_type() && sums->is_contiguous() && sums->numel() == M, "gemm_small: sums [M] of out's type");
  // Tiles of 32; where they are many, tiles of 64 read the operands half as often (weight gradients of 64 tokens 768 x 768 5.6 / 5.2 us, 2304 x 768 11.3 / 9.4, 512 x
  // 256 3.8 / 5.1; forward 640 tokens 2304 x 768 20.1 / 15.4, 768 x 768 8.8 / 9.7)
  const long tile = (at_ || !bt) && (M + 31) / 32 * ((N + 31) / 32) > 512 ? 64 : 32;
  const int tiles_n = (int)((N + tile - 1) / tile);
  LLMCTL_CHECK((M + tile - 1) / tile * tiles_n < (1l << 30), "gemm_small: too many tiles");
  auto ptr = [](const at::Tensor& t) { return reinterpret_cast<const unsigned short*>(t.data_ptr()); };
  return SmallGemm{ptr(a), ptr(b), out.data_ptr(), bias.has_value() ? ptr(*bias) : nullptr, sums.has_value() ? sums->data_ptr() : nullptr,
                   (long)a.stride(0), (long)b.stride(0), (long)out.stride(0), (int)M, (int)N, (int)K, f32, accumulate, add_sums, tiles_n, (int)act, (int)tile};
}
unsigned tiles_of(const SmallGemm& g) { return (unsigned)((g.M + g.tile - 1) / g.tile * g.tiles_n); }
}  // namespace

// out [M, N] (+)= act(A B^T + bias) (A [M, K], B [N, K]), A B (bt: B [K, N]) or A^T B (at and bt: A [K, M]); out bf16 or fp32.  N a multiple of 8, M where at, K where an operand
// runs along it; aligned rows.  bias bf16 [N] (not at); sums [M] (+)= the sums of A over K (at), of out's type.
void gemm_small(const at::Tensor& a, const at::Tensor& b, at::Tensor out, bool at_, bool bt, bool accumulate, const c10::optional<at::Tensor>& bias,
                const c10::optional<at::Tensor>& sums, bool add_sums, int64_t act) {
  const SmallGemm g = operands(a, b, out, at_, bt, accumulate, bias, sums, add_sums, act);
  if (g.M == 0 || g.N == 0) return;
  c10::DeviceGuard guard(a.device());
  const dim3 grid(tiles_of(g));
  const hipStream_t st = stream();
  if (at_) {
    if (g.tile == 64) gemm_small_kernel<true, true, 4, 2, 4><<<grid, 256, 0, st>>>(g);
    else gemm_small_kernel<true, true, 2, 2, 8><<<grid, 512, 0, st>>>(g);
  } else if (bt) {
    if (g.K >= 1024) gemm_small_kernel<false, true, 2, 4, 8><<<grid, 512, 0, st>>>(g);
    else gemm_small_kernel<false, true, 2, 4, 4><<<grid, 256, 0, st>>>(g);
  } else {
    if (g.tile == 64) gemm_small_kernel<false, false, 4, 2, 4><<<grid, 256, 0, st>>>(g);
    else gemm_small_kernel<false, false, 2, 4, 4><<<grid, 256, 0, st>>>(g);
  }
}

// dx = dy w and g (+)= dy^T x (sums (+)= dy's sums over the rows) of dy [T, O], w [O, I], x [T, I]: gemm_small's products in one launch
void gemm_small_back(const at::Tensor& dy, const at::Tensor& w, at::Tensor dx, const at::Tensor& x, at::Tensor g, bool accumulate,
                     const c10::optional<at::Tensor>& sums, bool add_sums) {
  const SmallGemm d = operands(dy, w, dx, false, true, false, c10::nullopt, c10::nullopt, false, 0);
  const SmallGemm v = operands(dy, x, g, true, true, accumulate, c10::nullopt, sums, add_sums, 0);
  LLMCTL_CHECK(v.tile == 32 && d.tile == 32 && d.M > 0 && d.N > 0 && v.M > 0 && v.N > 0, "gemm_small_back: tiles of 32 (at most 512 of the weight gradient)");
  c10::DeviceGuard guard(dy.device());
  const bool d_first = d.K >= v.K;
  const unsigned nd = tiles_of(d), nv = tiles_of(v);
  gemm_small_back_kernel<<<dim3(nd + nv), 512, 0, stream()>>>(d, v, (int)(d_first ? nd : nv), d_first);
}

TORCH_LIBRARY_IMPL(llmctl, CUDA, m) { 
  m.impl("gemm_small", &gemm_small);
  m.impl("gemm_small_back", &gemm_small_back);
}

}  // namespace llmctl
