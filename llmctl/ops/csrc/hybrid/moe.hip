// Routed experts without a host round trip: router (fp32 scores and choice), token copies grouped by expert on the
// device, both expert projections of all experts as one grouped MFMA product each (the activation in the first one's
// epilogue), and the weighted sum per token.
//
// What it replaces bounded a layer by its launches and its host synchronisation: counts read back, a sort, one pair of
// GEMMs and one activation pass per expert, a concatenation, an fp32 copy and an atomic add per token copy.  Measured at
// the bottom of this comment, with the sizes.
//
//   * moe_route_kernel: 16 tokens per workgroup, logits on the fp32 matrix cores, scores and choice in the same kernel: no
//     logits tensor, no fp32 copy of the rows.  Steps of up to 64 tokens whose norm is at hand are routed there (router_rows.h).
//   * moe_group_kernel: one workgroup per expert counts the choices and places its own: a stable counting sort, and the list of row
//     tiles that the grouped product walks.
//   * moe_wide_kernel (moe_wide.h): tiles of up to 288 x 128, K in 128s from 256 on.
//   * moe_tile_kernel: BM x BN tiles of one expert's rows, K in 64-deep steps through LDS, the global loads of the next step
//     (64-wide tiles: the next three) in registers under the MFMAs of this one.  16-byte chunks are swizzled by the row, so a wave's fragment
//     reads touch every bank slot equally.  The weight fragment is the MFMA row operand: a lane ends up with four neighbouring
//     columns of one token.  Gate and up columns of the same place belong to the same wave, which makes the gated activation
//     lane-local.  Consecutive tiles go to one XCD, in bands of eight row tiles that walk the columns together.
//   * moe_small_kernel (steps of at most 64 tokens: decode): weight streaming.  A workgroup owns 16 output rows of one expert
//     (gate and up: 2 x 16), its four waves split K; it finds its rows by scanning the choices itself, so no grouping pass
//     runs.  Below two copies per expert, experts that no token chose are not read; from there on, where nearly every one has some, a wave
//     asks for its first steps (8, or 4 from 33 tokens on) before it knows.
//   * moe_combine_kernel: out_t = sum_k w_tk y_tk (+ w x_t for experts without weights) (+ the shared expert), fp32; where the
//     result goes straight into the residual stream and a norm, their kernel sums instead (expert_rows.h).
//
// Other widths, and sizes that moe_wide_pays leaves, have tiles of 128 x 128 (96
// rows an expert and more) or 64 x 64: with few tiles the K loop of every workgroup is a chain of load latencies.  The large tile
// keeps one LDS buffer (32 KB) so that three workgroups fit a CU; the small one keeps three steps in flight (37 -> 30 us at 65 tokens).
//
// Measured, one MI355X, width 2048, 8 gated experts of 1024, top 2 (up / down, kernel times; all caches written over before each layer):
//   tokens      16          32         64        128        256        512       1024       2048       4096
//   us       27 / 15     27 / 15    29 / 17    32 / 16    37 / 19    42 / 21    50 / 25    50 / 25    97 / 49
// up to 64 tokens the bound is the weight stream (67 + 34 MB: 2.5 TB/s), from there on what a CU can have in flight (moe_wide.h).  On tiles of 128 x 128, 512 tokens take
// 47 / 26, 1024 55 / 30, 2048 67 / 39, 4096 98 / 59.
#include "expert_rows.h"
#include "router_rows.h"
#include "stream_linear.h"

namespace llmctl_hybrid {
namespace {

using bfrag = __attribute__((ext_vector_type(8))) __bf16;
using facc = __attribute__((ext_vector_type(4))) float;

constexpr int MAX_EXPERTS = MAX_ROUTED;  // pointers travel as kernel arguments
constexpr int SMALL_ROWS = 64;    // tokens of a step that take the weight-streaming form

struct ExpertPtrs {
  const bf16_t* p[MAX_EXPERTS];
};

__device__ __forceinline__ facc mfma(bfrag a, bfrag b, facc c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }
__device__ __forceinline__ bfrag as_frag(uint4 v) { return __builtin_bit_cast(bfrag, v); }

// act 0: relu(u)^2, 1: silu(g) * u, 2: gelu(u) (erf)
__device__ __forceinline__ float expert_act(int act, float u, float g) {
  if (act == 1) return g / (1.0f + expf(-g)) * u;
  if (act == 0) {
    const float r = fmaxf(u, 0.f);
    return r * r;
  }
  return gelu_erf(u);
}

// The tiled form rounds the first projection's results to the activation's type before the activation, as a product and an
// activation pass give them: over thousands of tokens a later router then sees the same numbers as behind per-expert products, and
// the same choices where two experts are nearly equal (unrounded, one token in some 3000 chose otherwise).
__device__ __forceinline__ float bf16_of(float v) { return __bfloat162float(__float2bfloat16(v)); }

// (a conditional expression on two lvalues selects between addresses, one of them a stack slot)
__device__ __forceinline__ uint4 load_or_zero(const bf16_t* p, bool in) {
  uint4 v = make_uint4(0, 0, 0, 0);
  if (in) v = *reinterpret_cast<const uint4*>(p);
  return v;
}

__device__ __forceinline__ unsigned pack2(float a, float b) {
  return (unsigned)__bfloat16_as_ushort(__float2bfloat16(a)) | ((unsigned)__bfloat16_as_ushort(__float2bfloat16(b)) << 16);
}

// ------------------------------------------------------------------------------------------------ router
// 16 tokens per workgroup on the fp32 matrix cores (bf16 rows are exact in fp32): lane (r, kg) loads eight neighbouring k of
// token r and of router output r, and MFMA step j multiplies element j of every lane's eight, so four k that lie 8 apart.  The sixteen
// waves take every sixteenth 32-deep block of the row, four of their blocks in flight; then every wave chooses for one token, its
// scores two per lane.  (A vector-unit form, tokens times outputs per lane and a reduction over the wave, took 7 us for 16 rows but
// 22 us for 2048 and 43 us for 4096, where this one takes 10 and 12.)
constexpr int ROUTE_T = 16, ROUTE_WAVES = 16;
__global__ __launch_bounds__(ROUTE_WAVES * 64) void moe_route_kernel(const bf16_t* __restrict__ x, long ldx, const float* __restrict__ w,
                                                                     RouterChoice c, int* __restrict__ idx, float* __restrict__ wgt, int T, int W) {
  const int E = c.E;
  constexpr int U = 4;
  __shared__ facc part[ROUTE_WAVES][4][ROUTE_T];  // [wave][outputs 4 kg ..][token]
  __shared__ float logits[ROUTE_T][MAX_EXPERTS];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r = lane & 15, kg = lane >> 4;
  const int t0 = blockIdx.x * ROUTE_T;
  const bf16_t* xp = x + (long)min(t0 + r, T - 1) * ldx + kg * 8;
  const int blocks = (W + 31) / 32;
  for (int e0 = 0; e0 < E; e0 += 16) {
    const float* wp = w + (long)min(e0 + r, E - 1) * W + kg * 8;
    facc acc = facc{0.f, 0.f, 0.f, 0.f};
    for (int b0 = wave; b0 < blocks; b0 += ROUTE_WAVES * U) {
      uint4 xv[U];
      float4 wv[U][2];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int k = (b0 + u * ROUTE_WAVES) * 32;
        xv[u] = make_uint4(0, 0, 0, 0);
        wv[u][0] = wv[u][1] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (k + kg * 8 < W) {  // W is a multiple of 8
          xv[u] = *reinterpret_cast<const uint4*>(xp + k);
          wv[u][0] = *reinterpret_cast<const float4*>(wp + k);
          wv[u][1] = *reinterpret_cast<const float4*>(wp + k + 4);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const unsigned xw[4] = {xv[u].x, xv[u].y, xv[u].z, xv[u].w};
        const float wf[8] = {wv[u][0].x, wv[u][0].y, wv[u][0].z, wv[u][0].w, wv[u][1].x, wv[u][1].y, wv[u][1].z, wv[u][1].w};
#pragma unroll
        for (int j = 0; j < 8; ++j)
          acc = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[j], __uint_as_float(j & 1 ? xw[j >> 1] & 0xffff0000u : xw[j >> 1] << 16), acc, 0, 0, 0);
      }
    }
    part[wave][kg][r] = acc;
    __syncthreads();
    if (tid < 64) {
      facc s = part[0][kg][r];
#pragma unroll
      for (int v = 1; v < ROUTE_WAVES; ++v) s += part[v][kg][r];
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (e0 + 4 * kg + i < E) logits[r][e0 + 4 * kg + i] = s[i];
    }
    __syncthreads();
  }
  for (int t = wave; t < ROUTE_T && t0 + t < T; t += ROUTE_WAVES) {
    choose_experts(logits[t], lane, c, idx + (long)(t0 + t) * c.top, wgt + (long)(t0 + t) * c.top);
  }
}

// ------------------------------------------------------------------------------------------------ grouping
// Row tiles of n rows: of BM each, or (WIDE_ROWS, moe_wide.h) of 256 but the last one, which has 33 to 288.
constexpr int WIDE_ROWS = 288, WIDE_HALF = 128;
__host__ __device__ __forceinline__ int row_tiles(int n, int BM) { return BM != WIDE_ROWS ? (n + BM - 1) / BM : n <= BM ? n > 0 : (n - 33) / 256 + 1; }
__host__ __device__ __forceinline__ bool half_tile(int n, int BM) {  // the last one has at most 128 rows
  return BM == WIDE_ROWS && n > 0 && n - 256 * (row_tiles(n, BM) - 1) <= WIDE_HALF;
}

// Workgroup e: where expert e's copies start, which they are (in token order), and its row tiles.  ``tiles``: [0] = their
// number without the half ones, [1] = that of the half ones (WIDE_ROWS), then (expert, first sorted row, rows) each, the half ones last.  Entries of experts without
// weights (>= E) are left out.
// A thread takes `per` neighbouring copies, so that one pass over them and one scan over the workgroup place them all; a pass for the counts and rounds of 1024 with two
// barriers each took, us, so: 2048 tokens, 8 experts, top 2 6.5 / 4.7, 3565 9.6 / 5.5; 2031
// tokens, 32 experts, top 4 10.9 / 7.4; 16384 copies, 8 experts 18.0 / 13.8, 32768 34.0 / 29.6, 65536 63.8 / 65.3, 131072 127 / 136.  (In chunks of 16384, with copies beyond the first
// read twice as well: 20000 copies 13.3, so 25.2.)
constexpr int GROUP_KEEP = 16;  // copies a thread keeps in registers between the two passes
__global__ __launch_bounds__(1024) void moe_group_kernel(const int* __restrict__ idx, int N, int E, int BM, int* __restrict__ perm,
                                                         int* __restrict__ tiles) {
  __shared__ int hist[MAX_EXPERTS];
  __shared__ int wsum[16];
  __shared__ int base[2];
  const int e = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  if (tid < MAX_EXPERTS) hist[tid] = 0;
  const int per = (N + 1023) / 1024, i0 = tid * per, n_i = max(0, min(per, N - i0));
  int v[GROUP_KEEP], mine = 0;
#pragma unroll
  for (int k = 0; k < GROUP_KEEP; ++k) {
    v[k] = -1;
    if (k < per && k < n_i) v[k] = idx[i0 + k];
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < GROUP_KEEP; ++k) {
    if (k >= per) break;
    mine += v[k] == e;
    if (v[k] >= 0 && v[k] < E) atomicAdd(&hist[v[k]], 1);
  }
  for (int k = GROUP_KEEP; k < n_i; ++k) {
    const int x = idx[i0 + k];
    mine += x == e;
    if (x < E) atomicAdd(&hist[x], 1);
  }
  int before = 0, all = 0;  // copies of e ahead of this thread's, and in all, within the wave: bit by bit of their numbers
  for (int b = 0; per >> b != 0; ++b) {
    const unsigned long long m = __ballot(mine >> b & 1);
    before += __popcll(m & ((1ull << lane) - 1ull)) << b;
    all += __popcll(m) << b;
  }
  if (lane == 0) wsum[wave] = all;
  __syncthreads();
  if (wave == 0) {
    int at = 0, tile = 0, half = 0, whole = 0;  // before this expert: rows, tiles, half tiles; whole tiles of all
#pragma unroll
    for (int j = lane; j < MAX_EXPERTS; j += 64) {
      if (j >= E) continue;
      const int n = row_tiles(hist[j], BM), h = half_tile(hist[j], BM);
      whole += n - h;
      if (j < e) at += hist[j], tile += n - h, half += h;
    }
    for (int o = 32; o > 0; o >>= 1)
      if (E > o) at += __shfl_xor(at, o, 64), tile += __shfl_xor(tile, o, 64), half += __shfl_xor(half, o, 64), whole += __shfl_xor(whole, o, 64);
    at = __builtin_amdgcn_readfirstlane(at), tile = __builtin_amdgcn_readfirstlane(tile);
    half = __builtin_amdgcn_readfirstlane(half), whole = __builtin_amdgcn_readfirstlane(whole);
    const int n = hist[e], nt = row_tiles(n, BM), h = half_tile(n, BM), step = BM == WIDE_ROWS ? 256 : BM;
    for (int k = lane; k < nt; k += 64) {
      int* d = tiles + 2 + 3 * (h && k == nt - 1 ? whole + half : tile + k);
      d[0] = e;
      d[1] = at + k * step;
      d[2] = k < nt - 1 ? step : n - k * step;
    }
    if (lane == 0) {
      if (e == E - 1) tiles[0] = whole, tiles[1] = half + h;
      base[0] = at;
    }
  }
  __syncthreads();
  int at = base[0] + before;
#pragma unroll
  for (int w = 0; w < 16; ++w) at += w < wave ? wsum[w] : 0;
#pragma unroll
  for (int k = 0; k < GROUP_KEEP; ++k) {
    if (k >= per) break;
    if (v[k] == e) perm[at++] = i0 + k;
  }
  for (int k = GROUP_KEEP; k < n_i; ++k)
    if (idx[i0 + k] == e) perm[at++] = i0 + k;
}

// ------------------------------------------------------------------------------------------------ tiles
enum { UP_GLU = 0, UP_PLAIN = 1, DOWN = 2, UP_GELU = 3 };  // UP_GELU: moe_wide.h
// Row tiles that walk the columns together: an XCD's neighbouring workgroups then share weights as well as rows.  One at a time, every row tile read its
// expert's weights from the memory side again.  Whole layer, us, one / eight at a time (2, 4, 16 and 32 lie between): 8 gated experts of 4096 x 8192, top 2,
// 2048 tokens 1476 / 1136, 16384 tokens 11072 / 7517; 2048 x 4096 at 2048 340 / 325, 16384 2138 / 1979; 2048 x 1024 at 2048 118 / 119.
constexpr int BAND = 8;

struct TileArgs {
  const bf16_t* a;  // UP: the step's rows [T, K]; DOWN: the activations by sorted row [N, K]
  long lda;
  ExpertPtrs w;
  long ldw;
  bf16_t* out;  // UP: activations by sorted row [N, cols]; DOWN: [N entries, cols]
  const int* perm;
  const int* tiles;
  int K, cols, top, act, ntile;  // cols: ff (UP) or width (DOWN); ntile: column tiles
  int max_tiles;                 // of rows (room in tiles)
};

template <int BM, int BN, int MODE, int PF, int NB, int OCC>
__global__ __launch_bounds__(256, OCC) void moe_tile_kernel(TileArgs g) {
  constexpr int BK = 64;
  constexpr int AR = BM / 32, BR = BN / 32;      // rows of each operand that a thread stages (16 B each)
  constexpr int MI = BM / 32, NI = BN / 32;      // 16 x 16 tiles of a wave: BM/2 x BN/2
  constexpr int IMG = (BM + BN) * BK;            // elements of one buffer
  __shared__ __attribute__((aligned(16))) bf16_t lds[NB * IMG];
  // real tiles, spread so that neighbours in the list stay on one XCD (blocks go round-robin over the 8 XCDs)
  const int real = g.tiles[0] * g.ntile;
  const int id = blockIdx.x;
  if (id >= real) return;
  const int q8 = real >> 3, r8 = real & 7, xcd = id & 7;
  const int tile = xcd * q8 + min(xcd, r8) + (id >> 3);
  const int first = tile / (BAND * g.ntile) * BAND, in = tile - first * g.ntile, high = min(BAND, g.tiles[0] - first);
  const int nt = in / high, mt = first + in - nt * high;
  const int e = g.tiles[2 + 3 * mt], row0 = g.tiles[3 + 3 * mt], rows = g.tiles[4 + 3 * mt];
  const bf16_t* __restrict__ w = g.w.p[e];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave & 1, wn = wave >> 1;
  const int chunk = tid & 7, srow = tid >> 3;  // staging: 8 chunks of 16 B per 64-deep row, 32 rows per pass
  constexpr int CT = MODE == UP_GLU ? BN / 2 : BN;  // output columns of a tile
  const int c0 = nt * CT;
  const bf16_t* ap[AR];
  const bf16_t* bp[BR];
#pragma unroll
  for (int i = 0; i < AR; ++i) {
    const int p = row0 + min(srow + 32 * i, rows - 1);
    const long r = MODE == DOWN ? (long)p : (long)(g.perm[p] / g.top);
    ap[i] = g.a + r * g.lda + chunk * 8;
  }
#pragma unroll
  for (int i = 0; i < BR; ++i) {
    const int r = srow + 32 * i;
    long wr;
    if constexpr (MODE == UP_GLU) {
      // wave column wn holds BN/4 gate rows, then the up rows of the same places
      const int h = BN / 4, wc = r / (2 * h), half = (r / h) & 1, j = r % h;
      wr = (long)half * g.cols + min(c0 + wc * h + j, g.cols - 1);
    } else {
      wr = min(c0 + r, g.cols - 1);
    }
    bp[i] = w + wr * g.ldw + chunk * 8;
  }
  uint4 ra[PF][AR], rb[PF][BR];
  auto fetch = [&](int k0, uint4 (&a)[AR], uint4 (&b)[BR]) {
    if (k0 + BK <= g.K) {
#pragma unroll
      for (int i = 0; i < AR; ++i) a[i] = *reinterpret_cast<const uint4*>(ap[i] + k0);
#pragma unroll
      for (int i = 0; i < BR; ++i) b[i] = *reinterpret_cast<const uint4*>(bp[i] + k0);
    } else {  // the last step of a K that is no multiple of 64 (it is one of 8): zeros past the end
#pragma unroll
      for (int i = 0; i < AR; ++i) a[i] = load_or_zero(ap[i] + k0, k0 + chunk * 8 < g.K);
#pragma unroll
      for (int i = 0; i < BR; ++i) b[i] = load_or_zero(bp[i] + k0, k0 + chunk * 8 < g.K);
    }
  };
  facc acc[MI][NI];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j) acc[i][j] = facc{0.f, 0.f, 0.f, 0.f};
  const int r16 = lane & 15, kg = lane >> 4;
  const int steps = (g.K + BK - 1) / BK;
#pragma unroll
  for (int u = 0; u < PF; ++u)
    if (u < steps) fetch(u * BK, ra[u], rb[u]);
  for (int sb = 0; sb < steps; sb += PF) {
#pragma unroll
    for (int u = 0; u < PF; ++u) {
      const int s = sb + u;
      if (s >= steps) break;
      bf16_t* A = lds + (NB == 2 ? (s & 1) * IMG : 0);
      bf16_t* B = A + BM * BK;
      {
        const int sw = (chunk ^ (srow & 7)) * 8;
#pragma unroll
        for (int i = 0; i < AR; ++i) *reinterpret_cast<uint4*>(A + (srow + 32 * i) * BK + sw) = ra[u][i];
#pragma unroll
        for (int i = 0; i < BR; ++i) *reinterpret_cast<uint4*>(B + (srow + 32 * i) * BK + sw) = rb[u][i];
      }
      __syncthreads();
      if (s + PF < steps) fetch((s + PF) * BK, ra[u], rb[u]);
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        const int sw = ((kk * 4 + kg) ^ (r16 & 7)) * 8;
        bfrag fa[MI], fb[NI];
#pragma unroll
        for (int i = 0; i < MI; ++i) fa[i] = as_frag(*reinterpret_cast<const uint4*>(A + (wm * (BM / 2) + i * 16 + r16) * BK + sw));
#pragma unroll
        for (int j = 0; j < NI; ++j) fb[j] = as_frag(*reinterpret_cast<const uint4*>(B + (wn * (BN / 2) + j * 16 + r16) * BK + sw));
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
          for (int j = 0; j < NI; ++j) acc[i][j] = mfma(fb[j], fa[i], acc[i][j]);
      }
      if (NB == 1) __syncthreads();  // with two buffers the next step's barrier is enough: it lies after this step's reads
    }
  }
  // lane: token row wm*BM/2 + 16 i + r16, columns 16 j + 4 kg .. + 3 of the wave's half
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    const int r = wm * (BM / 2) + i * 16 + r16;
    if (r >= rows) continue;
    const long orow = MODE == DOWN ? (long)g.perm[row0 + r] : (long)(row0 + r);
    bf16_t* o = g.out + orow * g.cols;
    if constexpr (MODE == UP_GLU) {
#pragma unroll
      for (int j = 0; j < NI / 2; ++j) {
        const int c = c0 + wn * (BN / 4) + j * 16 + kg * 4;
        if (c >= g.cols) continue;
        float v[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) v[t] = expert_act(1, bf16_of(acc[i][j + NI / 2][t]), bf16_of(acc[i][j][t]));
        *reinterpret_cast<uint2*>(o + c) = make_uint2(pack2(v[0], v[1]), pack2(v[2], v[3]));
      }
    } else {
#pragma unroll
      for (int j = 0; j < NI; ++j) {
        const int c = c0 + wn * (BN / 2) + j * 16 + kg * 4;
        if (c >= g.cols) continue;
        float v[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) v[t] = MODE == DOWN ? acc[i][j][t] : expert_act(g.act, bf16_of(acc[i][j][t]), 0.f);
        *reinterpret_cast<uint2*>(o + c) = make_uint2(pack2(v[0], v[1]), pack2(v[2], v[3]));
      }
    }
  }
}

}  // namespace
}  // namespace llmctl_hybrid
#include "moe_wide.h"
namespace llmctl_hybrid {
// Whether N copies for E experts run on tiles of up to 288 x 128 (moe_wide.h) rather than on tiles of 128 x 128 or, below 96 rows an expert, 64 x 64: both products' rounds, in
// units of a K-step of 64 of a round of 128 x 128 tiles (three to a CU; the fuller the chip is, the longer: 0.32).  The experts' rows are taken as random choices spread them.
// A round of 256 full tiles counts 0.42 a K-step and 3.3, one of half tiles, behind them, 0.24 and 2.8, gates 7.3 more (half of it in a half tile); 64 x 64 tiles 1.04 a K-step, four to a CU and no whole
// rounds.  The constants are fitted to the comparison, not to the times, at 1803 sizes (66 to 4096 tokens, widths 512 to 4096, 4 to 64 experts of 256 to 2048, top 1 to 6:
// profiles/expert_tiles.txt); fitted to one half of them they do as well on the other.  876 are taken, in 12 % less time; of all 24 are more than 5 % slower than the better choice, and
// together they take 0.2 % more than with it (1650 tokens of width 1024, 8 experts of 1024 with GELUs, top 6 103 / 114 us).  By rows per expert alone 99 were, 2612 tokens of width 1024, 32 gated experts of 512,
// top 4 86 / 94, 377 of width 2048, 8 of 256 40 / 51.
bool moe_wide_pays(int64_t N, int64_t E, int64_t W, int64_t ff, bool glu) {
  if (E < 1 || N < 48 * E || N > INT32_MAX || W % 128 != 0 || ff % 128 != 0 || W < 256 || ff < 256) return false;
  const int B = N >= 96 * E ? 128 : 64;
  const double mean = (double)N / E, dev = std::sqrt(mean * (1.0 - 1.0 / E));
  double full = 0.0, half = 0.0, other = 0.0;  // row tiles
  for (const auto& [z, p] : {std::pair{-1.22, 0.3}, {0.0, 0.4}, {1.22, 0.3}}) {
    const int n = (int)std::nearbyint(mean + z * dev), h = half_tile(n, WIDE_ROWS);
    full += E * p * (row_tiles(n, WIDE_ROWS) - h), half += E * p * h, other += E * p * row_tiles(std::max(n, 1), B);
  }
  double wide = 0.0, narrow = 0.0;
  for (const bool down : {false, true}) {
    const int64_t cols = down ? W : glu ? 2 * ff : ff, K = down ? ff : W;
    const double gates = glu && !down ? 7.3 : 0.0, steps = (double)K / 64, nt = (double)cols / 128, cf = 0.42 * steps + 3.3 + gates, ch = 0.24 * steps + 2.8 + gates / 2;
    const double span = std::ceil(full * nt / 256 - 0.04) * cf, left = half * nt * ch / 256 - 0.85 * std::max(0.0, span - full * nt * cf / 256);
    wide += span + (left > 0.0 ? std::ceil(left / ch - 0.04) * ch : 0.0);
    const double items = other * std::ceil((double)cols / B);
    narrow += steps * (B == 128 ? std::max(1.0, std::ceil(items / 768 - 0.1)) + 0.32 * items / 768 : 1.04 * items / 1024);
  }
  return wide < narrow;
}

namespace {
static_assert(WIDE_ROWS == llmctl::wide::ROWS, "row tiles");

// ------------------------------------------------------------------------------------------------ few tokens
struct SmallArgs {
  const bf16_t* a;  // UP: the step's rows [T, K]; DOWN: activations by entry [N, K]
  long lda;
  ExpertPtrs w;
  long ldw;
  void* out;  // UP: bf16 [N, cols]; DOWN: fp32 [N, cols]
  const int* idx;
  int N, K, cols, top, act, E;
  stream_linear::Args side;  // SIDE: the shared expert's product of the same rows, its workgroups behind the experts' in blockIdx.y
  int side_groups;
};

// SIDE: a shared expert's projection of the step's rows (form <1, MT, 4, 8> of stream_linear.h, so the bits are those of a launch of its own) rides along: it is
// as long as its launch and one round trip, and the experts' workgroups leave bandwidth over.  16 rows of width 2048, 8 experts of 1024 and a shared one of 1024: the
// four launches 6.9 + 4.6 + 9.8 + 10.6 us a layer, the two 13.4 + 12.4; a step of three layers 299 us, so 282.
template <int MT, int MODE, bool SIDE>
__global__ __launch_bounds__(256) void moe_small_kernel(SmallArgs g) {
  constexpr int NM = MODE == UP_GLU ? 2 : 1;
  constexpr int U = MT >= 4 ? 4 : 8;  // K steps in flight (16 took 27 + 18 us where 8 took 26 + 14)
  __shared__ int list[SMALL_ROWS];
  __shared__ int count;
  __shared__ facc red[4][MT * NM][64];
  if constexpr (SIDE) {
    if ((int)blockIdx.y >= g.E) {
      const int i = ((int)blockIdx.y - g.E) * (int)gridDim.x + (int)blockIdx.x;
      if (i < g.side_groups) stream_linear::workgroup<1, MT, 4, 8>(g.side, (unsigned)i, 0, reinterpret_cast<stream_linear::acc_t(*)[MT][64]>(red));
      return;
    }
  }
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int e = blockIdx.y, n0 = blockIdx.x * 16;
  const int r = lane & 15, kg = lane >> 4;
  const bf16_t* wp[NM];
  wp[0] = g.w.p[e] + (long)min(n0 + r, g.cols - 1) * g.ldw + 8 * kg;
  if constexpr (NM == 2) wp[1] = wp[0] + (long)g.cols * g.ldw;
  const int steps = (g.K + 31) / 32;
  const int per = (steps + 3) / 4;
  const int s0 = wave * per, s1 = min(s0 + per, steps);
  const int whole = min(s1, g.K / 32);  // steps without a tail
  uint4 wv[U][NM];
  auto fetch_w = [&](int s) {
    if (s + U <= whole) {
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int n = 0; n < NM; ++n) wv[u][n] = *reinterpret_cast<const uint4*>(wp[n] + (s + u) * 32);
    } else {
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int n = 0; n < NM; ++n) wv[u][n] = load_or_zero(wp[n] + (s + u) * 32, s + u < s1 && (s + u) * 32 + 8 * kg < g.K);
    }
  };
  // with two copies per expert or more nearly every expert runs: its first weights are on their way while the rows are found
  const bool early = g.N >= 2 * g.E;
  if (early) fetch_w(s0);
  if (wave == 0) {
    int c = 0;
    for (int i0 = 0; i0 < g.N; i0 += 64) {
      const int i = i0 + lane;
      const bool mine = i < g.N && g.idx[i] == e;
      const unsigned long long m = __ballot(mine);
      const int at = c + __popcll(m & ((1ull << lane) - 1ull));
      if (mine && at < SMALL_ROWS) list[at] = i;
      c += __popcll(m);
    }
    if (lane == 0) count = min(c, SMALL_ROWS);
  }
  __syncthreads();
  const int cnt = count;
  if (cnt == 0) return;
  if (!early) fetch_w(s0);
  const int mts = min(MT, (cnt + 15) / 16);
  const bf16_t* xp[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    const int en = list[min(m * 16 + r, cnt - 1)];
    xp[m] = g.a + (long)(MODE == DOWN ? en : en / g.top) * g.lda + 8 * kg;
  }
  facc acc[MT][NM];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int n = 0; n < NM; ++n) acc[m][n] = facc{0.f, 0.f, 0.f, 0.f};
  for (int s = s0; s < s1; s += U) {
    uint4 xv[U][MT];
    if (s + U <= whole) {
#pragma unroll
      for (int m = 0; m < MT; ++m)
        if (m == 0 || m < mts) {
#pragma unroll
          for (int u = 0; u < U; ++u) xv[u][m] = *reinterpret_cast<const uint4*>(xp[m] + (s + u) * 32);
        } else {
#pragma unroll
          for (int u = 0; u < U; ++u) xv[u][m] = make_uint4(0, 0, 0, 0);
        }
    } else {
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int m = 0; m < MT; ++m) xv[u][m] = load_or_zero(xp[m] + (s + u) * 32, m < mts && s + u < s1 && (s + u) * 32 + 8 * kg < g.K);
    }
    __builtin_amdgcn_sched_barrier(0);  // the whole batch in flight before the first MFMA
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int n = 0; n < NM; ++n) acc[m][n] = mfma(as_frag(wv[u][n]), as_frag(xv[u][m]), acc[m][n]);
    if (s + U < s1) fetch_w(s + U);
  }
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int n = 0; n < NM; ++n) red[wave][m * NM + n][lane] = acc[m][n];
  __syncthreads();
  for (int i = tid; i < MT * 64; i += 256) {
    const int m = i >> 6, l = i & 63, row = m * 16 + (l & 15), c = n0 + 4 * (l >> 4);
    if (row >= cnt || c >= g.cols) continue;
    facc s[NM];
#pragma unroll
    for (int n = 0; n < NM; ++n) {
      s[n] = red[0][m * NM + n][l];
#pragma unroll
      for (int v = 1; v < 4; ++v) s[n] += red[v][m * NM + n][l];
    }
    const long o = (long)list[row] * g.cols + c;
    if constexpr (MODE == DOWN) {
      *reinterpret_cast<float4*>(static_cast<float*>(g.out) + o) = make_float4(s[0][0], s[0][1], s[0][2], s[0][3]);
    } else {
      float v[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) v[t] = NM == 2 ? expert_act(1, s[NM - 1][t], s[0][t]) : expert_act(g.act, s[0][t], 0.f);
      *reinterpret_cast<uint2*>(static_cast<bf16_t*>(g.out) + o) = make_uint2(pack2(v[0], v[1]), pack2(v[2], v[3]));
    }
  }
}

// ------------------------------------------------------------------------------------------------ weighted sum
template <typename Y>
__device__ __forceinline__ void load_y8(const Y* p, float* v) {
  Vec16<Y>::load(p, v);
  if constexpr (Vec16<Y>::N == 4) Vec16<Y>::load(p + 4, v + 4);
}

template <typename Y>
__global__ __launch_bounds__(256) void moe_combine_kernel(const Y* __restrict__ y, const int* __restrict__ idx, const float* __restrict__ wgt,
                                                          const bf16_t* __restrict__ x, long ldx, const bf16_t* __restrict__ shared, long lds_,
                                                          const bf16_t* __restrict__ gate, long ldg, float* __restrict__ out, long T, int W,
                                                          int E, int top) {
  const int per = W >> 3;
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= T * per) return;
  const long t = i / per;
  const int c = (int)(i - t * per) * 8;
  float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  for (int k = 0; k < top; ++k) {
    const long en = t * top + k;
    const float w = wgt[en];
    float v[8];
    if (idx[en] < E) load_y8<Y>(y + en * W + c, v);
    else Vec16<bf16_t>::load(x + t * ldx + c, v);  // an expert without weights gives its input
#pragma unroll
    for (int j = 0; j < 8; ++j) s[j] = fmaf(w, v[j], s[j]);
  }
  if (shared != nullptr) {
    float v[8];
    Vec16<bf16_t>::load(shared + t * lds_ + c, v);
    const float gt = gate != nullptr ? 1.0f / (1.0f + expf(-ldf(gate + t * ldg))) : 1.0f;
#pragma unroll
    for (int j = 0; j < 8; ++j) s[j] = fmaf(gt, v[j], s[j]);
  }
  Vec16<float>::store(out + t * W + c, s);
  Vec16<float>::store(out + t * W + c + 4, s + 4);
}

// Expert weights as one [E, rows, K] tensor (any strides but a unit last one) or a list of [rows, K] tensors.
ExpertPtrs expert_ptrs(at::TensorList ws, int64_t& E, int64_t& rows, int64_t& K, long& ld, const char* name) {
  ExpertPtrs p{};
  HYB_CHECK(!ws.empty(), name, ": no experts");
  const bool stacked = ws.size() == 1 && ws[0].dim() == 3;
  E = stacked ? ws[0].size(0) : (int64_t)ws.size();
  HYB_CHECK(E >= 1 && E <= MAX_EXPERTS, name, ": 1 .. 128 experts");
  for (int64_t e = 0; e < E; ++e) {
    const at::Tensor& w = stacked ? ws[0] : ws[e];
    HYB_CHECK(w.is_cuda() && w.scalar_type() == at::kBFloat16 && (stacked || w.dim() == 2), name, ": bf16 GPU weights");
    const int64_t r = w.size(-2), k = w.size(-1), l = w.stride(-2);
    if (e == 0) rows = r, K = k, ld = l;
    HYB_CHECK(r == rows && k == K && l == ld && w.stride(-1) == 1, name, ": experts of one shape and layout");
    p.p[e] = reinterpret_cast<const bf16_t*>(w.data_ptr()) + (stacked ? e * w.stride(0) : 0);
    HYB_CHECK(reinterpret_cast<uintptr_t>(p.p[e]) % 16 == 0 && l % 8 == 0, name, ": rows aligned to 16 bytes");
  }
  return p;
}

bool rows16(const at::Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0 && t.stride(0) % 8 == 0 && t.stride(1) == 1; }

}  // namespace

RouterChoice router_choice(const at::Tensor& w, int64_t W, const c10::optional<at::Tensor>& bias, int64_t top, int64_t groups, int64_t keep, bool softmax,
                           bool renorm) {
  HYB_CHECK(w.is_cuda() && w.dim() == 2 && w.is_contiguous() && w.scalar_type() == at::kFloat && w.size(1) == W && reinterpret_cast<uintptr_t>(w.data_ptr()) % 16 == 0,
            "router: contiguous fp32 [E, W]");
  const int64_t E = w.size(0);
  HYB_CHECK(E >= 1 && E <= MAX_EXPERTS && top >= 1 && top <= E && top <= 64, "1 .. 128 router outputs, top in 1 .. min(E, 64)");
  HYB_CHECK(groups >= 1 && E % groups == 0 && keep >= 1 && keep <= groups && top <= keep * (E / groups), "experts split into equal groups; top fits the kept groups");
  if (bias.has_value()) HYB_CHECK(bias->is_cuda() && bias->is_contiguous() && bias->scalar_type() == at::kFloat && bias->numel() == E, "bias: fp32 [E]");
  return RouterChoice{bias.has_value() ? bias->data_ptr<float>() : nullptr, (int)E, (int)top, (int)groups, (int)keep, softmax ? 1 : 0, renorm ? 1 : 0};
}

// The chosen experts (int32 [T, top]) and their weights (fp32 [T, top]) of rows x [T, W] under the fp32 router weight [E, W].
std::tuple<at::Tensor, at::Tensor> moe_route(const at::Tensor& x, const at::Tensor& w, const c10::optional<at::Tensor>& bias, int64_t top,
                                             int64_t groups, int64_t keep, bool softmax, bool renorm) {
  HYB_CHECK(x.is_cuda() && x.dim() == 2 && x.scalar_type() == at::kBFloat16 && x.size(1) % 8 == 0 && rows16(x), "x: bf16 [T, W], aligned rows");
  const RouterChoice c = router_choice(w, x.size(1), bias, top, groups, keep, softmax, renorm);
  const int64_t T = x.size(0), W = x.size(1);
  c10::DeviceGuard guard(x.device());
  at::Tensor idx = at::empty({T, top}, x.options().dtype(at::kInt)), wgt = at::empty({T, top}, x.options().dtype(at::kFloat));
  if (T == 0) return {idx, wgt};
  moe_route_kernel<<<dim3((unsigned)((T + ROUTE_T - 1) / ROUTE_T)), ROUTE_WAVES * 64, 0, cur_stream()>>>(
      reinterpret_cast<const bf16_t*>(x.data_ptr()), x.stride(0), w.data_ptr<float>(), c, idx.data_ptr<int>(), wgt.data_ptr<float>(), (int)T, (int)W);
  return {idx, wgt};
}

// Results of the chosen experts of every row of x, [T * top, W] by entry: fp32 for few tokens, else bf16.  ``act``: 0 relu^2, 1 silu-gated
// (up weights hold [gate ; up]), 2 gelu.  idx >= the number of experts: an expert that gives its input, whose entries are not written.
namespace {
// A shared expert's two products beside the experts': z = act(x w_up^T + bias) on its first act_cols columns, y = z[:, :act_cols] w_down^T.
struct SharedExpert {
  const at::Tensor *up, *bias, *down;
  int64_t act_cols;
  at::Tensor z, y;
};
bool side_rides(int64_t M, int64_t N, int64_t K) {
  const stream_linear::Form f = stream_linear::form_of((int)M, (int)N, (int)K);
  return M <= 32 && f.nt == 1 && f.nw == 4 && f.u == 8;
}

at::Tensor expert_rows(const at::Tensor& x, const at::Tensor& idx, const at::Tensor& wgt, at::TensorList up, at::TensorList down, int64_t act, SharedExpert* sh,
                       int64_t form = 0) {
  int64_t E, R, W, E2, W2, ff;
  long ldu, ldd;
  const ExpertPtrs pu = expert_ptrs(up, E, R, W, ldu, "up"), pd = expert_ptrs(down, E2, W2, ff, ldd, "down");
  HYB_CHECK(act >= 0 && act <= 2, "act: 0 relu2, 1 gated silu, 2 gelu");
  HYB_CHECK(E == E2 && W == W2 && R == (act == 1 ? 2 * ff : ff) && W % 8 == 0 && ff % 8 == 0, "up and down weights fit each other");
  HYB_CHECK(x.is_cuda() && x.dim() == 2 && x.scalar_type() == at::kBFloat16 && x.size(1) == W && rows16(x), "x: bf16 [T, W], aligned rows");
  const int64_t T = x.size(0), top = idx.size(1), N = T * top;
  HYB_CHECK(idx.is_cuda() && idx.is_contiguous() && idx.scalar_type() == at::kInt && idx.dim() == 2 && idx.size(0) == T, "idx: int32 [T, top]");
  HYB_CHECK(wgt.is_cuda() && wgt.is_contiguous() && wgt.scalar_type() == at::kFloat && wgt.sizes() == idx.sizes(), "weights: fp32 [T, top]");
  HYB_CHECK(N < ((int64_t)1 << 30), "too many token copies");
  c10::DeviceGuard guard(x.device());
  const hipStream_t st = cur_stream();
  const bool small = T <= SMALL_ROWS;
  at::Tensor y = at::empty({N, W}, x.options().dtype(small ? at::kFloat : at::kBFloat16));
  if (T == 0) return y;
  at::Tensor a = at::empty({N, ff}, x.options());
  const bf16_t* xp = reinterpret_cast<const bf16_t*>(x.data_ptr());
  bf16_t* ap = reinterpret_cast<bf16_t*>(a.data_ptr());
  if (small) {
    SmallArgs u{xp, (long)x.stride(0), pu, ldu, ap, idx.data_ptr<int>(), (int)N, (int)W, (int)ff, (int)top, (int)act, (int)E, {}, 0};
    SmallArgs d{ap, (long)ff, pd, ldd, y.data_ptr(), idx.data_ptr<int>(), (int)N, (int)ff, (int)W, (int)top, (int)act, (int)E, {}, 0};
    dim3 gu((unsigned)((ff + 15) / 16), (unsigned)E), gd((unsigned)((W + 15) / 16), (unsigned)E);
    if (sh != nullptr) {
      const int64_t C = sh->up->size(0);
      sh->z = at::empty({T, C}, x.options());
      sh->y = at::empty({T, W}, x.options());
      auto ptr = [](const at::Tensor& t) { return reinterpret_cast<const bf16_t*>(t.data_ptr()); };
      u.side = stream_linear::Args{xp, (long)x.stride(0), ptr(*sh->up), (long)sh->up->stride(0), sh->bias != nullptr ? ptr(*sh->bias) : nullptr, sh->z.data_ptr(),
                                   (int)T, (int)C, (int)W, act == 0 ? 3 : 1, (int)sh->act_cols, 0};
      d.side = stream_linear::Args{ptr(sh->z), (long)C, ptr(*sh->down), (long)sh->down->stride(0), nullptr, sh->y.data_ptr(), (int)T, (int)W, (int)sh->act_cols, 0, 0, 0};
      auto ride = [](SmallArgs& g, dim3& grid) {
        g.side.rows = stream_linear::form_of(g.side.M, g.side.N, g.side.K).rows;
        g.side_groups = (g.side.N + g.side.rows - 1) / g.side.rows;
        grid.y += ((unsigned)g.side_groups + grid.x - 1) / grid.x;
      };
      ride(u, gu);
      ride(d, gd);
    }
    auto go = [&](auto mt) {
      constexpr int MT = decltype(mt)::value;
      if constexpr (MT <= 2) {
        if (sh != nullptr) {
          moe_small_kernel<MT, UP_PLAIN, true><<<gu, 256, 0, st>>>(u);
          moe_small_kernel<MT, DOWN, true><<<gd, 256, 0, st>>>(d);
          return;
        }
      }
      if (act == 1) moe_small_kernel<MT, UP_GLU, false><<<gu, 256, 0, st>>>(u);
      else moe_small_kernel<MT, UP_PLAIN, false><<<gu, 256, 0, st>>>(u);
      moe_small_kernel<MT, DOWN, false><<<gd, 256, 0, st>>>(d);
    };
    if (T <= 16) go(std::integral_constant<int, 1>{});
    else if (T <= 32) go(std::integral_constant<int, 2>{});
    else go(std::integral_constant<int, 4>{});
  } else {
    const bool wide = form != 1 && (moe_wide_pays(N, E, W, ff, act == 1) || (form == 2 && W % 128 == 0 && ff % 128 == 0 && W >= 256 && ff >= 256)) && T * x.stride(0) < ((int64_t)1 << 30) && N * ff < ((int64_t)1 << 30) && R * ldu < ((int64_t)1 << 30) &&
                      W * ldd < ((int64_t)1 << 30);
    const int BM = wide ? WIDE_ROWS : N >= 96 * E ? 128 : 64, BN = wide ? llmctl::wide::COLS : BM;
    const int64_t mt = wide ? N / 256 + E : (N + BM - 1) / BM + E;  // no more row tiles than this
    at::Tensor ints = at::empty({N + 2 + 3 * mt}, idx.options());
    int* perm = ints.data_ptr<int>();
    int* tiles = perm + N;
    moe_group_kernel<<<dim3((unsigned)E), 1024, 0, st>>>(idx.data_ptr<int>(), (int)N, (int)E, BM, perm, tiles);
    const int64_t cu = act == 1 ? BN / 2 : BN;
    TileArgs u{xp, (long)x.stride(0), pu, ldu, ap, perm, tiles, (int)W, (int)ff, (int)top, (int)act, (int)((ff + cu - 1) / cu), (int)mt};
    TileArgs d{ap, (long)ff, pd, ldd, reinterpret_cast<bf16_t*>(y.data_ptr()), perm, tiles, (int)ff, (int)W, (int)top, (int)act, (int)((W + BN - 1) / BN), (int)mt};
    if (wide) {  // (16 more: what the two runs of an XCD are rounded up by)
      const dim3 gu((unsigned)(mt * u.ntile + 16)), gd((unsigned)(mt * d.ntile + 16));
      if (act == 1) moe_wide_kernel<UP_GLU><<<gu, 256, 0, st>>>(u);
      else if (act == 0) moe_wide_kernel<UP_PLAIN><<<gu, 256, 0, st>>>(u);
      else moe_wide_kernel<UP_GELU><<<gu, 256, 0, st>>>(u);
      moe_wide_kernel<DOWN><<<gd, 256, 0, st>>>(d);
      return y;
    }
    const dim3 gu((unsigned)(mt * u.ntile)), gd((unsigned)(mt * d.ntile));
    if (BM == 128) {
      if (act == 1) moe_tile_kernel<128, 128, UP_GLU, 1, 1, 3><<<gu, 256, 0, st>>>(u);
      else moe_tile_kernel<128, 128, UP_PLAIN, 1, 1, 3><<<gu, 256, 0, st>>>(u);
      moe_tile_kernel<128, 128, DOWN, 1, 1, 3><<<gd, 256, 0, st>>>(d);
    } else {
      if (act == 1) moe_tile_kernel<64, 64, UP_GLU, 3, 2, 3><<<gu, 256, 0, st>>>(u);
      else moe_tile_kernel<64, 64, UP_PLAIN, 3, 2, 3><<<gu, 256, 0, st>>>(u);
      moe_tile_kernel<64, 64, DOWN, 3, 2, 3><<<gd, 256, 0, st>>>(d);
    }
  }
  return y;
}

}  // namespace

at::Tensor moe_expert_rows(const at::Tensor& x, const at::Tensor& idx, const at::Tensor& wgt, at::TensorList up, at::TensorList down, int64_t act) {
  return expert_rows(x, idx, wgt, up, down, act, nullptr);
}

// Whether moe_expert_rows_shared takes a shared expert of these sizes: M rows of width K to N columns, the first ff of them back to K.
bool moe_shared_rides(int64_t M, int64_t N, int64_t K, int64_t ff) { return M >= 1 && M <= 32 && ff >= 8 && ff <= N && side_rides(M, N, K) && side_rides(M, K, ff); }

// moe_expert_rows of at most 32 rows, and a shared expert's products in the same launches: (experts' rows, act(x w_sup^T + bias) with the activation on
// the first act_cols columns, those columns' product with w_sdown).  act: 0 relu^2, 2 gelu.
std::tuple<at::Tensor, at::Tensor, at::Tensor> moe_expert_rows_shared(const at::Tensor& x, const at::Tensor& idx, const at::Tensor& wgt, at::TensorList up,
                                                                      at::TensorList down, int64_t act, const at::Tensor& w_sup,
                                                                      const c10::optional<at::Tensor>& b_sup, int64_t act_cols, const at::Tensor& w_sdown) {
  HYB_CHECK(x.dim() == 2 && w_sup.dim() == 2 && w_sdown.dim() == 2 && (act == 0 || act == 2), "shared expert: matrices, relu^2 or gelu");
  const int64_t M = x.size(0), K = x.size(1), N = w_sup.size(0);
  HYB_CHECK(moe_shared_rides(M, N, K, act_cols) && act_cols % 8 == 0 && N % 8 == 0, "shared expert: sizes (moe_shared_rides)");
  for (const at::Tensor* w : {&w_sup, &w_sdown})
    HYB_CHECK(w->is_cuda() && w->scalar_type() == at::kBFloat16 && rows16(*w), "shared expert: bf16 weights, aligned rows");
  HYB_CHECK(w_sup.size(1) == K && w_sdown.size(0) == K && w_sdown.size(1) == act_cols, "shared expert: weights fit each other");
  if (b_sup.has_value())
    HYB_CHECK(b_sup->is_cuda() && b_sup->scalar_type() == at::kBFloat16 && b_sup->is_contiguous() && b_sup->numel() == N, "shared expert: bias bf16 [N]");
  SharedExpert sh{&w_sup, b_sup.has_value() ? &*b_sup : nullptr, &w_sdown, act_cols, {}, {}};
  const at::Tensor y = expert_rows(x, idx, wgt, up, down, act, &sh);
  return {y, sh.z, sh.y};
}

ExpertRows expert_rows_of(const at::Tensor& y, const at::Tensor& idx, const at::Tensor& wgt, const at::Tensor& x,
                          const c10::optional<at::Tensor>& shared, const c10::optional<at::Tensor>& gate, int64_t experts) {
  HYB_CHECK(x.is_cuda() && x.dim() == 2 && x.scalar_type() == at::kBFloat16 && rows16(x), "x: bf16 [T, W], aligned rows");
  const int64_t T = x.size(0), W = x.size(1);
  HYB_CHECK(idx.is_cuda() && idx.is_contiguous() && idx.scalar_type() == at::kInt && idx.dim() == 2 && idx.size(0) == T, "idx: int32 [T, top]");
  HYB_CHECK(wgt.is_cuda() && wgt.is_contiguous() && wgt.scalar_type() == at::kFloat && wgt.sizes() == idx.sizes(), "weights: fp32 [T, top]");
  HYB_CHECK(y.is_cuda() && y.is_contiguous() && y.dim() == 2 && y.size(0) == idx.numel() && y.size(1) == W && W % 8 == 0 &&
                (y.scalar_type() == at::kFloat || y.scalar_type() == at::kBFloat16) && reinterpret_cast<uintptr_t>(y.data_ptr()) % 16 == 0,
            "experts' rows: contiguous fp32 or bf16 [T * top, W]");
  if (shared.has_value())
    HYB_CHECK(shared->is_cuda() && shared->dim() == 2 && shared->scalar_type() == at::kBFloat16 && shared->size(0) == T && shared->size(1) == W && rows16(*shared),
              "shared: bf16 [T, W], aligned rows");
  if (gate.has_value())
    HYB_CHECK(shared.has_value() && gate->is_cuda() && gate->scalar_type() == at::kBFloat16 && gate->dim() == 2 && gate->size(0) == T, "gate: bf16 [T, 1]");
  return ExpertRows{y.data_ptr(), idx.data_ptr<int>(), wgt.data_ptr<float>(), reinterpret_cast<const bf16_t*>(x.data_ptr()), (long)x.stride(0),
                    shared.has_value() ? reinterpret_cast<const bf16_t*>(shared->data_ptr()) : nullptr, shared.has_value() ? (long)shared->stride(0) : 0,
                    gate.has_value() ? reinterpret_cast<const bf16_t*>(gate->data_ptr()) : nullptr, gate.has_value() ? (long)gate->stride(0) : 0,
                    (int)experts, (int)idx.size(1)};
}

// sum_k wgt[t, k] y[t, k] (+ sigmoid(gate_t) shared_t) of moe_expert_rows' results, fp32 [T, W]
at::Tensor moe_sum(const at::Tensor& y, const at::Tensor& idx, const at::Tensor& wgt, const at::Tensor& x, const c10::optional<at::Tensor>& shared,
                   const c10::optional<at::Tensor>& gate, int64_t experts) {
  const ExpertRows m = expert_rows_of(y, idx, wgt, x, shared, gate, experts);
  const int64_t T = x.size(0), W = x.size(1);
  c10::DeviceGuard guard(x.device());
  at::Tensor out = at::empty({T, W}, x.options().dtype(at::kFloat));
  if (T == 0) return out;
  auto sum = [&](auto* tag) {
    using Y = std::remove_pointer_t<decltype(tag)>;
    moe_combine_kernel<Y><<<dim3((unsigned)((T * (W / 8) + 255) / 256)), 256, 0, cur_stream()>>>(
        static_cast<const Y*>(m.y), m.idx, m.wgt, m.x, m.ldx, m.shared, m.ld_shared, m.gate, m.ld_gate, out.data_ptr<float>(), (long)T, (int)W, m.E, m.top);
  };
  if (y.scalar_type() == at::kFloat) sum((float*)nullptr);
  else sum((bf16_t*)nullptr);
  return out;
}

// form (tests, sweeps): 0 the faster tiles (moe_wide_pays), 1 those of 64 or 128 rows, 2 those of moe_wide.h where they take the widths
at::Tensor moe_experts(const at::Tensor& x, const at::Tensor& idx, const at::Tensor& wgt, at::TensorList up, at::TensorList down, int64_t act,
                       const c10::optional<at::Tensor>& shared, const c10::optional<at::Tensor>& gate, int64_t form) {
  const at::Tensor y = expert_rows(x, idx, wgt, up, down, act, nullptr, form);
  return moe_sum(y, idx, wgt, x, shared, gate, up.size() == 1 && up[0].dim() == 3 ? up[0].size(0) : (int64_t)up.size());
}

}  // namespace llmctl_hybrid
