// All layers of a decode step in one launch, for a few rows of a small pre-norm model (LayerNorm, biases, GELU, learned positions, full heads of 64): the
// embedding, every layer with its paged cache, the final norm.
//
// Bound of what it replaces: the chain of launches.  A layer of gpt2-125m is five kernels of 4 to 7 us (3.5 is an empty one's share of a graph) around 14 MB of
// weights, 3 us of HBM time.  Here 128 workgroups stay for the whole step; each owns the same share of every projection's outputs and asks for its weights of the
// next product before it waits for that product's operand, so the weights' way is hidden and what is left is the way of the operands.
//
// Operands travel as 8-byte words {value, tag}, written and polled with relaxed agent-scope accesses, which pass the XCDs' L2s by: a word that carries its own
// tag needs no flag, no barrier and no fence (an agent fence writes an L2 back: a grid barrier with fences measured 20 us, with a counter of relaxed accesses
// 4.3, such words 1.5 us for 512 among 64 workgroups, 2.2 among 128).  The tag is the layer, counted on over all steps (32 bits, of the MLP's words the low 16); the
// count lives in the workspace.  Words of rows and spans that a step does not have get its last tag all the same, so that none is older than the step before, whose
// tags no layer of this one has, and the count may wrap.
// Layer: qkv -> heads (a workgroup per head, row and span of keys) -> output projection -> up -> down, five such exchanges.  A word's place is used once a
// layer.  Nobody writes it again before all have read it: between two writes of any place every workgroup takes part in the down projection's exchange, which
// every workgroup waits for, and each sends its part of that after it has read what the layer sent before.
//
// A workgroup waits only for workgroups that run: each takes a number at the start; the step begins when all have one or, after the gate's time, with those that
// have (any number works: the 128 shares go round); later ones find the gate closed and leave.  So no launch beside it, however long, can stop it for good.
// The gate's time is what fewer workgroups cost: as much for every round of shares beyond the first as that round takes, so a step beside another stream's kernels
// takes at most about twice what the best choice would have (after a fixed 200 us some went through with one workgroup).  gpt2-125m, context 129, us a step by
// workgroups: 128 164, 127 208, 64 247, 32 361, 16 587, 7 1234, 1 7671; four rows 253 .. 17614.  Beside causal attention of 4 x 4096 tokens, 32 heads (670 us a
// launch), us a step, median and longest of 540: 688, 1050; after 200 us 671, 10926; the chain of launches 1539, 1709.  Beside products of 8192 930 (the chain 23400),
// of 2048 278 (555), copies 428 (871).
// Waits are bounded all the same: a step that overran ends with NaN rows and sets a word of the host's.
//
// fp32 throughout but for weights, cache rows, the MLP's activations (three to a word, rounded as between two launches) and the normed result; the sums of a
// product run over 64 lanes, then pairwise, whatever the number of workgroups.
//
// What it took (one row, gpt2-125m, context 129, whole step; five launches a layer 369 us): 64 workgroups of 1024 threads 369 us, registers spilt; 512 threads and
// the pointers in LDS 282; global, not flat, loads 270; no load under a condition (its use waits for all loads) 254; the next weights asked for after a
// product's results are sent 234; 128 workgroups 219; asking again only for missing words 214; three activations to a word 206.  Now, us, launches / this: one row
// context 129 381 / 203, 700 406 / 233, 2000 432 / 252; at 129 two rows 396 / 239, three 418 / 294, four 420 / 297.  Of a layer's 13 us half is the words' way.
#include "common.h"

namespace llmctl {
namespace {

constexpr int PARTS = 128, WAVES = 8, THREADS = WAVES * 64, MAX_LAYERS = 32, MAX_ROWS = 4, R = 4;  // R: MLP width over hidden
constexpr int D = 64, U = 4;  // head size; cache tokens that a lane has in flight
constexpr int SPAN = U * WAVES * 8;                    // keys of a workgroup, where there are workgroups to share them out to
constexpr unsigned CLOSED = 1u << 30;

using u64 = unsigned long long;
using bf16 = unsigned short;
using gbf16 = const __attribute__((address_space(1))) unsigned short;
using b4 = __attribute__((ext_vector_type(2))) unsigned;  // four bf16
using gb4 = const __attribute__((address_space(1))) b4;

// a pointer that was kept in LDS, as the global one that it is and in scalar registers: through a flat one every wait for LDS would wait for the weights too
__device__ __forceinline__ gbf16* global(const bf16* p) {
  const u64 a = (u64)p;
  const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)a), hi = __builtin_amdgcn_readfirstlane((unsigned)(a >> 32));
  return (gbf16*)(((u64)hi << 32) | lo);
}

struct LayerW {
  const bf16 *n1w, *n1b, *wqkv, *bqkv, *wo, *bo, *n2w, *n2b, *wu, *bu, *wd, *bd;
};

struct Control {  // the workspace starts with this, zero before the first step
  unsigned gate, left, base, late;  // left: workgroups that are through, and above bit 16 those that saw the step lost
};
struct Wait {
  Control* ctl;
  int spins;  // tries of a wait
};

struct StepArgs {
  LayerW layer[MAX_LAYERS];
  const bf16 *nw, *nb, *table, *ptable;
  bf16 *kc, *vc, *out;
  const int64_t *ids, *slots;
  const int *pos, *bt, *ctx;
  Wait wait;
  u64* ws;
  unsigned* lost;  // nullptr or the host's word that a lost step sets
  long rows, prows, layer_stride;  // of the tables; elements of a layer's cache
  float eps, scale;
  int L, B, heads, block, max_blocks, gate_ticks;  // a round's, of the 100 MHz clock
};

template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
// sum over the wave in every lane: quads, halves and rows of 16 by lane permutes, then the rows by swaps
__device__ __forceinline__ float lanes_sum(float v) {
  v += dpp<0xB1>(v);   // lane ^ 1
  v += dpp<0x4E>(v);   // lane ^ 2
  v += dpp<0x141>(v);  // mirrored halves of 8
  v += dpp<0x140>(v);  // mirrored rows of 16
  auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(p[0]) + __uint_as_float(p[1]);
  p = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(p[0]) + __uint_as_float(p[1]);
}

__device__ __forceinline__ float lanes_max(float v) {
  v = fmaxf(v, dpp<0xB1>(v));
  v = fmaxf(v, dpp<0x4E>(v));
  v = fmaxf(v, dpp<0x141>(v));
  v = fmaxf(v, dpp<0x140>(v));
  auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = fmaxf(__uint_as_float(p[0]), __uint_as_float(p[1]));
  p = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(p[0]), __uint_as_float(p[1]));
}
// sum of the lanes that share their place among eight
__device__ __forceinline__ float groups_sum(float v) {
  v += dpp<0x128>(v);  // the row of 16 turned by 8
  auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(p[0]) + __uint_as_float(p[1]);
  p = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(p[0]) + __uint_as_float(p[1]);
}

__device__ __forceinline__ void put_word(u64* p, u64 v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ void send(u64* p, float v, unsigned tag) { put_word(p, ((u64)tag << 32) | __float_as_uint(v)); }
__device__ __forceinline__ unsigned peek(const unsigned* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
// whether to stop waiting: after so many tries of anybody's, the step is lost
__device__ __forceinline__ bool give_up(int n, Wait w) {
  if ((n & 4095) != 0 && n < w.spins) return false;
  if (n >= w.spins) __hip_atomic_store(&w.ctl->late, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return n >= w.spins || peek(&w.ctl->late) != 0;
}
__device__ __forceinline__ u64 word(const u64* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ float take(const u64* p, unsigned tag, Wait wait) {
  for (int n = 1;; ++n) {
    const u64 v = word(p);
    if ((unsigned)(v >> 32) == tag) return __uint_as_float((unsigned)v);
    if (give_up(n, wait)) return __uint_as_float(0x7fc00000u);
  }
}
// count words, eight of a thread's in flight; put(i, word) for each.  BITS: of the tag, at the top
template <int BITS, typename Put>
__device__ __forceinline__ void gather(const u64* src, int count, unsigned tag, Wait wait, Put put) {
  constexpr int W = 8;
  for (int i0 = threadIdx.x; i0 < count; i0 += W * THREADS) {
    u64 v[W];
    unsigned miss = 0;  // only what is still missing is asked for again: everybody polls beside those that compute
#pragma unroll
    for (int j = 0; j < W; ++j) miss |= i0 + j * THREADS < count ? 1u << j : 0u;
    for (int n = 1; miss != 0; ++n) {
#pragma unroll
      for (int j = 0; j < W; ++j)
        if (miss >> j & 1) v[j] = word(src + i0 + j * THREADS);
#pragma unroll
      for (int j = 0; j < W; ++j)
        if ((miss >> j & 1) && (unsigned)(v[j] >> (64 - BITS)) == (tag & (unsigned)((1ull << BITS) - 1))) miss &= ~(1u << j);
      if (miss != 0 && give_up(n, wait)) {
#pragma unroll
        for (int j = 0; j < W; ++j)
          if (miss >> j & 1) v[j] = 0x7fc07fc07fc07fc0ull;
        miss = 0;
      }
    }
#pragma unroll
    for (int j = 0; j < W; ++j)
      if (i0 + j * THREADS < count) put(i0 + j * THREADS, v[j]);
  }
}
// fp32 words into LDS
__device__ __forceinline__ void gather_f32(float* dst, const u64* src, int count, unsigned tag, Wait wait) {
  gather<32>(src, count, tag, wait, [&](int i, u64 v) { dst[i] = __uint_as_float((unsigned)v); });
}

__device__ __forceinline__ void widen(b4 v, float (&o)[4]) {
  o[0] = __uint_as_float(v.x << 16), o[1] = __uint_as_float(v.x & 0xffff0000u);
  o[2] = __uint_as_float(v.y << 16), o[3] = __uint_as_float(v.y & 0xffff0000u);
}

// rows of a weight [*, ld] that a wave owns in share v: outputs v * n + WAVES u + wave (u < NU) over columns [k0, k0 + 256 KC); past the share: its last row again
template <int KC, int NU>
struct Rows {
  b4 w[NU][KC];
  __device__ __forceinline__ void load(const bf16* p, long ld, int first, int n, int wave, int lane) {
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      gbf16* q = global(p) + (long)(first + min(WAVES * u + wave, n - 1)) * ld;
#pragma unroll
      for (int c = 0; c < KC; ++c) w[u][c] = *(gb4*)(q + c * 256 + lane * 4);
    }
  }
};

// the same for the down projection, whose units are quarters of its sums: unit i of a share is output i / R, quarter i % R
template <int KC, int NU>
struct Down {
  b4 w[NU][KC];
  __device__ __forceinline__ void load(const bf16* p, int first, int wave, int lane) {
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      const int i = min(WAVES * u + wave, 256 * KC / PARTS * R - 1);
      gbf16* q = global(p) + (long)(first + i / R) * (R * 256 * KC) + (i % R) * (256 * KC);
#pragma unroll
      for (int c = 0; c < KC; ++c) w[u][c] = *(gb4*)(q + c * 256 + lane * 4);
    }
  }
};

// lane u of the wave: dot of its unit u with x
template <int KC, int NU>
__device__ __forceinline__ float dots(const b4 (&w)[NU][KC], const float (&x)[KC][4], int lane) {
  float out = 0.f;
#pragma unroll
  for (int u = 0; u < NU; ++u) {
    float s[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < KC; ++c) {
      float t[4];
      widen(w[u][c], t);
#pragma unroll
      for (int j = 0; j < 4; ++j) s[j] += t[j] * x[c][j];
    }
    const float r = lanes_sum((s[0] + s[1]) + (s[2] + s[3]));
    out = lane == u ? r : out;
  }
  return out;
}

template <int KC>
__device__ __forceinline__ void read_row(const float* s, int lane, float (&x)[KC][4]) {
#pragma unroll
  for (int c = 0; c < KC; ++c) {
    const float4 v = *reinterpret_cast<const float4*>(s + c * 256 + lane * 4);
    x[c][0] = v.x, x[c][1] = v.y, x[c][2] = v.z, x[c][3] = v.w;
  }
}

template <int KC>
__device__ __forceinline__ void layernorm(float (&x)[KC][4], const b4 (&w)[KC], const b4 (&b)[KC], float eps) {
  float s = 0.f, q = 0.f;
#pragma unroll
  for (int c = 0; c < KC; ++c)
#pragma unroll
    for (int j = 0; j < 4; ++j) s += x[c][j];
  const float mean = lanes_sum(s) * (1.f / (256 * KC));
#pragma unroll
  for (int c = 0; c < KC; ++c)
#pragma unroll
    for (int j = 0; j < 4; ++j) q += (x[c][j] - mean) * (x[c][j] - mean);
  const float rs = rsqrtf(lanes_sum(q) * (1.f / (256 * KC)) + eps);
#pragma unroll
  for (int c = 0; c < KC; ++c) {
    float g[4], h[4];
    widen(w[c], g);
    widen(b[c], h);
#pragma unroll
    for (int j = 0; j < 4; ++j) x[c][j] = (x[c][j] - mean) * rs * g[j] + h[j];
  }
}

__device__ __forceinline__ float gelu(float v) {
  return 0.5f * v * (1.0f + tanhf(0.7978845608028654f * (v + 0.044715f * v * v * v)));
}

// KC: hidden / 256; ROWS: rows at the most, two at a time through a product
template <int KC, int ROWS>
__global__ __launch_bounds__(THREADS, 1) void decode_layers_kernel(StepArgs g) {
  constexpr int H = 256 * KC, F = R * H, NQ = 3 * H / PARTS, NO = H / PARTS, NF = F / PARTS, ND = R * NO, WF = (NF + 2) / 3;
  constexpr int UQ = (NQ + WAVES - 1) / WAVES, UO = (NO + WAVES - 1) / WAVES, UF = (NF + WAVES - 1) / WAVES, UD = (ND + WAVES - 1) / WAVES;
  __shared__ __attribute__((aligned(16))) float xs[ROWS][H], as[ROWS][H], hs[ROWS][F];
  __shared__ float qkv[3][D], part[WAVES][D + 2], red[ROWS][ND], ups[ROWS][NF + 2];
  __shared__ LayerW layers[MAX_LAYERS];  // (read from the arguments, a layer's line of them is fetched when the layer starts)
  __shared__ int who[2];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const Wait wait = g.wait;
  Control* ctl = wait.ctl;
  // ---- the gate
  unsigned ticket = 0;
  if (tid == 0) ticket = __hip_atomic_fetch_add(&ctl->gate, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const unsigned base = peek(&ctl->base);
  if (tid == 0) {
    int n = 0;
    if (!(ticket & CLOSED) && (ticket & 0xffffu) < gridDim.x) {
      const long t0 = wall_clock64();
      unsigned seen = peek(&ctl->gate);
      for (;;) {
        const unsigned count = min(seen & 0xffffu, gridDim.x);  // (no more shares than there are, whoever else took numbers here)
        if (seen & CLOSED) n = (seen >> 16) & 0xff;
        else if (count == gridDim.x) n = (int)count;
        if (n != 0) break;
        // (rounds that these would take, less the one that all take; a second at the most)
        if (wall_clock64() - t0 >= min((long)g.gate_ticks * ((PARTS + (int)count - 1) / (int)count - 1), 100000000l)) {
          unsigned want = seen;
          if (__hip_atomic_compare_exchange_strong(&ctl->gate, &want, seen | CLOSED | (count << 16), __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                   __HIP_MEMORY_SCOPE_AGENT))
            n = (int)count;
          else
            seen = want;
        } else {
          seen = peek(&ctl->gate);
        }
      }
    }
    who[0] = (int)(ticket & 0xffffu), who[1] = n;
  }
  // ---- the rows' embeddings, and the first weights, meanwhile
  for (int i = tid; i < g.B * H; i += THREADS) {
    const int b = i / H, c = i - b * H;
    const int64_t id = g.ids[b];
    const long p = g.pos[b];
    CUDA_KERNEL_ASSERT(id >= 0 && id < g.rows && p >= 0 && p < g.prows);
    xs[b][c] = bf2f(g.table[id * H + c]) + bf2f(g.ptable[p * H + c]);
  }
  {
    const u64* from = reinterpret_cast<const u64*>(g.layer);
    for (int i = tid; i < g.L * (int)(sizeof(LayerW) / 8); i += THREADS) reinterpret_cast<u64*>(layers)[i] = from[i];
  }
  int top = 1;  // the longest context
  for (int b = 0; b < g.B; ++b) top = max(top, g.ctx[b]);
  __syncthreads();
  const int me = who[0], N = who[1];
  const int HB = g.heads * g.B, splits = max(1, min(min(PARTS / HB, ROWS * F / (D + 2)), (top - 1 + SPAN - 1) / SPAN)), items = HB * splits;
  // places of the words: qkv [B][3H], heads [B][H], after the output projection [B][H], up [B][F], down [B][H], partial heads [items][D + 2]
  u64* const pq = g.ws;
  u64* const pa = pq + (long)MAX_ROWS * 3 * H;
  u64* const px = pa + (long)MAX_ROWS * H;
  u64* const ph = px + (long)MAX_ROWS * H;
  u64* const py = ph + (long)MAX_ROWS * F;
  u64* const ps = py + (long)MAX_ROWS * H;

  bool late = false;  // a wait of this workgroup, or one that it has heard of, ran out (thread 0's)
  if (N != 0) {
    Rows<KC, UQ> wq;
    Rows<KC, UO> wo;
    Rows<KC, UF> wu;
    Down<KC, UD> wd;
    b4 nw[KC], nb[KC];
    auto norm_of = [&](const bf16* w, const bf16* b) __attribute__((always_inline)) {
#pragma unroll
      for (int c = 0; c < KC; ++c) {
        nw[c] = *(gb4*)(global(w) + c * 256 + lane * 4);
        nb[c] = *(gb4*)(global(b) + c * 256 + lane * 4);
      }
    };
    // lane u holds its unit's bias
    auto bias_of = [&](const bf16* b, int first, int n) __attribute__((always_inline)) { return bf2f(global(b)[first + min(WAVES * lane + wave, n - 1)]); };
    // an item of the heads: row b, head h, the sp-th span of its cached keys [k0, k1); lanes: eight tokens at a time, eight lanes to a token
    struct Item {
      int b, h, sp, k0, k1;
    };
    auto item = [&](int it) __attribute__((always_inline)) {
      Item x;
      const int bh = it / splits;
      x.sp = it - bh * splits, x.b = bh / g.heads, x.h = bh - x.b * g.heads;
      const int keys = g.ctx[x.b] - 1, per = (keys + splits - 1) / splits;
      x.k0 = min(x.sp * per, keys), x.k1 = min(x.k0 + per, keys);
      return x;
    };
    const int tg = lane >> 3, sub = lane & 7;
    // where the lane's tokens of a pass lie in a layer's cache, in rows of eight
    auto find = [&](const Item& x, int t0, unsigned (&at)[U]) __attribute__((always_inline)) {
      const int* bt = g.bt + (long)x.b * g.max_blocks;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int t = min(t0 + (u * WAVES + wave) * 8 + tg, x.k1 - 1);
        at[u] = ((unsigned)bt[t / g.block] * (unsigned)g.block + (unsigned)(t % g.block)) * (unsigned)(H / 8) + (unsigned)(x.h * (D / 8) + sub);
      }
    };
    auto fetch = [&](int l, const unsigned (&at)[U], uint4 (&kv)[U], uint4 (&vv)[U]) __attribute__((always_inline)) {
      const uint4 *kc = reinterpret_cast<const uint4*>(g.kc + l * g.layer_stride), *vc = reinterpret_cast<const uint4*>(g.vc + l * g.layer_stride);
#pragma unroll
      for (int u = 0; u < U; ++u) kv[u] = kc[at[u]], vv[u] = vc[at[u]];
    };
    uint4 kv0[U], vv0[U];
    unsigned at0[U] = {};  // (no keys: the cache's first rows are read and not used)
    // Loads are asked for a phase ahead and never under a condition: where a register's load may or may not be the last one, its use waits for all.
    const Item mine = item(min(me, items - 1));
    if (me < items && mine.k0 < mine.k1) find(mine, mine.k0, at0);
    norm_of(layers[0].n1w, layers[0].n1b);
    float bq = bias_of(layers[0].bqkv, me * NQ, NQ);
    wq.load(layers[0].wqkv, H, me * NQ, NQ, wave, lane);
    fetch(0, at0, kv0, vv0);
    for (int l = 0; l < g.L; ++l) {
      const LayerW& w = layers[l];
      const unsigned tag = base + l + 1;
      // ---- qkv
      if (l > 0) {
        gather_f32(xs[0], py, g.B * H, tag - 1, wait);
        __syncthreads();
      }
      auto qkv_of = [&](const Rows<KC, UQ>& r, float bias, int v) __attribute__((always_inline)) {
#pragma unroll ROWS == 1 ? 1 : 2
        for (int b = 0; b < ROWS; ++b) {
          float x[KC][4];
          read_row(xs[b], lane, x);
          layernorm(x, nw, nb, g.eps);
          const float s = dots(r.w, x, lane) + bias;
          if (b < g.B && lane < UQ && WAVES * lane + wave < NQ) send(pq + (long)b * 3 * H + v * NQ + WAVES * lane + wave, s, tag);
        }
      };
      qkv_of(wq, bq, me);
      wo.load(w.wo, H, me * NO, NO, wave, lane);
      const float bo = bias_of(w.bo, me * NO, NO);
      for (int v = me + N; v < PARTS; v += N) {
        Rows<KC, UQ> r;
        r.load(w.wqkv, H, v * NQ, NQ, wave, lane);
        qkv_of(r, bias_of(w.bqkv, v * NQ, NQ), v);
      }
      // ---- heads
      for (int it = me; it < items; it += N) {
        const Item x = it == me ? mine : item(it);
        const int b = x.b, h = x.h, k1 = x.k1;
        uint4 kv[U], vv[U];
#pragma unroll
        for (int u = 0; u < U; ++u) kv[u] = kv0[u], vv[u] = vv0[u];
        if (it != me && x.k0 < k1) {
          unsigned at[U];
          find(x, x.k0, at);
          fetch(l, at, kv, vv);
        }
        if (tid < 3 * D) {
          const int which = tid >> 6, d = tid & 63;
          float t = take(pq + (long)b * 3 * H + which * H + h * D + d, tag, wait);
          if (which != 0) {  // as the cache holds it
            const bf16 r = f2bf(t);
            t = bf2f(r);
            const long slot = g.slots[b];
            if (x.sp == 0 && slot >= 0) (which == 1 ? g.kc : g.vc)[l * g.layer_stride + slot * H + h * D + d] = r;
          }
          qkv[which][d] = t;
        }
        __syncthreads();
        float q[8], o[8], m = -INFINITY, sum = 0.f;
#pragma unroll
        for (int j = 0; j < 8; ++j) q[j] = qkv[0][sub * 8 + j] * g.scale * 1.44269504088896340736f, o[j] = 0.f;
        auto score = [&](const float (&k)[8], bool in) __attribute__((always_inline)) {
          float s = 0.f;
#pragma unroll
          for (int j = 0; j < 8; ++j) s += q[j] * k[j];
          s += dpp<0xB1>(s);
          s += dpp<0x4E>(s);
          s += dpp<0x141>(s);
          return in ? s : -INFINITY;
        };
        for (int t0 = x.k0; t0 < k1; t0 += U * WAVES * 8) {
          if (t0 > x.k0) {
            unsigned at[U];
            find(x, t0, at);
            fetch(l, at, kv, vv);
          }
          float s[U], mn = m;
#pragma unroll
          for (int u = 0; u < U; ++u) {
            float k[8];
            load8(reinterpret_cast<const bf16*>(&kv[u]), k);
            s[u] = score(k, t0 + (u * WAVES + wave) * 8 + tg < k1);
            mn = fmaxf(mn, s[u]);
          }
          const float top_s = mn == -INFINITY ? 0.f : mn;  // (scores that are not numbers are no maximum, and come through the exponentials)
          const float keep = exp2f(m - top_s);
          m = mn;
          sum *= keep;
#pragma unroll
          for (int j = 0; j < 8; ++j) o[j] *= keep;
#pragma unroll
          for (int u = 0; u < U; ++u) {
            const float e = exp2f(s[u] - top_s);
            float v[8];
            load8(reinterpret_cast<const bf16*>(&vv[u]), v);
            sum += e;
#pragma unroll
            for (int j = 0; j < 8; ++j) o[j] += e * v[j];
          }
        }
        // the step's own token, in the last span; then the wave's eight groups of lanes to their common maximum
        const bool own = x.sp == splits - 1 && wave == 0 && tg == 0;
        float kn[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) kn[j] = qkv[1][sub * 8 + j];
        const float sn = score(kn, own), mw = lanes_max(fmaxf(m, sn));
        const float top_w = mw == -INFINITY ? 0.f : mw, keep = exp2f(m - top_w), en = exp2f(sn - top_w);
        sum = groups_sum(sum * keep + en);
#pragma unroll
        for (int j = 0; j < 8; ++j) o[j] = groups_sum(o[j] * keep + en * qkv[2][sub * 8 + j]);
        if (lane < 8) {
#pragma unroll
          for (int j = 0; j < 8; ++j) part[wave][sub * 8 + j] = o[j];
          if (lane == 0) part[wave][D] = mw, part[wave][D + 1] = sum;
        }
        __syncthreads();
        if (tid < D) {
          float M = -INFINITY, S = 0.f, O = 0.f;
#pragma unroll
          for (int i = 0; i < WAVES; ++i) M = fmaxf(M, part[i][D]);
#pragma unroll
          for (int i = 0; i < WAVES; ++i) {
            const float e = M == -INFINITY ? 0.f : exp2f(part[i][D] - M);
            S += part[i][D + 1] * e;
            O += part[i][tid] * e;
          }
          if (splits == 1) {
            send(pa + (long)b * H + h * D + tid, O / S, tag);
          } else {
            u64* p = ps + (long)it * (D + 2);
            send(p + tid, O, tag);
            if (tid == 0) send(p + D, M, tag);
            if (tid == 1) send(p + D + 1, S, tag);
          }
        }
        if (it + N < items) __syncthreads();  // (qkv and part are used again)
      }
      if (splits > 1) {
        for (int it = me; it < items; it += N) {
          if (it % splits) continue;  // the first span's workgroup adds them
          float* buf = &hs[0][0];
          gather_f32(buf, ps + (long)it * (D + 2), splits * (D + 2), tag, wait);
          __syncthreads();
          if (tid < D) {
            float M = -INFINITY, S = 0.f, O = 0.f;
            for (int s = 0; s < splits; ++s) M = fmaxf(M, buf[s * (D + 2) + D]);
            for (int s = 0; s < splits; ++s) {
              const float e = exp2f(buf[s * (D + 2) + D] - M);  // (the step's own token is in one of them: M is finite)
              S += buf[s * (D + 2) + D + 1] * e;
              O += buf[s * (D + 2) + tid] * e;
            }
            send(pa + (long)(it / splits) * D + tid, O / S, tag);
          }
          __syncthreads();
        }
      }
      // ---- output projection
      gather_f32(as[0], pa, g.B * H, tag, wait);
      __syncthreads();
      auto out_of = [&](const Rows<KC, UO>& r, float bias, int v) __attribute__((always_inline)) {
#pragma unroll ROWS == 1 ? 1 : 2
        for (int b = 0; b < ROWS; ++b) {
          float x[KC][4];
          read_row(as[b], lane, x);
          const float s = dots(r.w, x, lane) + bias;
          const int o = v * NO + WAVES * lane + wave;
          if (b < g.B && lane < UO && WAVES * lane + wave < NO) send(px + (long)b * H + o, xs[b][o] + s, tag);
        }
      };
      out_of(wo, bo, me);
      wu.load(w.wu, H, me * NF, NF, wave, lane);
      norm_of(w.n2w, w.n2b);
      const float bu = bias_of(w.bu, me * NF, NF);
      for (int v = me + N; v < PARTS; v += N) {
        Rows<KC, UO> r;
        r.load(w.wo, H, v * NO, NO, wave, lane);
        out_of(r, bias_of(w.bo, v * NO, NO), v);
      }
      // ---- up
      gather_f32(xs[0], px, g.B * H, tag, wait);
      __syncthreads();
      auto up_of = [&](const Rows<KC, UF>& r, float bias, int share) __attribute__((always_inline)) {
#pragma unroll ROWS == 1 ? 1 : 2
        for (int b = 0; b < ROWS; ++b) {
          float x[KC][4];
          read_row(xs[b], lane, x);
          layernorm(x, nw, nb, g.eps);
          const float s = dots(r.w, x, lane) + bias;
          if (b < g.B && lane < UF && WAVES * lane + wave < NF) ups[b][WAVES * lane + wave] = gelu(s);
        }
        __syncthreads();
        if (tid < g.B * WF) {  // three to a word, rounded as they ever were between the two products
          const int b = tid / WF, i = tid - b * WF;
          u64 v = (u64)(tag & 0xffffu) << 48;
#pragma unroll
          for (int j = 0; j < 3; ++j) v |= (u64)f2bf(ups[b][3 * i + j]) << (16 * j);
          put_word(ph + ((long)b * PARTS + share) * WF + i, v);
        }
        if (N < PARTS) __syncthreads();  // (ups is used again)
      };
      up_of(wu, bu, me);
      wd.load(w.wd, me * NO, wave, lane);
      const float bd = bf2f(global(w.bd)[me * NO + tid % NO]);
      for (int v = me + N; v < PARTS; v += N) {
        Rows<KC, UF> r;
        r.load(w.wu, H, v * NF, NF, wave, lane);
        up_of(r, bias_of(w.bu, v * NF, NF), v);
      }
      // ---- down
      gather<16>(ph, g.B * PARTS * WF, tag, wait, [&](int i, u64 v) {
        const int b = i / (PARTS * WF), k = i - b * PARTS * WF, o = k % WF * 3;
        float* dst = hs[b] + k / WF * NF + o;
#pragma unroll
        for (int j = 0; j < 3; ++j)
          if (o + j < NF) dst[j] = bf2f((bf16)(v >> (16 * j)));
      });
      __syncthreads();
      auto down_of = [&](const Down<KC, UD>& r, float bias, int v) __attribute__((always_inline)) {
#pragma unroll ROWS == 1 ? 1 : 2
        for (int b = 0; b < ROWS; ++b) {
#pragma unroll
          for (int u = 0; u < UD; ++u) {
            const int i = WAVES * u + wave;
            float x[KC][4];
            read_row(hs[b] + (min(i, ND - 1) % R) * H, lane, x);
            b4 one[1][KC];
#pragma unroll
            for (int c = 0; c < KC; ++c) one[0][c] = r.w[u][c];
            const float s = dots(one, x, lane);
            if (b < g.B && lane == 0 && i < ND) red[b][i] = s;
          }
        }
        __syncthreads();
        if (tid < g.B * NO) {
          const int b = tid / NO, o = tid - b * NO;
          float s = bias + xs[b][v * NO + o];
#pragma unroll
          for (int q = 0; q < R; ++q) s += red[b][o * R + q];
          send(py + (long)b * H + v * NO + o, s, tag);
        }
        if (N < PARTS) __syncthreads();  // (red is used again)
      };
      down_of(wd, bd, me);
      const int next = min(l + 1, g.L - 1);
      const LayerW& n = layers[next];
      wq.load(n.wqkv, H, me * NQ, NQ, wave, lane);
      norm_of(n.n1w, n.n1b);
      bq = bias_of(n.bqkv, me * NQ, NQ);
      fetch(next, at0, kv0, vv0);
      for (int v = me + N; v < PARTS; v += N) {
        Down<KC, UD> r;
        r.load(w.wd, v * NO, wave, lane);
        down_of(r, bf2f(global(w.bd)[v * NO + tid % NO]), v);
      }
    }
    // ---- the words that this step has not written (nobody waits for them)
    {
      late = peek(&ctl->late) != 0;
      const unsigned last = base + g.L;
      auto age = [&](u64* p, int from, int to, u64 v) __attribute__((always_inline)) {
        for (int i = from + me * THREADS + tid; i < to; i += N * THREADS) put_word(p + i, v);
      };
      const u64 v = (u64)last << 32;
      age(pq, g.B * 3 * H, MAX_ROWS * 3 * H, v);
      age(pa, g.B * H, MAX_ROWS * H, v);
      age(px, g.B * H, MAX_ROWS * H, v);
      age(py, g.B * H, MAX_ROWS * H, v);
      age(ph, g.B * PARTS * WF, MAX_ROWS * PARTS * WF, (u64)(last & 0xffffu) << 48);
      age(ps, splits > 1 ? items * (D + 2) : 0, PARTS * (D + 2), v);
    }
    // ---- the final norm: row b by whoever holds share b
    for (int v = me; v < g.B; v += N) {
      gather_f32(as[v], py + (long)v * H, H, base + g.L, wait);
      __syncthreads();
      if (wave == 0) {
        norm_of(g.nw, g.nb);
        float x[KC][4];
        read_row(as[v], lane, x);
        layernorm(x, nw, nb, g.eps);
        late |= peek(&ctl->late) != 0;
#pragma unroll
        for (int c = 0; c < KC; ++c) {
          bf16 o[4];
#pragma unroll
          for (int j = 0; j < 4; ++j) o[j] = late ? (bf16)0x7fc0 : f2bf(x[c][j]);
          *reinterpret_cast<uint2*>(g.out + (long)v * H + c * 256 + lane * 4) = make_uint2(o[0] | ((unsigned)o[1] << 16), o[2] | ((unsigned)o[3] << 16));
        }
      }
    }
  }
  // ---- the last one out readies the workspace for the next step
  __syncthreads();
  if (tid != 0) return;
  const unsigned out = 1u + (late ? 1u << 16 : 0u);
  const unsigned left = out + __hip_atomic_fetch_add(&ctl->left, out, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if ((left & 0xffffu) == gridDim.x) {
    if (left >> 16 && g.lost != nullptr) __hip_atomic_store(g.lost, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    auto put = [](unsigned* p, unsigned v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
    put(&ctl->base, base + g.L);
    put(&ctl->late, 0u);
    put(&ctl->left, 0u);
    put(&ctl->gate, 0u);
  }
}

const bf16* row_ptr(const at::Tensor& t, int64_t rows, int64_t cols, const char* what) {
  LLMCTL_CHECK(t.is_cuda() && t.is_contiguous() && t.scalar_type() == at::kBFloat16 && t.numel() == rows * cols &&
                   (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0,
               "decode_layers: ", what, ": contiguous, aligned bf16 of ", rows, " x ", cols);
  return bf_ptr(t);
}

}  // namespace

int64_t decode_layers_words(int64_t hidden) {  // 8-byte words of a workspace
  return (int64_t)sizeof(Control) / 8 + MAX_ROWS * hidden * (3 + 1 + 1 + R + 1) + (int64_t)PARTS * (D + 2);
}

// The final norm's rows [B, H] of a decode step: ``w`` holds per layer the attention norm (weight, bias), QKV, output projection, MLP norm, up and
// down (weight, bias each), then the final norm.  k, v: the cache [L, blocks, block, heads, 64]; workspace: int64 [decode_layers_words], zero
// before its first step and used by one step at a time.  lost: pinned host memory, set to 1 by a step whose waits ran out (``spins`` tries), whose rows are NaN.
at::Tensor decode_layers(const at::Tensor& ids, const at::Tensor& positions, const at::Tensor& slots, const at::Tensor& block_tables,
                         const at::Tensor& ctx, const at::Tensor& table, const at::Tensor& ptable, at::TensorList w, at::Tensor k, at::Tensor v,
                         double eps, at::Tensor workspace, int64_t workgroups, int64_t gate_us, const c10::optional<at::Tensor>& lost, int64_t spins) {
  const int64_t B = ids.numel(), H = table.size(1), L = ((int64_t)w.size() - 2) / 12, heads = H / D;
  LLMCTL_CHECK(table.dim() == 2 && H % 256 == 0 && H >= 256 && H <= 1024 && B >= 1 && B <= MAX_ROWS && L >= 1 && L <= MAX_LAYERS && (int64_t)w.size() == 12 * L + 2,
               "decode_layers: up to 4 rows, 32 layers of 256 to 1024 columns");
  LLMCTL_CHECK(workgroups >= 1 && workgroups <= PARTS, "decode_layers: 1 to 128 workgroups");
  LLMCTL_CHECK(gate_us >= 0 && gate_us <= 1000000, "decode_layers: the gate's time for a round");
  LLMCTL_CHECK(spins >= 1 && spins <= (1 << 21), "decode_layers: 1 to 2^21 tries of a wait");
  LLMCTL_CHECK(!lost.has_value() || (lost->device().is_cpu() && lost->is_pinned() && lost->scalar_type() == at::kInt && lost->numel() == 1),
               "decode_layers: lost: one int32 of pinned memory");
  auto ints = [&](const at::Tensor& t, at::ScalarType type, int64_t n) {
    return t.is_cuda() && t.is_contiguous() && t.scalar_type() == type && t.numel() == n;
  };
  LLMCTL_CHECK(ints(ids, at::kLong, B) && ints(slots, at::kLong, B) && ints(positions, at::kInt, B) && ints(ctx, at::kInt, B) && block_tables.dim() == 2 &&
                   ints(block_tables, at::kInt, B * block_tables.size(1)) && block_tables.size(1) >= 1,
               "decode_layers: ids, slots int64 [B], positions, context lengths int32 [B], block tables int32 [B, n]");
  LLMCTL_CHECK(ints(workspace, at::kLong, decode_layers_words(H)), "decode_layers: workspace");
  for (const at::Tensor* c : {&k, &v})
    LLMCTL_CHECK(c->is_cuda() && c->is_contiguous() && c->scalar_type() == at::kBFloat16 && c->dim() == 5 && c->size(0) == L && c->size(3) == heads &&
                     c->size(4) == D && c->sizes() == k.sizes() && (reinterpret_cast<uintptr_t>(c->data_ptr()) & 15) == 0,
                 "decode_layers: cache bf16 [L, blocks, block, heads, 64]");
  LLMCTL_CHECK(k.numel() / L / 8 < ((int64_t)1 << 32), "decode_layers: a layer's cache below 64 GB");
  const c10::DeviceGuard guard(ids.device());
  StepArgs a = {};
  const int64_t F = R * H;
  for (int64_t l = 0; l < L; ++l) {
    const at::Tensor* t = &w[12 * l];
    a.layer[l] = LayerW{row_ptr(t[0], 1, H, "norm"), row_ptr(t[1], 1, H, "norm"), row_ptr(t[2], 3 * H, H, "qkv"), row_ptr(t[3], 1, 3 * H, "qkv bias"),
                        row_ptr(t[4], H, H, "output"), row_ptr(t[5], 1, H, "output bias"), row_ptr(t[6], 1, H, "norm"), row_ptr(t[7], 1, H, "norm"),
                        row_ptr(t[8], F, H, "up"), row_ptr(t[9], 1, F, "up bias"), row_ptr(t[10], H, F, "down"), row_ptr(t[11], 1, H, "down bias")};
  }
  a.nw = row_ptr(w[12 * L], 1, H, "final norm"), a.nb = row_ptr(w[12 * L + 1], 1, H, "final norm");
  a.table = row_ptr(table, table.size(0), H, "embedding"), a.ptable = row_ptr(ptable, ptable.size(0), H, "positions");
  at::Tensor out = at::empty({B, H}, table.options());
  a.kc = bf_mut(k), a.vc = bf_mut(v), a.out = bf_mut(out);
  a.ids = ids.data_ptr<int64_t>(), a.slots = slots.data_ptr<int64_t>();
  a.pos = positions.data_ptr<int32_t>(), a.bt = block_tables.data_ptr<int32_t>(), a.ctx = ctx.data_ptr<int32_t>();
  a.wait = Wait{reinterpret_cast<Control*>(workspace.data_ptr<int64_t>()), (int)spins};
  if (lost.has_value()) {
    void* p = nullptr;
    LLMCTL_HIP_CHECK(hipHostGetDevicePointer(&p, lost->data_ptr<int32_t>(), 0));
    a.lost = static_cast<unsigned*>(p);
  }
  a.ws = reinterpret_cast<u64*>(workspace.data_ptr<int64_t>()) + sizeof(Control) / 8;
  a.rows = table.size(0), a.prows = ptable.size(0), a.layer_stride = k.numel() / L;
  a.eps = (float)eps, a.scale = 0.125f;
  a.L = (int)L, a.B = (int)B, a.heads = (int)heads, a.block = (int)k.size(2), a.max_blocks = (int)block_tables.size(1), a.gate_ticks = (int)gate_us * 100;
  const dim3 grid((unsigned)workgroups);
  auto s = stream();
  auto go = [&](auto kc) {
    constexpr int KC = decltype(kc)::value;
    if (B == 1) hipLaunchKernelGGL((decode_layers_kernel<KC, 1>), grid, dim3(THREADS), 0, s, a);
    else if (B == 2) hipLaunchKernelGGL((decode_layers_kernel<KC, 2>), grid, dim3(THREADS), 0, s, a);
    else hipLaunchKernelGGL((decode_layers_kernel<KC, MAX_ROWS>), grid, dim3(THREADS), 0, s, a);
  };
  if (H == 256) go(std::integral_constant<int, 1>{});
  else if (H == 512) go(std::integral_constant<int, 2>{});
  else if (H == 768) go(std::integral_constant<int, 3>{});
  else go(std::integral_constant<int, 4>{});
  return out;
}

TORCH_LIBRARY_IMPL(llmctl, CUDA, m) { m.impl("decode_layers", &decode_layers); }

}  // namespace llmctl
