// Grouped expert products on tiles of up to 288 rows x 128 columns (moe.hip), K in 128s from 256 on.
//
// Bound: the lines that a CU can have on their way (some 90 of 128 bytes, whatever the ring holds): a K-tile of 256 rows is 384 lines, 0.7 us where they come from L2 and 1.0
// where an expert's weights come from HBM, against 0.43 us of MFMAs; so the tile is as large as leaves the chip full.  Four waves, one per SIMD, 128 x 64 of a tile each, a
// ring of three K-tiles of 64 in LDS filled by LDS-DMA (the schedule of gemm_tall.hip, which see; here both operands are K-contiguous, and a lane's DMA offset is its row's, so
// that gathered rows cost nothing).
// Row tiles have 256 rows but the last one of an expert, which takes what is left, 33 to 288: a power of two of tokens gives an expert a multiple of 256 copies, give or
// take the square root, and with tiles of 256 half of the experts had one more tile, of a few rows (2048 tokens, 8 experts, top 2: 16 row tiles for 20).  Rows 256 to 287
// are a ninth block of 16 rows of each wave, 8 MFMAs a K-tile more.  Tiles of at most 128 rows run half the MFMAs and loads, four K-tiles ahead; they are dealt out last, to
// the CUs that are done first.
// us, tiles of 128 x 128 / these: width 2048, 8 experts of 1024, up (gated) and down, 459 tokens 36.5, 21.7 / 25.4, 15.0, 1021 46.9, 27.0 / 34.8, 20.3, 3035 83, 47 / 66, 39;
// without gates 3011 tokens 49, 46 / 33, 36; width 4096, 8 of 1408, gated, 1511 tokens 118, 65 / 100, 54; 32 experts, width 1024, 1699 tokens 32, 29 / 26, 24, but gated
// 2612 tokens, a third of whose tiles start a new round, 70, 39 / 78, 39.
#pragma once
#include "gemm64_tiles.h"

namespace llmctl_hybrid {
namespace {
namespace wide {
using llmctl::A_HI;
using llmctl::A_LO;
using llmctl::B_H0;
using llmctl::bar;
using llmctl::bdma16;
using llmctl::f32x4_t;
using llmctl::frag;
using llmctl::g4w_pair;
using llmctl::g4w_pair_dma;
using llmctl::HALF;
using llmctl::i32x4_t;
using llmctl::K_;
using llmctl::make_rsrc;
using llmctl::swr;
using llmctl::tile_pos;
using llmctl::wait_vm;
using frag8 = llmctl::attn::bf16x8_t;

constexpr int ROWS = 288, COLS = 128, TK = 64, A_X = 3;  // A_X: the image of rows 256 on, behind the three halves
constexpr int SLOT = 3 * HALF + 4096, SLOT_H = 2 * HALF;  // a K-tile: A_lo, A_hi, B, A_x; of a half tile: A_lo, B

// 16 wait states between the MFMAs (or zeroes) that wrote a row block's accumulators and what reads them
__device__ __forceinline__ void fence_row(f32x4_t (&a)[4]) { asm volatile("s_nop 7\n\ts_nop 7" : "+a"(a[0]), "+a"(a[1]), "+a"(a[2]), "+a"(a[3])); }

struct Tile {
  const bf16_t* a;  // row r of the tile at a + row_of(r) * lda
  const bf16_t* b;  // the expert's weight
  int K;
};

// B's first N K-tiles go out before the rows of A are known (a load of the copies' list).
template <int N>
__device__ __forceinline__ void first_b(const Tile& t_, const unsigned (&vb)[4], unsigned char* smem, int slot, int img) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  i32x4_t rb = make_rsrc(t_.b);
  asm volatile("s_nop 7" : "+s"(rb));
#pragma unroll
  for (int t = 0; t < N; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) bdma16(rb, vb[i], (unsigned)t * (TK * 2), llmctl::attn::lds_addr(smem) + wave * 1024 + t * slot + img + i * 4096);
}

// MB row blocks of 16 a wave: 8, or 9 with rows from 256 on.  va: the thread's DMA offsets of A's pieces (lo 4, hi 4, x 1), vb of B's.
template <int MB>
__device__ __forceinline__ void run(const Tile& t_, const unsigned (&va)[9], const unsigned (&vb)[4], unsigned char* smem, f32x4_t (&acc)[9][4]) {
  constexpr bool X = MB == 9;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), wr = wave >> 1, wc = wave & 1;
  const int KT = t_.K / TK;  // even, >= 4
  i32x4_t ra = make_rsrc(t_.a), rb = make_rsrc(t_.b);
  asm volatile("s_nop 7" : "+s"(ra), "+s"(rb));  // lane-read scalars to the first DMA piece that uses them
  const unsigned lds0 = llmctl::attn::lds_addr(smem) + wave * 1024;
  auto issue = [&](auto kind_c, int t, int slot, auto n_c) __attribute__((always_inline)) {
    constexpr int kind = decltype(kind_c)::value, n = decltype(n_c)::value;
#pragma unroll
    for (int i = 0; i < n; ++i) {
      const unsigned l = lds0 + slot + kind * HALF + i * 4096, so = (unsigned)t * (TK * 2);
      if constexpr (kind == B_H0) bdma16(rb, vb[i], so, l);
      else bdma16(ra, va[kind == A_LO ? i : kind == A_HI ? 4 + i : 8], so, l);
    }
  };
  frag8 a_lo[4][2], a_hi[4][2], a_x[2], b[2][4][2];
#pragma unroll
  for (int i = 0; i < MB; ++i) {
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    fence_row(acc[i]);
  }
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    issue(K_<A_LO>{}, t, t * SLOT, K_<4>{});
    issue(K_<A_HI>{}, t, t * SLOT, K_<4>{});
    if constexpr (X) issue(K_<A_X>{}, t, t * SLOT, K_<1>{});
  }
  issue(K_<A_LO>{}, 2, 2 * SLOT, K_<2>{});
  wait_vm<X ? 16 : 14>();  // B, A_lo(0)
  bar();
#pragma unroll
  for (int ks = 0; ks < 2; ++ks)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      a_lo[i][ks] = frag<false>(smem + A_LO * HALF, wr * 64 + 16 * i, ks, lane);
      b[0][i][ks] = frag<false>(smem + B_H0 * HALF, wc * 64 + 16 * i, ks, lane);
    }
  wait_vm<X ? 7 : 6>();  // A_hi(0) (A_x(0)), A_lo(1)
  __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
  bar();

  // as in gemm_tall.hip: DMA 2 = both phases issue, 1 = only the first, 0 = none; WAIT: vmcnt at the end (-1: last).  A_x(t) goes where A_hi(t) does.
  auto ktile = [&](auto par_c, auto dma_c, auto wait_c, int t, int s0, int s1, int s2) __attribute__((always_inline)) {
    constexpr int P = decltype(par_c)::value, DMA = decltype(dma_c)::value, WAIT = decltype(wait_c)::value;
    constexpr bool NEXT = WAIT >= 0;
    const unsigned so0 = (unsigned)(t + 2) * (TK * 2), l0 = lds0 + s2;
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      const int ks = q >> 3, i = (q >> 1) & 3, j = (q & 1) * 2;
      if (DMA >= 1 && (q % 3 == 0 || (X && q == 14))) {
        const int n = q == 14 ? 6 : q / 3, kind = n < 2 ? A_LO : n < 6 ? A_HI : A_X, pc = n < 2 ? 2 + n : n < 6 ? n - 2 : 0;
        g4w_pair_dma(acc[i][j], acc[i][j + 1], a_lo[i][ks], b[P][j][ks], b[P][j + 1][ks], va[n < 2 ? pc : n < 6 ? 4 + pc : 8], ra, so0, l0 + kind * HALF + pc * 4096);
      } else {
        g4w_pair(acc[i][j], acc[i][j + 1], a_lo[i][ks], b[P][j][ks], b[P][j + 1][ks]);
      }
      if (q < 8) a_hi[q & 3][q >> 2] = frag<false>(smem + s0 + A_HI * HALF, wr * 64 + 16 * (q & 3), q >> 2, lane);
      else if (NEXT && q < 12) b[P ^ 1][q & 3][0] = frag<false>(smem + s1 + B_H0 * HALF, wc * 64 + 16 * (q & 3), 0, lane);
      else if (X && q >= 12 && q < 14) a_x[q - 12] = frag<false>(smem + s0 + A_X * HALF, wr * 16, q - 12, lane);
    }
    const unsigned so1 = (unsigned)(t + 3) * (TK * 2), l1 = lds0 + s0;
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      const int ks = q >> 3, i = (q >> 1) & 3, j = (q & 1) * 2;
      if (DMA == 2 && q % 3 == 0) {
        const int n = q / 3, kind = n < 4 ? B_H0 : A_LO, pc = n & 3;
        g4w_pair_dma(acc[4 + i][j], acc[4 + i][j + 1], a_hi[i][ks], b[P][j][ks], b[P][j + 1][ks], n < 4 ? vb[pc] : va[pc], n < 4 ? rb : ra, so1,
                     l1 + kind * HALF + pc * 4096);
      } else {
        g4w_pair(acc[4 + i][j], acc[4 + i][j + 1], a_hi[i][ks], b[P][j][ks], b[P][j + 1][ks]);
      }
      if (NEXT && q < 8) a_lo[q & 3][q >> 2] = frag<false>(smem + s1 + A_LO * HALF, wr * 64 + 16 * (q & 3), q >> 2, lane);
      else if (NEXT && q < 12) b[P ^ 1][q & 3][1] = frag<false>(smem + s1 + B_H0 * HALF, wc * 64 + 16 * (q & 3), 1, lane);
    }
    if constexpr (X) {
#pragma unroll
      for (int q = 0; q < 4; ++q) g4w_pair(acc[8][(q & 1) * 2], acc[8][(q & 1) * 2 + 1], a_x[q >> 1], b[P][(q & 1) * 2][q >> 1], b[P][(q & 1) * 2 + 1][q >> 1]);
    }
    if constexpr (NEXT) {
      wait_vm<NEXT ? WAIT : 0>();
      __builtin_amdgcn_s_waitcnt(0xC07F);
      bar();
    }
  };
  int s0 = 0, s1 = SLOT, s2 = 2 * SLOT;
  auto turn = [&]() __attribute__((always_inline)) {
    const int s = s0;
    s0 = s1, s1 = s2, s2 = s;
  };
  constexpr int ALL = X ? 11 : 10, LAST = X ? 5 : 4;
  for (int t = 0; t < KT - 4; t += 2) {
    ktile(K_<0>{}, K_<2>{}, K_<ALL>{}, t, s0, s1, s2);
    turn();
    ktile(K_<1>{}, K_<2>{}, K_<ALL>{}, t + 1, s0, s1, s2);
    turn();
  }
  ktile(K_<0>{}, K_<2>{}, K_<ALL>{}, KT - 4, s0, s1, s2);
  turn();
  ktile(K_<1>{}, K_<1>{}, K_<LAST>{}, KT - 3, s0, s1, s2);
  turn();
  ktile(K_<0>{}, K_<0>{}, K_<0>{}, KT - 2, s0, s1, s2);
  turn();
  ktile(K_<1>{}, K_<0>{}, K_<-1>{}, KT - 1, s0, s1, s2);
#pragma unroll
  for (int i = 4; i < MB; ++i) fence_row(acc[i]);
}

// A tile of at most 128 rows: A_lo alone, its image row r the tile's row r; a ring of four K-tiles, one phase of 32 MFMAs each:
//   phase t   MFMA [a(t), b(t)]   read a, b(t+1)   issue A, B(t+4) (the slot of t, last read before the barrier ahead)   vmcnt(16): A, B(t+2) have landed
__device__ __forceinline__ void run_half(const Tile& t_, const unsigned (&va)[9], const unsigned (&vb)[4], unsigned char* smem, f32x4_t (&acc)[9][4]) {
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), wr = wave >> 1, wc = wave & 1;
  const int KT = t_.K / TK;
  i32x4_t ra = make_rsrc(t_.a), rb = make_rsrc(t_.b);
  asm volatile("s_nop 7" : "+s"(ra), "+s"(rb));
  const unsigned lds0 = llmctl::attn::lds_addr(smem) + wave * 1024;
  frag8 a[2][4][2], b[2][4][2];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    fence_row(acc[i]);
  }
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    if (t >= 2) {  // (B(0), B(1): first_b)
#pragma unroll
      for (int i = 0; i < 4; ++i) bdma16(rb, vb[i], (unsigned)t * (TK * 2), lds0 + t * SLOT_H + HALF + i * 4096);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) bdma16(ra, va[i], (unsigned)t * (TK * 2), lds0 + t * SLOT_H + i * 4096);
  }
  wait_vm<20>();  // A, B(0)
  bar();
#pragma unroll
  for (int ks = 0; ks < 2; ++ks)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      a[0][i][ks] = frag<false>(smem, wr * 64 + 16 * i, ks, lane);
      b[0][i][ks] = frag<false>(smem + HALF, wc * 64 + 16 * i, ks, lane);
    }
  wait_vm<16>();  // A, B(1)
  __builtin_amdgcn_s_waitcnt(0xC07F);
  bar();
  auto phase = [&](auto par_c, auto dma_c, auto wait_c, int t) __attribute__((always_inline)) {
    constexpr int P = decltype(par_c)::value, WAIT = decltype(wait_c)::value;
    constexpr bool DMA = decltype(dma_c)::value != 0, NEXT = WAIT >= 0;
    const unsigned so = (unsigned)(t + 4) * (TK * 2), l = lds0 + (t & 3) * SLOT_H;
    const unsigned char* next = smem + ((t + 1) & 3) * SLOT_H;
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      const int ks = q >> 3, i = (q >> 1) & 3, j = (q & 1) * 2;
      if (DMA && (q & 1)) {
        const int pc = (q >> 1) & 3;
        g4w_pair_dma(acc[i][j], acc[i][j + 1], a[P][i][ks], b[P][j][ks], b[P][j + 1][ks], q < 8 ? vb[pc] : va[pc], q < 8 ? rb : ra, so,
                     l + (q < 8 ? HALF : 0) + pc * 4096);
      } else {
        g4w_pair(acc[i][j], acc[i][j + 1], a[P][i][ks], b[P][j][ks], b[P][j + 1][ks]);
      }
      if constexpr (NEXT) {
        if (q < 8) b[P ^ 1][q & 3][q >> 2] = frag<false>(next + HALF, wc * 64 + 16 * (q & 3), q >> 2, lane);
        else a[P ^ 1][q & 3][(q - 8) >> 2] = frag<false>(next, wr * 64 + 16 * (q & 3), (q - 8) >> 2, lane);
      }
    }
    if constexpr (NEXT) {
      wait_vm<NEXT ? WAIT : 0>();
      __builtin_amdgcn_s_waitcnt(0xC07F);
      bar();
    }
  };
  for (int t = 0; t < KT - 4; t += 2) {
    phase(K_<0>{}, K_<1>{}, K_<16>{}, t);
    phase(K_<1>{}, K_<1>{}, K_<16>{}, t + 1);
  }
  phase(K_<0>{}, K_<0>{}, K_<8>{}, KT - 4);
  phase(K_<1>{}, K_<0>{}, K_<0>{}, KT - 3);
  phase(K_<0>{}, K_<0>{}, K_<0>{}, KT - 2);
  phase(K_<1>{}, K_<0>{}, K_<-1>{}, KT - 1);
#pragma unroll
  for (int i = 0; i < 4; ++i) fence_row(acc[i]);
}
}  // namespace wide

// silu(g) u; the hardware's exponential and reciprocal are good to an ulp, a result is rounded to 8 bits
__device__ __forceinline__ float silu_mul(float g, float u) { return g * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * g)) * u; }

// (The activation is a parameter: with a branch on it in the 144 places of an epilogue the instructions came from memory, 10 us a launch.)
template <int MODE>
__global__ __launch_bounds__(256, 1) __attribute__((amdgpu_waves_per_eu(1, 1))) void moe_wide_kernel(TileArgs g) {
  using namespace wide;
  __shared__ __attribute__((aligned(1024))) unsigned char smem[3 * SLOT];
  // the tiles of more than 128 rows, an equal run of them to each XCD, then the others
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), wr = wave >> 1, wc = wave & 1;
  int ent[3];  // lane m: row tile m (asked for with the numbers of tiles, not after them)
#pragma unroll
  for (int i = 0; i < 3; ++i) ent[i] = g.tiles[2 + 3 * min(lane, g.max_tiles - 1) + i];
  const int n_full = g.tiles[0], n_half = g.tiles[1], xcd = blockIdx.x & 7;
  int k = blockIdx.x >> 3, count = n_full, list = 0, x = xcd;
  int q8 = n_full * g.ntile >> 3, r8 = n_full * g.ntile & 7;
  if (k >= q8 + (x < r8)) {
    k -= q8 + (x < r8);
    count = n_half, list = n_full, x = 7 - xcd;
    q8 = n_half * g.ntile >> 3, r8 = n_half * g.ntile & 7;
    if (k >= q8 + (x < r8)) return;
  }
  const int tile = x * q8 + min(x, r8) + k;
  const int first = tile / (BAND * g.ntile) * BAND, in = tile - first * g.ntile, high = min(BAND, count - first);
  const int nt = in / high, mt = list + first + in - nt * high;
  int e, row0, rows;
  if (mt < 64) {
    e = __builtin_amdgcn_readlane(ent[0], mt), row0 = __builtin_amdgcn_readlane(ent[1], mt), rows = __builtin_amdgcn_readlane(ent[2], mt);
  } else {
    e = g.tiles[2 + 3 * mt], row0 = g.tiles[3 + 3 * mt], rows = g.tiles[4 + 3 * mt];
  }
  const bool half = rows <= 128;
  constexpr int CT = MODE == UP_GLU ? COLS / 2 : COLS;  // output columns of a tile
  const int c0 = nt * CT;
  // DMA offsets: piece i of an image holds its rows 32 i + tid / 8, chunk tid % 8 of a K-tile's eight at its swizzled place
  unsigned va[9], vb[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int ir = 32 * i + (tid >> 3);
    int row;
    if constexpr (MODE == UP_GLU) {  // of a wave's 64 columns the first half are gate rows, then the up rows of the same places
      row = (ir >> 5 & 1) * g.cols + c0 + (ir >> 6) * 32 + (ir & 31);
    } else {
      row = c0 + ir;
    }
    vb[i] = (unsigned)row * (unsigned)(g.ldw * 2) + (unsigned)(((tid & 7) ^ swr(ir)) << 4);
  }
  const Tile t{MODE == DOWN ? g.a + (long)row0 * g.lda : g.a, g.w.p[e], g.K};
  if (half) first_b<2>(t, vb, smem, SLOT_H, HALF);
  else first_b<3>(t, vb, smem, SLOT, B_H0 * HALF);
  const int kg = lane >> 4, i16 = lane & 15;
  auto row_of = [&](int i) __attribute__((always_inline)) { return i == 8 ? 256 + wr * 16 + i16 : wr * (half ? 64 : 128) + 16 * i + i16; };
  int orow[9];  // DOWN: where the lane's rows of the result go
#pragma unroll
  for (int i = 0; i < 9; ++i) {
    const int ir = 32 * (i & 3) + (tid >> 3);
    const int r = i == 8 ? 256 + (tid >> 3) : half ? ir : i < 4 ? tile_pos<A_LO>(ir) : tile_pos<A_HI>(ir);
    const int p = min(r, rows - 1);
    const unsigned row = MODE == DOWN ? (unsigned)p : (unsigned)(g.perm[row0 + p] / g.top);
    va[i] = row * (unsigned)(g.lda * 2) + (unsigned)(((tid & 7) ^ swr(i == 8 ? tid >> 3 : ir)) << 4);
    if constexpr (MODE == DOWN) orow[i] = g.perm[row0 + min(row_of(i), rows - 1)];
  }
  // lane holds [16 i + (l & 15)][16 j + 4 (l >> 4) + r] of its wave's part; 16 bytes to a lane: lanes of neighbouring groups swap halves of two column tiles
  auto out = [&](const f32x4_t (&a)[4], int i) __attribute__((always_inline)) {
    const int r = row_of(i);
    const long o = MODE == DOWN ? (long)orow[i] : (long)(row0 + r);
    auto put = [&](const float (&x0)[4], const float (&x1)[4], int c) __attribute__((always_inline)) {
      float v[8];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const auto s = __builtin_amdgcn_permlane16_swap(__float_as_uint(x0[q]), __float_as_uint(x1[q]), false, false);
        v[q] = __uint_as_float(s[0]);
        v[4 + q] = __uint_as_float(s[1]);
      }
      c += 16 * (kg & 1) + 8 * (kg >> 1);
      if (r < rows) Vec16<bf16_t>::store(g.out + o * g.cols + c, v);
    };
    float x[2][4];
    if constexpr (MODE == UP_GLU) {
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) x[j][q] = silu_mul(bf16_of(a[j][q]), bf16_of(a[j + 2][q]));
      put(x[0], x[1], c0 + wc * 32);
    } else {
#pragma unroll
      for (int jp = 0; jp < 2; ++jp) {
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int q = 0; q < 4; ++q) x[j][q] = MODE == DOWN ? a[2 * jp + j][q] : expert_act(MODE == UP_GELU ? 2 : 0, bf16_of(a[2 * jp + j][q]), 0.f);
        put(x[0], x[1], c0 + wc * 64 + 32 * jp);
      }
    }
  };
  auto whole = [&](auto mb_c) __attribute__((always_inline)) {
    constexpr int MB = decltype(mb_c)::value;
    f32x4_t acc[9][4];
    if constexpr (MB == 4) run_half(t, va, vb, smem, acc);
    else run<MB>(t, va, vb, smem, acc);
#pragma unroll
    for (int i = 0; i < MB; ++i) out(acc[i], i);
  };
  if (half) whole(K_<4>{});
  else if (rows <= 256) whole(K_<8>{});
  else whole(K_<9>{});
}

}  // namespace
}  // namespace llmctl_hybrid
