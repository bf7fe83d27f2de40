// Grouped expert products on tiles of up to 288 rows x 128 columns (moe.hip), K in 128s from 256 on.
//
// The loop and what bounds it: wide_tiles.h; the tile is as large as leaves the chip full.
// Row tiles have 256 rows but the last one of an expert, which takes what is left, 33 to 288: a power of two of tokens gives an expert a multiple of 256 copies, give or
// take the square root, and with tiles of 256 half of the experts had one more tile, of a few rows (2048 tokens, 8 experts, top 2: 16 row tiles for 20).  Tiles of at
// most 128 rows are dealt out last, to the CUs that are done first.
// us, tiles of 128 x 128 / these, kernel times after the caches are written over: width 2048, 8 experts of 1024, up (gated) and down, 459 tokens 47, 26 / 39, 20, 1021 56, 31 / 50, 24, 3035 86, 49 /
// 81, 42; erf GELUs 2911 tokens 54, 41 / 50, 42, 3011 55, 48 / 54, 42; width 4096, 8 of 1408, gated, 1511 tokens 132, 70 / 136, 58; 32 experts of 512, width 1024, top 4, 1699 tokens 28, 23 / 28, 22, but
// gated 2612 tokens, whose tiles make two rounds of one and a half, 43, 28 / 57, 30 (moe_wide_pays leaves them to the others).
#pragma once
#include "wide_tiles.h"

namespace llmctl_hybrid {
namespace {
// (The activation is a parameter: with a branch on it in the 144 places of an epilogue the instructions came from memory, 10 us a launch.)
template <int MODE>
__global__ __launch_bounds__(256, 1) __attribute__((amdgpu_waves_per_eu(1, 1))) void moe_wide_kernel(TileArgs g) {
  using namespace llmctl::wide;
  using llmctl::A_HI;
  using llmctl::A_LO;
  using llmctl::B_H0;
  using llmctl::f32x4_t;
  using llmctl::HALF;
  using llmctl::K_;
  using llmctl::swr;
  using llmctl::tile_pos;
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
        for (int q = 0; q < 4; ++q) x[j][q] = expert_act(1, bf16_of(a[j + 2][q]), bf16_of(a[j][q]));
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
