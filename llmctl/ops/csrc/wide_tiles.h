// Products x w^T, both operands K-contiguous, on tiles of up to 288 rows x 128 columns, K in 128s from 256 on: four waves, one per SIMD, 128 x 64 of a tile each, a ring of
// three K-tiles of 64 in LDS filled by LDS-DMA, the schedule of gemm_tall.hip (which see).  A lane's DMA offset is its row's, so gathered rows cost nothing.  Rows 256 to 287
// of a tile are a ninth block of 16 rows of each wave, 8 MFMAs a K-tile more; tiles of at most 128 rows run half the MFMAs and loads, four K-tiles ahead.
// Bound: the lines that a CU can have on their way (some 90 of 128 bytes, whatever the ring holds): a K-tile of 256 rows is 384 lines, 0.7 us where they come from L2 and
// 1.0 where one operand comes from HBM, against 0.43 us of MFMAs.
// Shared by the routed experts (hybrid/moe_wide.h) and gemm_rows.hip.
#pragma once
#include "gemm64_tiles.h"

namespace llmctl {
namespace {
namespace wide {
using frag8 = attn::bf16x8_t;

constexpr int ROWS = 288, COLS = 128, A_X = 3;  // A_X: the image of rows 256 on, behind the three halves
constexpr int SLOT = 3 * HALF + 4096, SLOT_H = 2 * HALF;  // a K-tile: A_lo, A_hi, B, A_x; of a half tile: A_lo, B

// 16 wait states between the MFMAs (or zeroes) that wrote a row block's accumulators and what reads them
__device__ __forceinline__ void fence_row(f32x4_t (&a)[4]) { asm volatile("s_nop 7\n\ts_nop 7" : "+a"(a[0]), "+a"(a[1]), "+a"(a[2]), "+a"(a[3])); }

struct Tile {
  const unsigned short* a;  // what the DMA offsets of the tile's rows start from
  const unsigned short* b;  // of B's
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
    for (int i = 0; i < 4; ++i) bdma16(rb, vb[i], (unsigned)t * (TK * 2), attn::lds_addr(smem) + wave * 1024 + t * slot + img + i * 4096);
}

// MB row blocks of 16 a wave: 8, or 9 with rows from 256 on.  va: the thread's DMA offsets of A's pieces (lo 4, hi 4, x 1), vb of B's.
template <int MB>
__device__ __forceinline__ void run(const Tile& t_, const unsigned (&va)[9], const unsigned (&vb)[4], unsigned char* smem, f32x4_t (&acc)[9][4]) {
  constexpr bool X = MB == 9;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), wr = wave >> 1, wc = wave & 1;
  const int KT = t_.K / TK;  // even, >= 4
  i32x4_t ra = make_rsrc(t_.a), rb = make_rsrc(t_.b);
  asm volatile("s_nop 7" : "+s"(ra), "+s"(rb));  // lane-read scalars to the first DMA piece that uses them
  const unsigned lds0 = attn::lds_addr(smem) + wave * 1024;
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
  const unsigned lds0 = attn::lds_addr(smem) + wave * 1024;
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

}  // namespace
}  // namespace llmctl
