// Backward products on 256 x 128 tiles: data gradients dy W (W read K-major) and weight gradients dy^T x, bf16 in, for the sizes that leave the 256 x 256
// tiles of gemm64.hip short of workgroups.
//
// Bound: the MFMAs where the tiles fill the chip; below that the fill.  8192 x 768 is 96 tiles of 256 x 256 for 256 CUs and 192 of 256 x 128; a 768 x 3072
// weight gradient over 8192 tokens is 36, cut in K to get to 144 at four partial sums an entry, against 72 and three.
//
// Layout: four waves, one per SIMD, 128 x 64 each (acc 8 x 4), a ring of three K-tiles of 64 in LDS (48 KB each: the images A_lo, A_hi and B_h0 of
// gemm64_tiles.h) filled by LDS-DMA.  A K-tile is two phases of 32 MFMAs; fragments are read in the phase before their use, one to a statement of two MFMAs,
// b twice, by K-tile parity; the DMA pieces go out every third statement; one barrier:
//   P0(t)  MFMA rows 0-3 [a_lo(t), b(t)]   read a_hi(t), b(t+1) first half      issue A_lo(t+2) second half, A_hi(t+2)
//   P1(t)  MFMA rows 4-7 [a_hi(t), b(t)]   read a_lo(t+1), b(t+1) second half   issue B(t+3), A_lo(t+3) first half
//          vmcnt(10) + barrier: B, A_lo(t+2) and A_hi(t+1) have landed
// Each piece's slot was last read before the barrier that precedes it: B, A_lo(t) by P1(t-1), A_hi(t) by P0(t).  The last three K-tiles issue nothing that does
// not exist and wait for what is left.  Pieces eight to a half phase queued up in the address unit (a 768 x 3072 product over 8192 tokens in 72 workgroups: 89.2
// us, so 79.7); twelve in P1, a longer time to arrive, 106.7.
// LDS moves (128 + 64) x 64 operand entries per wave and K-tile and takes in the 48 KB of another: 1.1 times the MFMAs' 1024 clocks at 128 bytes a clock, where
// the 256 x 256 tiles are at 0.75; on a full chip those are a fifth faster (8192 x 4096 x 4096: 190 us, here 234).  gemm_tall_splits weighs the two.
// Measured on one MI355X, us, 256 x 256 tiles / these: data gradients of 8192 tokens 768 x 768 21.6 / 14.0, 2304 x 768 44.7 / 29.5, 3072 x 768 52.6 / 46.5,
// 2048 x 4096 x 4096 71.0 / 54.3; weight gradients 768 x 768 30.1 / 23.1, 2304 x 768 42.3 / 35.9, 768 x 3072 56.5 / 46.2.
#include "gemm_tall.h"
#include "gemm64_tiles.h"

#include <functional>
#include <queue>

namespace llmctl {
using namespace attn;
namespace {

constexpr int TALL_N = 128, SLOT = 3 * HALF;
enum : int { OUT_STORE = 0, OUT_ADD = 1, OUT_STORE_F32 = 2, OUT_ADD_F32 = 3 };

struct TallArgs {
  const unsigned short* a;
  const unsigned short* b;
  void* c;
  float* ws;  // [splits][M][N] fp32 partial sums (splits > 1), then with a bias [splits][M]
  void* bias;     // BIAS: [M], of c's type
  int bias_add;
  long lda, ldb, ldc;
  int M, N, K;
  int tiles_m, tiles_n, splits;
};

// 16 wait states between what wrote four rows of accumulators (their zeroes, the last phase's 32 MFMAs) and what reads them
template <int R>
__device__ __forceinline__ void fence_rows(f32x4_t (&acc)[8][4]) {
  asm volatile("s_nop 7\n\ts_nop 7"
               : "+a"(acc[R][0]), "+a"(acc[R][1]), "+a"(acc[R][2]), "+a"(acc[R][3]), "+a"(acc[R + 1][0]), "+a"(acc[R + 1][1]), "+a"(acc[R + 1][2]),
                 "+a"(acc[R + 1][3]), "+a"(acc[R + 2][0]), "+a"(acc[R + 2][1]), "+a"(acc[R + 2][2]), "+a"(acc[R + 2][3]), "+a"(acc[R + 3][0]),
                 "+a"(acc[R + 3][1]), "+a"(acc[R + 3][2]), "+a"(acc[R + 3][3]));
}

// one MFMA; the two wait states are for operands that the compiler writes just ahead (a constant's copies: it does not look into the statement)
__device__ __forceinline__ void mfma_acc(f32x4_t& c, const bf16x8_t& a, const bf16x8_t& b) {
  asm volatile("s_nop 1\n\tv_mfma_f32_16x16x32_bf16 %0, %2, %1, %0" : "+a"(c) : "v"(a), "v"(b) : "memory");
}

template <int OUT>
__device__ __forceinline__ void put1(void* out, int m, float v, int add) {
  if constexpr (OUT >= OUT_STORE_F32) {
    float* p = static_cast<float*>(out) + m;
    *p = add ? *p + v : v;
  } else {
    unsigned short* p = static_cast<unsigned short*>(out) + m;
    *p = f2bf(add ? bf2f(*p) + v : v);
  }
}

// BIAS (weight gradients): dy's column sums, this product's row sums of A, ride along.  The waves of the first four tile columns take one of the tile's 16-row
// blocks each, two more MFMAs against ones to a K-tile's 64 (a pass over dy and a launch to add its parts were 10 to 14 us a bias, 48 of them in a gpt2-125m step
// of 8192 tokens: the step 12174 us, so 11860).  The block's fragments are read where its image is: of A_lo(t+1) in P1(t), of A_hi(t) in P0(t).
// Not AT: rows past the last are read as zeros or not at all, and not stored.
template <bool AT, int OUT, bool BIAS>
__device__ __forceinline__ void tall_workgroup(const TallArgs& args, int block, unsigned char* smem) {
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wr = wave >> 1, wc = wave & 1;
  const long lda = args.lda, ldb = args.ldb;

  // item: split outermost, then groups of four tile rows, row innermost; each XCD takes a contiguous run of them, so its L2 holds the panels that it shares
  const int n_items = args.tiles_m * args.tiles_n * args.splits;
  const int q8 = n_items / 8, r8 = n_items % 8, x = block % 8;
  const int item = (x < r8 ? x * (q8 + 1) : r8 * (q8 + 1) + (x - r8) * q8) + block / 8;
  const int tiles = args.tiles_m * args.tiles_n;
  const int sp = item / tiles, wg = item - sp * tiles;
  const int grp = wg / (4 * args.tiles_n), gsz = min(4, args.tiles_m - grp * 4), inner = wg - grp * 4 * args.tiles_n;
  const int tm = grp * 4 + inner % gsz, tn = inner / gsz;
  const int pairs = (args.K + 2 * TK - 1) / (2 * TK);  // AT: the last pair of K-tiles may be part full
  const int k0 = 2 * (int)((long)pairs * sp / args.splits), KT = 2 * (int)((long)pairs * (sp + 1) / args.splits) - k0;

  i32x4_t ra = AT ? make_rsrc(args.a + (long)tm * TM)
                  : make_rsrc_n(args.a + (long)tm * TM * lda, (unsigned)min(((long)(min(args.M - tm * TM, TM) - 1) * lda + args.K) * 2, 0x7fffffffL));
  i32x4_t rb = make_rsrc(args.b + (long)tn * TALL_N);
  // AT: the last two K-tiles through buffers of their own that start with them and end with the last token's row, so that what is read past it is zero (a row
  // past the end starts past the range: the rows do not overlap)
  i32x4_t ta[2], tb[2];
  if constexpr (AT) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int gk = 2 * pairs - 2 + i, rows = args.K - gk * TK;
      ta[i] = make_rsrc_n(args.a + (long)gk * TK * lda + (long)tm * TM, rows > 0 ? (unsigned)(((long)(min(rows, TK) - 1) * lda + args.M - tm * TM) * 2) : 0u);
      tb[i] = make_rsrc_n(args.b + (long)gk * TK * ldb + (long)tn * TALL_N, rows > 0 ? (unsigned)(((long)(min(rows, TK) - 1) * ldb + args.N - tn * TALL_N) * 2) : 0u);
    }
    asm volatile("s_nop 7" : "+s"(ta[0]), "+s"(ta[1]), "+s"(tb[0]), "+s"(tb[1]));
  }
  asm volatile("s_nop 7" : "+s"(ra), "+s"(rb));  // lane-read scalars to the first DMA piece that uses them
  // K-tile t of the item: its buffer and offset
  auto src = [&](bool is_b, int t, unsigned step, unsigned& so) __attribute__((always_inline)) {
    const int gk = k0 + t, i = gk - (2 * pairs - 2);
    i32x4_t r = is_b ? rb : ra;
    so = (unsigned)gk * step;
    if constexpr (AT) {
      if (i >= 0) {
        r = is_b ? (i ? tb[1] : tb[0]) : (i ? ta[1] : ta[0]);
        so = 0;
      }
    }
    return r;
  };
  const unsigned a_step = AT ? (unsigned)(TK * lda * 2) : (unsigned)(TK * 2), b_step = (unsigned)(TK * ldb * 2);
  unsigned vo[3][4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    vo[A_LO][i] = stage_voff<AT, A_LO, NT4>(i, tid, lda);
    vo[A_HI][i] = stage_voff<AT, A_HI, NT4>(i, tid, lda);
    vo[B_H0][i] = stage_voff<true, B_H0, NT4>(i, tid, ldb);
  }
  const unsigned lds0 = lds_addr(smem) + wave * 1024;
  auto issue = [&](auto kind_c, int t, int slot, auto n_c) __attribute__((always_inline)) {
    constexpr int kind = decltype(kind_c)::value, n = decltype(n_c)::value;
    unsigned so;
    const i32x4_t r = src(kind == B_H0, t, kind == B_H0 ? b_step : a_step, so);
#pragma unroll
    for (int i = 0; i < n; ++i) bdma16(r, vo[kind][i], so, lds0 + slot + kind * HALF + i * 4096);
  };

  f32x4_t acc[8][4];
  bf16x8_t a_lo[4][2], a_hi[4][2], b[2][4][2];
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  fence_rows<0>(acc);
  fence_rows<4>(acc);
  const int blk = tn * 2 + wc;  // BIAS: of this tile's eight row blocks of a wave row
  const bool sum_lo = BIAS && blk < 4, sum_hi = BIAS && blk >= 4 && blk < 8;
  f32x4_t bacc = {0.f, 0.f, 0.f, 0.f};
  bf16x8_t bf[2];
  bf16x8_t ones = __builtin_bit_cast(bf16x8_t, s8_t{0x3f80, 0x3f80, 0x3f80, 0x3f80, 0x3f80, 0x3f80, 0x3f80, 0x3f80});
  if constexpr (BIAS) asm volatile("s_nop 7" : "+a"(bacc), "+v"(ones));  // (kept: not made anew for each use)
  auto bias_frag = [&](const unsigned char* img) __attribute__((always_inline)) {
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) bf[ks] = frag<AT>(img, wr * 64 + 16 * (blk & 3), ks, lane);
  };

  issue(K_<B_H0>{}, 0, 0, K_<4>{});
  issue(K_<A_LO>{}, 0, 0, K_<4>{});
  issue(K_<A_HI>{}, 0, 0, K_<4>{});
  issue(K_<B_H0>{}, 1, SLOT, K_<4>{});
  issue(K_<A_LO>{}, 1, SLOT, K_<4>{});
  issue(K_<A_HI>{}, 1, SLOT, K_<4>{});
  issue(K_<B_H0>{}, 2, 2 * SLOT, K_<4>{});
  issue(K_<A_LO>{}, 2, 2 * SLOT, K_<2>{});
  wait_vm<22>();
  bar();
#pragma unroll
  for (int ks = 0; ks < 2; ++ks)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      a_lo[i][ks] = frag<AT>(smem + A_LO * HALF, wr * 64 + 16 * i, ks, lane);
      b[0][i][ks] = frag<true>(smem + B_H0 * HALF, wc * 64 + 16 * i, ks, lane);
    }
  if constexpr (BIAS) {
    if (sum_lo) bias_frag(smem + A_LO * HALF);
  }
  wait_vm<10>();
  __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
  bar();

  // K-tile t in ring slot s0; s1, s2: those of t + 1 and t + 2.  DMA: 2 = both phases issue, 1 = only P0 does, 0 = none; WAIT: vmcnt at the end (-1: last)
  auto ktile = [&](auto par_c, auto dma_c, auto wait_c, int t, int s0, int s1, int s2) __attribute__((always_inline)) {
    constexpr int P = decltype(par_c)::value, DMA = decltype(dma_c)::value, WAIT = decltype(wait_c)::value;
    constexpr bool NEXT = WAIT >= 0;
    unsigned so0, soa, sob;
    const i32x4_t ra0 = src(false, t + 2, a_step, so0);
    const unsigned l0 = lds0 + s2;
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      const int ks = q >> 3, i = (q >> 1) & 3, j = (q & 1) * 2;
      if (DMA >= 1 && q % 3 == 0) {
        const int n = q / 3, kind = n < 2 ? A_LO : A_HI, pc = n < 2 ? 2 + n : n - 2;
        g4w_pair_dma(acc[i][j], acc[i][j + 1], a_lo[i][ks], b[P][j][ks], b[P][j + 1][ks], vo[kind][pc], ra0, so0, l0 + kind * HALF + pc * 4096);
      } else {
        g4w_pair(acc[i][j], acc[i][j + 1], a_lo[i][ks], b[P][j][ks], b[P][j + 1][ks]);
      }
      if (q < 8) a_hi[q & 3][q >> 2] = frag<AT>(smem + s0 + A_HI * HALF, wr * 64 + 16 * (q & 3), q >> 2, lane);
      else if (NEXT && q < 12) b[P ^ 1][q & 3][0] = frag<true>(smem + s1 + B_H0 * HALF, wc * 64 + 16 * (q & 3), 0, lane);
      if constexpr (BIAS) {
        if (q == 12 && sum_hi) bias_frag(smem + s0 + A_HI * HALF);
      }
    }
    const i32x4_t ra1 = src(false, t + 3, a_step, soa), rb1 = src(true, t + 3, b_step, sob);
    const unsigned l1 = lds0 + s0;
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      const int ks = q >> 3, i = (q >> 1) & 3, j = (q & 1) * 2;
      if (DMA == 2 && q % 3 == 0) {
        const int n = q / 3, kind = n < 4 ? B_H0 : A_LO, pc = n & 3;
        g4w_pair_dma(acc[4 + i][j], acc[4 + i][j + 1], a_hi[i][ks], b[P][j][ks], b[P][j + 1][ks], vo[kind][pc], n < 4 ? rb1 : ra1, n < 4 ? sob : soa,
                     l1 + kind * HALF + pc * 4096);
      } else {
        g4w_pair(acc[4 + i][j], acc[4 + i][j + 1], a_hi[i][ks], b[P][j][ks], b[P][j + 1][ks]);
      }
      if (NEXT && q < 8) a_lo[q & 3][q >> 2] = frag<AT>(smem + s1 + A_LO * HALF, wr * 64 + 16 * (q & 3), q >> 2, lane);
      else if (NEXT && q < 12) b[P ^ 1][q & 3][1] = frag<true>(smem + s1 + B_H0 * HALF, wc * 64 + 16 * (q & 3), 1, lane);
      if constexpr (BIAS) {
        if ((q == 4 || q == 8) && blk < 8) mfma_acc(bacc, bf[q / 4 - 1], ones);
        if (NEXT && q == 12 && sum_lo) bias_frag(smem + s1 + A_LO * HALF);
      }
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
  for (int t = 0; t < KT - 4; t += 2) {  // KT even, >= 4
    ktile(K_<0>{}, K_<2>{}, K_<10>{}, t, s0, s1, s2);
    turn();
    ktile(K_<1>{}, K_<2>{}, K_<10>{}, t + 1, s0, s1, s2);
    turn();
  }
  ktile(K_<0>{}, K_<2>{}, K_<10>{}, KT - 4, s0, s1, s2);
  turn();
  ktile(K_<1>{}, K_<1>{}, K_<4>{}, KT - 3, s0, s1, s2);
  turn();
  ktile(K_<0>{}, K_<0>{}, K_<0>{}, KT - 2, s0, s1, s2);
  turn();
  ktile(K_<1>{}, K_<0>{}, K_<-1>{}, KT - 1, s0, s1, s2);
  fence_rows<4>(acc);

  // lane holds C[wr * 128 + 16 i + (l & 15)][wc * 64 + 16 j + 4 (l >> 4) + r]
  const int g = lane >> 4, i16 = lane & 15;
  const long row0 = (long)tm * TM + wr * 128 + i16;
  const int col0 = tn * TALL_N + wc * 64;
  if constexpr (BIAS) {
    asm volatile("s_nop 7\n\ts_nop 7" : "+a"(bacc));
    if (blk < 8 && g == 0) {  // bacc[r]: row l & 15 of the block, the same in every r and g
      const int m = tm * TM + wr * 128 + 16 * blk + i16;
      if (args.splits > 1) args.ws[((long)args.splits * args.N + sp) * args.M + m] = bacc[0];
      else put1<OUT>(args.bias, m, bacc[0], args.bias_add);
    }
  }
  if (args.splits > 1 || OUT >= OUT_STORE_F32) {
    const bool part = args.splits > 1;
    const long ld = part ? args.N : args.ldc;
    float* C = (part ? args.ws + (long)sp * args.M * args.N : static_cast<float*>(args.c)) + row0 * ld + col0 + 4 * g;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      f32x4_t old[4];
      const bool add = OUT == OUT_ADD_F32 && !part;
      if (add) {
#pragma unroll
        for (int j = 0; j < 4; ++j) old[j] = *reinterpret_cast<const f32x4_t*>(C + 16 * i * ld + 16 * j);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) *reinterpret_cast<f32x4_t*>(C + 16 * i * ld + 16 * j) = add ? acc[i][j] + old[j] : acc[i][j];
    }
    return;
  }
  // bf16, 16 bytes to a lane: lanes of neighbouring groups swap halves of two column tiles
  unsigned short* C = static_cast<unsigned short*>(args.c) + row0 * args.ldc + col0 + 16 * (g & 1) + 8 * (g >> 1);
  const int rows = AT ? TM : args.M - (tm * TM + wr * 128 + i16);  // (the lanes that swap hold one row)
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int jp = 0; jp < 2; ++jp) {
      unsigned short* p = C + 16 * i * args.ldc + 32 * jp;
      float v[8];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(acc[i][2 * jp][e]), __float_as_uint(acc[i][2 * jp + 1][e]), false, false);
        v[e] = __uint_as_float(r[0]);
        v[4 + e] = __uint_as_float(r[1]);
      }
      if constexpr (OUT == OUT_ADD) {
        float old[8];
        load8(p, old);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] += old[e];
      }
      if (16 * i < rows) store8(p, v);
    }
}

template <bool AT, int OUT, bool BIAS>
__global__ __launch_bounds__(NT4, 1) __attribute__((amdgpu_waves_per_eu(1, 1))) void gemm_tall_kernel(TallArgs args) {
  __shared__ __attribute__((aligned(1024))) unsigned char smem[3 * SLOT];
  tall_workgroup<AT, OUT, BIAS>(args, (int)blockIdx.x, smem);
}

// A layer's two gradients in one launch: the longer items first, n_first of them, and the others on the CUs that have none or are done.
template <int OUT, bool BIAS>
__global__ __launch_bounds__(NT4, 1) __attribute__((amdgpu_waves_per_eu(1, 1))) void gemm_tall_back_kernel(TallArgs data, TallArgs weight, int n_first, bool data_first) {
  __shared__ __attribute__((aligned(1024))) unsigned char smem[3 * SLOT];
  const bool first = (int)blockIdx.x < n_first;
  const int block = (int)blockIdx.x - (first ? 0 : n_first);
  if (first == data_first) tall_workgroup<false, OUT_STORE, false>(data, block, smem);
  else tall_workgroup<true, OUT, BIAS>(weight, block, smem);
}

// out (+)= the partial sums, added in the order of K; a thread's 8 columns of a row
template <int OUT, bool BIAS>
__global__ __launch_bounds__(256) void gemm_tall_reduce(TallArgs args) {
  const long e = ((long)blockIdx.x * 256 + threadIdx.x) * 8;  // M N is a multiple of 2048
  const long row = e / args.N, col = e - row * args.N, MN = (long)args.M * args.N;
  float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  const float* W = args.ws + e;
  if (BIAS && e / 8 < args.M) {  // (N >= 512: threads enough)
    const float* B = args.ws + args.splits * MN + e / 8;
    float t = 0.f;
#pragma unroll 4
    for (int s = 0; s < args.splits; ++s) t += B[(long)s * args.M];
    put1<OUT>(args.bias, (int)(e / 8), t, args.bias_add);
  }
#pragma unroll 4
  for (int s = 0; s < args.splits; ++s) {
    const f32x4_t x0 = *reinterpret_cast<const f32x4_t*>(W + s * MN), x1 = *reinterpret_cast<const f32x4_t*>(W + s * MN + 4);
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] += x0[j], v[4 + j] += x1[j];
  }
  if constexpr (OUT >= OUT_STORE_F32) {
    f32x4_t* p = reinterpret_cast<f32x4_t*>(static_cast<float*>(args.c) + row * args.ldc + col);
    f32x4_t lo = {v[0], v[1], v[2], v[3]}, hi = {v[4], v[5], v[6], v[7]};
    if constexpr (OUT == OUT_ADD_F32) lo += p[0], hi += p[1];
    p[0] = lo;
    p[1] = hi;
  } else {
    unsigned short* p = static_cast<unsigned short*>(args.c) + row * args.ldc + col;
    if constexpr (OUT == OUT_ADD) {
      float old[8];
      load8(p, old);
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] += old[j];
    }
    store8(p, v);
  }
}

template <bool AT>
void launch(const TallArgs& g, int out) {
  const dim3 grid(g.tiles_m * g.tiles_n * g.splits), red((unsigned)((long)g.M * g.N / 2048));
  auto go = [&](auto out_c) {
    constexpr int OUT = decltype(out_c)::value;
    auto with = [&](auto bias_c) {
      constexpr bool BIAS = decltype(bias_c)::value;
      hipLaunchKernelGGL((gemm_tall_kernel<AT, OUT, BIAS>), grid, dim3(NT4), 0, stream(), g);
      if (g.splits > 1) hipLaunchKernelGGL((gemm_tall_reduce<OUT, BIAS>), red, dim3(256), 0, stream(), g);
    };
    if constexpr (AT) {
      if (g.bias != nullptr) return with(std::true_type{});
    }
    with(std::false_type{});
  };
  switch (out) {
    case OUT_STORE: go(K_<OUT_STORE>{}); break;
    case OUT_ADD: go(K_<OUT_ADD>{}); break;
    case OUT_STORE_F32: go(K_<OUT_STORE_F32>{}); break;
    default: go(K_<OUT_ADD_F32>{}); break;
  }
}

}  // namespace

namespace {
// us of `items` workgroups, one to a CU at a time, of k K-tiles each: `empty` + `full` times the share of the chip that is filled a K-tile, `fixed` a workgroup
double rounds_us(double items, double k, double empty, double full, double fixed) {
  const double cus = num_cus(), whole = std::floor(items / cus), rest = items - whole * cus;
  return whole * (k * (empty + full) + fixed) + (rest > 0 ? k * (empty + full * rest / cus) + fixed : 0.0);
}
double pairs_of(long K) { return (double)((K + 2 * TK - 1) / (2 * TK)); }
double split_k(double pairs, int S) { return 2.0 * std::ceil(pairs / S); }
constexpr double TALL_EMPTY = 0.743, TALL_FULL = 0.06, TALL_FIXED = 5.4;
double reduce_us(long M, long N, int S) { return S > 1 ? 5.8 + (double)M * N * S * 8.0 / 9.6e6 : 0.0; }
double wide_us(long K, long n_main, long n_tail, int splits) {  // gemm64's 256 x 256 tiles
  const double kt = 2.0 * pairs_of(K);
  double us = rounds_us((double)n_main, kt, 0.92, 0.36, 10.4);
  if (n_tail > 0) us += rounds_us((double)n_tail * splits, kt / splits, 0.92, 0.36, 10.4);
  if (n_tail > 0 && splits > 1) us += 8.2 + (double)n_tail * TM * TN * splits * 8.0 / 14.7e6;
  return us;
}
}  // namespace

// K-ranges for this kernel where it is the faster one, else 0.  n_main whole tiles of 256 x 256 and n_tail in `splits` ranges each are gemm64's plan.  Both
// times from the sizes, us: a round costs its K-tiles and a fixed part (fill and store), a K-tile of 64 more the fuller the chip is (0.74 here on an empty one, 0.80
// on a full one; 0.92 and 1.28 there); partial sums cost a launch and their bytes, written and read.  Ranges stay at four K-tiles and more, what the peeled loop
// takes.  Constants fitted to 540 sizes, both layouts, 256 to 24576 rows, operands from HBM (profiles/backward_tiles.txt): the choice is within 0.5 % of the faster one
// on average; by it these tiles take 13 % less time than 256 x 256 ones everywhere, and in 5 sizes 3 to 7 % more (12288 x 2048 x 1536 71.9, here 77.2).  The margin
// keeps long single rounds of less than the chip on the others, which their last K-tiles' loads hold up here (2560 x 2560 weight gradients over 16384 rows 191 there,
// here 250; 5120 x 1280 over 6144 80 and 97).
// us_of: the faster one's time.
int gemm_tall_splits(long M, long N, long K, long n_main, long n_tail, int splits, double* us_of) {
  double limit = wide_us(K, n_main, n_tail, splits);
  if (us_of != nullptr) *us_of = limit;
  limit *= 0.972;
  int best = 0;
  for (int S = 1; S <= 16 && K >= 4L * TK * S; ++S) {
    const double us = rounds_us((double)(M / TM) * (N / TALL_N) * S, split_k(pairs_of(K), S), TALL_EMPTY, TALL_FULL, TALL_FIXED) + reduce_us(M, N, S);
    if (us < limit) limit = us, best = S;
  }
  if (us_of != nullptr && best > 0) *us_of = limit;
  return best;
}

// K-ranges of the weight gradient where a layer's two gradients, dy w and dy^T x of T tokens, O outputs and I inputs, take less time in one launch
// (gemm_tall_back) than in two, of either kind of tiles; else 0.  The second launch's workgroups start on the CUs that the first ones leave idle: 8192 tokens of
// a 768 x 3072 layer are 192 and 216 workgroups, 64 and 40 CUs idle.  two_us is the time of the two by the model above (data gradients whose tokens are no
// multiple of 256 go to the library, which takes as long as these tiles), and the one launch's the end of a list of workgroups, longest first, dealt out to the CUs.
// Constants fitted to 330 sizes (256 to 9216 tokens, 256 to 6144 outputs, 256 to 4096 inputs; profiles/backward_pairs.txt): what the rule picks takes 21 % less time
// than two launches on average and 1 % more than the best choice; in one of 257 sizes 2 % more than two (3328 x 5120 x 1024 90.3, so 91.8).  More ranges have to save 2 %: by less than
// that 7168 x 3072 x 768 went into six, 94.9, where two launches are 85.7 and four ranges 80.2.
// us, two launches / one: 8192 tokens 768 x 768 40.2 / 34.0, 2304 x 768 76.3 / 70.0, 3072 x 768 99.4 / 87.7, 768 x 3072 106.8 / 97.7; 1326 tokens 768 x 3072 37.4 /
// 24.0; but 8192 x 4096 x 4096 373 / 436, where 256 x 256 tiles fill the chip.
constexpr double BACK_TILE = 0.76, BACK_FIXED = 4.0, BACK_MARGIN = 1.05, BACK_MORE = 0.98;
int64_t gemm_tall_back_splits(int64_t T, int64_t O, int64_t I, bool bias, double two_us) {
  if (T < 4 * TK || O <= 0 || I <= 0 || O % TM != 0 || I % TN != 0 || (bias && I < 4 * TALL_N)) return 0;
  const long nd = (T + TM - 1) / TM * (I / TALL_N), tiles = O / TM * (I / TALL_N);
  if (nd + tiles > 8L * num_cus()) return 0;  // (rounds enough to fill the last one's gap)
  const double d_us = O / TK * BACK_TILE + BACK_FIXED;
  double limit = two_us * BACK_MARGIN;
  int64_t best = 0;
  for (int S = 1; S <= 16 && T >= 4L * TK * S; ++S) {
    const double w_us = split_k(pairs_of(T), S) * BACK_TILE + BACK_FIXED;
    std::priority_queue<double, std::vector<double>, std::greater<double>> cus(std::greater<double>(), std::vector<double>(num_cus(), 0.0));
    double end = 0.0;
    auto deal = [&](long n, double us) {
      for (long i = 0; i < n; ++i) {
        const double t = cus.top() + us;
        cus.pop();
        cus.push(t);
        end = std::max(end, t);
      }
    };
    if (d_us >= w_us) deal(nd, d_us), deal(tiles * S, w_us);
    else deal(tiles * S, w_us), deal(nd, d_us);
    const double us = end + (S > 1 ? 4.5 + (double)O * I * S * 8.0 / 7.0e6 : 0.0);
    if (us < limit * (best == 0 ? 1.0 : BACK_MORE)) limit = us, best = S;
  }
  return best;
}

namespace {
// the operands of one product; ragged: rows of A (not transposed) that fill no whole tile
TallArgs tall_args(const at::Tensor& a, const at::Tensor& b, const at::Tensor& out, bool at_, int64_t splits, const c10::optional<at::Tensor>& bias, bool bias_add, bool ragged) {
  LLMCTL_CHECK(a.dim() == 2 && b.dim() == 2 && out.dim() == 2 && a.is_cuda() && b.is_cuda() && out.is_cuda(), "gemm_tall: 2-D GPU operands");
  const bool f32 = out.scalar_type() == at::kFloat;
  LLMCTL_CHECK(a.scalar_type() == at::kBFloat16 && b.scalar_type() == at::kBFloat16 && (f32 || out.scalar_type() == at::kBFloat16),
               "gemm_tall: bf16 operands, bf16 or fp32 out");
  const long M = at_ ? a.size(1) : a.size(0), K = at_ ? a.size(0) : a.size(1), N = b.size(1);
  LLMCTL_CHECK(b.size(0) == K && out.size(0) == M && out.size(1) == N, "gemm_tall: shapes");
  LLMCTL_CHECK(M > 0 && N > 0 && (M % TM == 0 || ragged) && N % TALL_N == 0 && (at_ || K % (2 * TK) == 0) && splits >= 1 && (K + 2 * TK - 1) / (2 * TK) >= 2 * splits,
               "gemm_tall: M in 256s, N (and K, but for a transposed A) in 128s, two pairs of K-tiles of 64 to a split, the last of them part full at most");
  LLMCTL_CHECK(!at_ || K % (2 * TK) == 0 || (a.stride(0) >= M && b.stride(0) >= N), "gemm_tall: rows that do not overlap");
  LLMCTL_CHECK(at_ || M % TM == 0 || a.stride(0) >= K, "gemm_tall: rows that do not overlap");
  auto rows16 = [](const at::Tensor& t, int per) {
    return t.stride(1) == 1 && t.stride(0) % per == 0 && (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0;
  };
  LLMCTL_CHECK(rows16(a, 8) && rows16(b, 8) && rows16(out, f32 ? 4 : 8), "gemm_tall: 16-byte aligned rows, unit column stride");
  const long a_span = (at_ ? K : (long)TM) * a.stride(0) * 2, b_span = K * b.stride(0) * 2;
  LLMCTL_CHECK(a_span < (1L << 31) && b_span < (1L << 31) && M * N / 2048 < (1L << 31), "gemm_tall: operand too large for 32-bit offsets");
  LLMCTL_CHECK(!bias.has_value() || (at_ && N >= 4 * TALL_N && bias->is_cuda() && bias->is_contiguous() && bias->numel() == M &&
                                     bias->scalar_type() == out.scalar_type()),
               "gemm_tall: a bias goes with a transposed A and 512 columns, [M] of out's type");
  return TallArgs{bf_ptr(a), bf_ptr(b), out.data_ptr(), nullptr, bias.has_value() ? bias->data_ptr() : nullptr, bias_add, (long)a.stride(0), (long)b.stride(0),
                  (long)out.stride(0), (int)M, (int)N, (int)K, (int)((M + TM - 1) / TM), (int)(N / TALL_N), (int)splits};
}
// room for the partial sums of more than one range
at::Tensor tall_room(TallArgs& g, const at::Tensor& a) {
  if (g.splits <= 1) return {};
  at::Tensor ws = at::empty({(long)g.splits * g.M * (g.N + 1)}, a.options().dtype(at::kFloat));
  g.ws = ws.data_ptr<float>();
  return ws;
}
}  // namespace

// out [M, N] (+)= A B with B [K, N] and A [M, K], or [K, M] where at; out bf16 or fp32.  M a multiple of 256, N of 128 and, not where at, K of 128; two pairs of
// K-tiles to a split, 256 of K, of which the last one of a transposed A has more than 128.
// bias [M] (+)= the row sums of A, of out's type (at, N >= 512).
void gemm_tall(const at::Tensor& a, const at::Tensor& b, at::Tensor out, bool at_, bool accumulate, int64_t splits, const c10::optional<at::Tensor>& bias,
               bool bias_add) {
  TallArgs g = tall_args(a, b, out, at_, splits, bias, bias_add, false);
  const c10::DeviceGuard guard(a.device());
  const at::Tensor ws = tall_room(g, a);
  const int o = (out.scalar_type() == at::kFloat ? OUT_STORE_F32 : OUT_STORE) + (accumulate ? 1 : 0);
  if (at_) launch<true>(g, o);
  else launch<false>(g, o);
}

// A layer's two gradients in one launch: dx = dy w of any number of rows, g (+)= dy^T x in `splits` ranges of the tokens and, where given, db (+)= dy's column
// sums.  dy [T, O], w [O, I], x [T, I]; O in 256s, I in 128s (with db from 512 on), T >= 256 a split.
void gemm_tall_back(const at::Tensor& dy, const at::Tensor& w, at::Tensor dx, const at::Tensor& x, at::Tensor g, bool accumulate, int64_t splits,
                    const c10::optional<at::Tensor>& db, bool add) {
  LLMCTL_CHECK(dx.scalar_type() == at::kBFloat16, "gemm_tall_back: dx bf16");
  const TallArgs d = tall_args(dy, w, dx, false, 1, c10::nullopt, false, true);
  TallArgs v = tall_args(dy, x, g, true, splits, db, add, false);
  const c10::DeviceGuard guard(dy.device());
  const at::Tensor ws = tall_room(v, dy);
  const int nd = d.tiles_m * d.tiles_n, nv = v.tiles_m * v.tiles_n * v.splits;
  const bool d_first = d.K / TK >= 2 * (((v.K + 2 * TK - 1) / (2 * TK) + v.splits - 1) / v.splits);
  auto go = [&](auto out_c) {
    constexpr int OUT = decltype(out_c)::value;
    auto with = [&](auto bias_c) {
      constexpr bool BIAS = decltype(bias_c)::value;
      hipLaunchKernelGGL((gemm_tall_back_kernel<OUT, BIAS>), dim3(nd + nv), dim3(NT4), 0, stream(), d, v, d_first ? nd : nv, d_first);
      if (v.splits > 1) hipLaunchKernelGGL((gemm_tall_reduce<OUT, BIAS>), dim3((unsigned)((long)v.M * v.N / 2048)), dim3(256), 0, stream(), v);
    };
    if (v.bias != nullptr) with(std::true_type{});
    else with(std::false_type{});
  };
  const bool f32 = g.scalar_type() == at::kFloat;
  if (f32 && accumulate) go(K_<OUT_ADD_F32>{});
  else if (f32) go(K_<OUT_STORE_F32>{});
  else if (accumulate) go(K_<OUT_ADD>{});
  else go(K_<OUT_STORE>{});
}

TORCH_LIBRARY_IMPL(llmctl, CUDA, m) {
  m.impl("gemm_tall", &gemm_tall);
  m.impl("gemm_tall_back", &gemm_tall_back);
}

}  // namespace llmctl
