// Latent attention on the matrix cores (bf16; MFMA 32x32x16) for prompt portions, and for decode rows whose many heads share their
// keys (decode_tiles_pay); other decode rows: row_decode.hip.
//
// The cache row [latent | rotary key] of width R is key and, in its first ``rank`` entries, value; the
// queries come in the same layout (see latent_attn.hip).  This is the flash-attention forward of the
// framework's paged prefill kernel re-cut for that layout:
//   * a workgroup (4 waves) owns 128 query rows = TB tokens x HB heads of one sequence (HB = 1 for
//     long portions, = the head count for decode rows and short portions, where the heads of a token
//     fill the tile and share every key row);
//   * tiles of 64 keys, gathered through the block table into LDS once per workgroup: a "row image"
//     of all of R (in column blocks of 128) for S^T = K Q^T, and a "transposed-read image" of the
//     column blocks that hold this workgroup's value columns for O^T += V^T P^T;
//   * Q fragments stay in registers for the whole key loop; softmax is lane-local (query on the lane),
//     exp2 domain, deferred rescale; the sink starts the running maximum and the denominator;
//   * the key loop runs only over the tiles that the rows' windows touch.
// Bound: at one wave a SIMD (keys wider than 128) the chain of a tile, fill requests, scores, softmax, values; the MFMAs are a fifth of it.  What a tile's chain held beside
// them, us a layer, 2048 tokens x 16 heads, keys of 192, window 1024 (three layers 206 us, so 143): a block-table entry used right where it was loaded (the wave that looked the
// slots up waited for HBM in every tile), a slot lookup in LDS per DMA piece, score fragments read just ahead of their MFMAs, a branch per masked element.  The other forms: 16 heads
// over 4 kv groups, sigmoid weights, five portions of 2911 tokens 126 us, so 76; keys of 128, window 1024, 2048 + 1331 tokens 68.5, so 55.7.  With the blocks of a head on one XCD,
// whose L2 then holds its keys, alone: 126, so 113.
// Value columns beyond 256 go to further workgroups (blockIdx.z), which recompute the scores.
// Shapes it takes: R and rank multiples of 8, R <= 640; anything else runs the generic kernels.
#include "attn_common.h"
#include "hybrid_common.h"

namespace llmctl_hybrid {
using namespace llmctl::attn;

namespace {
constexpr int LKB = 64;         // keys per tile
constexpr int LROWB = 256;      // bytes of one row of a 128-column block image
constexpr int LIMG = LKB * LROWB;
constexpr float kRescaleTh = 8.f;
constexpr float kLog2e = 1.4426950408889634f;

struct LArgs {
  const unsigned short* qa;
  const unsigned short* cache;
  unsigned short* out;
  const int* bt;
  const int* cu;
  const int* ctx;
  const float* sink;    // nullptr: no sink
  const float* hscale;  // nullptr or a factor on every head's scores
  const float* ofreq;   // nullptr, or [rk / 2]: the output's neighbour pairs are turned back by -position * ofreq
  const float* dist_a;  // SIG forms: [H] each; dist_a ln(1 + dist_b (i - j)) is taken off the scaled score and a visible
  const float* dist_b;  // key weighs sigmoid(score + sig_bias); dist_a may be nullptr (no penalty)
  const float* sig_bias;
  int H, R, rk, bs, maxb, window, HB, nvt;
  int G, rs, koff, chunk, hpg;  // kv groups, row width, key's first column, chunk mask size, head tiles per group
  int keep;                     // the window spares the keys at positions below this
  float scale_log2;
  float cap_log2, cap_inv2;     // CAP forms: x (log2 domain) = cap_log2 * tanh(s * scale); cap_inv2 = 2 log2(e) scale / cap
  // SPLIT forms: the key range of a decode row is spread over blockIdx.x (few sequences would otherwise leave the chip idle): each split
  // writes its unnormalised fp32 output and (running maximum, denominator) here, and row_merge joins them
  int xcd;  // prompt forms: the heads (a multiple of eight) are shared out to the XCDs
  int nsplit;
  const unsigned short* gate;  // nullptr, or RowAttnOpts::gate
  long gate_st;
  int gate_per;
  float* ws_o;   // [rows, nsplit, rk]
  float* ws_ml;  // [rows, nsplit, 2]
};

// ROT: the output's neighbour pairs are turned back by the query's position (a.ofreq); a template flag
// so that the forms without it keep their register budget.  SIG: the weights are sigmoids of the scores
// (after the distance penalty), not a softmax: no running maximum, no rescale, no denominator (l = 1).  CAP: the scaled score
// s becomes cap tanh(s / cap) before masks and softmax (tanh y = 1 - 2 / (1 + e^(2y))).  SPLIT: decode rows, one query per sequence (no
// a.cu), nsplit workgroups for a row's keys.
// Keys and values up to 128 wide: two workgroups per CU (64.5 KB of images each; held to 256 registers, one's softmax runs beside the
// other's products).  16 heads over 4 kv groups, portions of 2048 and 1331 tokens: 156 us at one per CU (200 + 96 registers),
// 100 so.  Wider keys stay at one: 192-wide keys took 108 us against 99, with one set of images instead of two 107.
// Prompts with keys of 129 to 256 columns: one workgroup's images fill a CU, so it has eight waves there, two on the same 32 query rows: the first takes the first 32 keys of
// every tile, the other the rest, each with a maximum, denominator and output of its own, which meet in LDS at the end: one's
// softmax runs beside the other's products.  2048 tokens x 16 heads, keys of 192, window 1024: 52.5 us, so 43.4.  (Wider keys or values have no registers for it; of keys up to 128
// two workgroups of four waves share a CU.)
constexpr bool two_key_groups(int nks, int ndb, bool split) { return !split && nks > 8 && nks <= 16 && ndb <= 4; }

template <int NKS, int NDB, bool ROT, bool SIG = false, bool CAP = false, bool SPLIT = false>
__global__ __launch_bounds__(two_key_groups(NKS, NDB, SPLIT) ? 512 : 256, (NKS <= 8 && NDB <= 4) || two_key_groups(NKS, NDB, SPLIT) ? 2 : 1) void latent_attn_mfma_kernel(LArgs a) {
  constexpr bool KG2 = two_key_groups(NKS, NDB, SPLIT);
  constexpr int KBN = KG2 ? 1 : 2, NW = KG2 ? 8 : 4;  // blocks of 32 keys that a wave takes of a tile; waves
  constexpr int NCB = (NKS + 7) / 8;
  constexpr int NTB = (NDB + 3) / 4;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  // the tile images: one set, or two (the fill of tile t + 1 then runs beside the products of tile t)
  // where two fit LDS
  constexpr int BUFB = (NCB + NTB) * LIMG;
  constexpr bool DB = 2 * BUFB + 1024 <= 160 * 1024;

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = KG2 ? (tid >> 6) & 3 : tid >> 6;
  const int kgrp = KG2 ? __builtin_amdgcn_readfirstlane(tid >> 8) : 0;
  const int r = lane & 31, hh = lane >> 5;
  // workgroups go round the XCDs in order; the blocks of a head, and the heads of a kv group, read the same keys, so they are dealt to one XCD and its L2
  unsigned bx = blockIdx.x, by = blockIdx.y, bz = blockIdx.z;
  if (!SPLIT && a.xcd) {
    const unsigned slice = gridDim.x * gridDim.y, l = bx + gridDim.x * by + slice * bz, v = (l & 7) * (gridDim.z / 8 * slice) + (l >> 3);
    bz = v / slice, by = (v - bz * slice) / gridDim.x, bx = v - bz * slice - by * gridDim.x;
  }
  const int n = by;
  const int hg = bz / a.nvt, v0 = (bz % a.nvt) * (NDB * 32);
  const int P = a.H / a.G;                       // query heads per kv group
  const int grp = hg / a.hpg, hsub = (hg % a.hpg) * a.HB;  // this workgroup's kv group, its first head inside it
  const int q_begin = SPLIT ? n : a.cu[n];
  const int qlen = SPLIT ? 1 : a.cu[n + 1] - q_begin;
  const int HB = a.HB, TB = 128 / HB;
  // prompt portions: the last query blocks of a sequence see the most keys; they are dispatched first
  const int split = SPLIT ? bx : 0;
  const int tok0 = SPLIT ? 0 : (int)(gridDim.x - 1 - bx) * TB;
  if (tok0 >= qlen) return;
  const int ctx = a.ctx[n];
  const int pos0 = ctx - qlen;
  const int row = wave * 32 + r;
  const int my_tok = tok0 + row / HB, my_head = grp * P + hsub + row % HB;
  const bool valid = my_tok < qlen && hsub + row % HB < P;
  const int tokc = min(my_tok, qlen - 1), headc = grp * P + min(hsub + row % HB, P - 1);
  const int my_pos = pos0 + tokc;
  const int* btn = a.bt + (long)n * a.maxb;

  bf16x8_t qf[NKS];
  {
    const unsigned short* Qp = a.qa + ((long)(q_begin + tokc) * a.H + headc) * a.R;
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) {
      const int col = ks * 16 + 8 * hh;
      uint4 v = make_uint4(0, 0, 0, 0);
      if (col < a.R) v = gload16(Qp + col);
      qf[ks] = __builtin_bit_cast(bf16x8_t, v);
    }
  }
  f32x16 o[NDB];
#pragma unroll
  for (int d = 0; d < NDB; ++d)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[d][i] = 0.f;
  float m_i = -INFINITY, l_i = 0.f;
  if (a.sink != nullptr && split == 0 && kgrp == 0) {  // the sink: one unit of mass at its own logit, counted by the first split
    m_i = a.sink[headc] * kLog2e;
    l_i = 1.0f;
  }
  const float my_scale = a.scale_log2 * (a.hscale != nullptr ? a.hscale[headc] : 1.0f);
  float pen_a = 0.f, pen_b = 0.f, sig_b2 = 0.f;
  if constexpr (SIG) {
    m_i = 0.f;
    l_i = split == 0 && kgrp == 0 ? 1.f : 0.f;
    if (a.dist_a != nullptr) pen_a = a.dist_a[headc], pen_b = a.dist_b[headc];
    sig_b2 = a.sig_bias[headc] * kLog2e;
  }

  const int first_pos = pos0 + tok0, last_pos = pos0 + min(tok0 + TB, qlen) - 1;
  // the first key a query at position p may see: inside its window and inside its chunk
  auto first_key = [&](int p) { return max(max(p - a.window + 1, (p / a.chunk) * a.chunk), 0); };
  const int t_first = first_key(first_pos) / LKB, t_end = last_pos / LKB + 1;
  // tiles before the window whose first keys it spares (those of the chunk of the block's first row; a block that
  // spans two chunks meets the second one inside the window's tiles): the key loop runs over them first.  Loop
  // index i in [t_lo, t_hi) stands for tile i < n_kept ? kept0 + i : t_first + i - n_kept.
  const int kept0 = ((first_pos / a.chunk) * a.chunk) / LKB;
  const int n_kept = a.keep > 0 ? max(min((a.keep + LKB - 1) / LKB, t_first) - kept0, 0) : 0;
  auto tile_of = [&](int i) { return i < n_kept ? kept0 + i : t_first + i - n_kept; };
  int t_lo = 0, t_hi = n_kept + t_end - t_first;
  if constexpr (SPLIT) {
    const int per = (t_hi + a.nsplit - 1) / a.nsplit;
    t_lo = split * per;
    t_hi = min(t_hi, t_lo + per);
  }
  // this wave's rows: positions [w_first, w_last]
  const int w_first = pos0 + min(tok0 + (wave * 32) / HB, qlen - 1);
  const int w_last = pos0 + min(tok0 + (wave * 32 + 31) / HB, qlen - 1);
  const bool wave_live = tok0 + (wave * 32) / HB < qlen && hsub + (HB >= 32 ? (wave * 32) % HB : 0) < P;
  const int w_lo = first_key(w_first), my_lo = first_key(my_pos);
  const int my_c0 = (my_pos / a.chunk) * a.chunk;  // first position of this row's chunk
  const int w_lo_last = first_key(w_last);  // first_key never decreases with the position
  // lane-only parts of the LDS read addresses, so that the key loop adds constants to them
  int tr_lo[4], tr_hi[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) tr_frag_offs<128>(c * 32, lane, tr_lo[c], tr_hi[c]);
  // K fragment of k-step ks, rows kb * 32 + r: chunk (2 ks + hh) ^ (r & 15) = (2 ks) ^ (hh ^ (r & 15))
  const int k_row = r * LROWB, k_x = (hh ^ (r & 15)) << 4;

  const int wave_u = __builtin_amdgcn_readfirstlane(tid >> 6);
  const unsigned lds_base = lds_addr(smem);
  // cache slots of a tile's 64 keys, looked up in the block table one tile ahead (double-buffered)
  int* slot_lds = reinterpret_cast<int*>(smem + (DB ? 2 : 1) * BUFB);
  auto load_slots = [&](int t, int buf) {
    if (tid < LKB) {
      const int key = min(t * LKB + tid, ctx - 1);
      slot_lds[buf * LKB + tid] = btn[key / a.bs] * a.bs + key % a.bs;
    }
  };
  // LDS-DMA fill: every wave instruction moves 4 key rows x 256 B of one image straight from the cache
  // to LDS (no registers, all pieces of the tile in flight at once); the images' swizzles are applied
  // to the source chunk.  Keys past the context and columns past the row read a valid neighbour instead
  // (finite data): such keys are masked below and such columns meet zero Q entries or are never stored.
  // A wave's rows of an image are 16 (32) apart, so their swizzle is one number and its slots serve all images.
  const int frow = wave_u * 4 + (lane >> 4), fch = lane & 15;
  int fcol[NCB + NTB];
#pragma unroll
  for (int img = 0; img < NCB + NTB; ++img) {
    const int col = img < NCB ? a.koff + (img * 16 + (fch ^ swz_row<128>(frow))) * 8 : ((v0 / 128 + (img - NCB)) * 16 + (fch ^ swz_tr<128>(frow))) * 8;
    fcol[img] = min(col, a.rs - 8);
  }
  auto fill = [&](int sbuf, int ibuf) {
    int slot[16 / NW];
#pragma unroll
    for (int j = 0; j < 16 / NW; ++j) slot[j] = slot_lds[sbuf * LKB + 4 * NW * j + frow];
#pragma unroll
    for (int j = 0; j < 16 / NW; ++j) {
      const unsigned short* base = a.cache + ((long)slot[j] * a.G + grp) * a.rs;
#pragma unroll
      for (int img = 0; img < NCB + NTB; ++img) dma16(base + fcol[img], lds_base + (unsigned)(ibuf * BUFB + img * LIMG + (wave_u + NW * j) * 1024));
    }
  };
  // double-buffered form: the slots of tile t + 2 are requested BEFORE the fill of tile t + 1 is issued and
  // stored to LDS at the top of the next iteration, so that no wave waits on its own fill in between (a
  // wave's memory operations complete in order)
  int pend = 0, pend_in = 0;  // the block, as the table holds it (an operation on it here would wait for it), and the place in the block
  auto ask_slot = [&](int t) {
    const int key = min(t * LKB + tid, ctx - 1);
    pend = btn[key / a.bs];
    pend_in = key % a.bs;
  };
  if (t_lo < t_hi) load_slots(tile_of(t_lo), 0);
  if constexpr (DB) {
    if (t_lo < t_hi) {
      __syncthreads();
      if (t_lo + 1 < t_hi && tid < LKB) ask_slot(tile_of(t_lo + 1));
      fill(0, 0);
    }
  }
  for (int t = t_lo; t < t_hi; ++t) {
    const int sbuf = (t - t_lo) & 1;
    const unsigned char* Ks = smem + (DB ? sbuf * BUFB : 0);
    const unsigned char* Vs = Ks + NCB * LIMG;
    if constexpr (DB) {
      // tile t was requested one iteration ago.  After the barrier every wave's pieces of it have landed,
      // every wave is done with tile t - 1 (its images may be overwritten) and the slots of t + 1 are visible
      if (t + 1 < t_hi && tid < LKB) slot_lds[(sbuf ^ 1) * LKB + tid] = pend * a.bs + pend_in;
      vm_wait<0>();
      __syncthreads();
      if (t + 2 < t_hi && tid < LKB) ask_slot(tile_of(t + 2));
      if (t + 1 < t_hi) fill(sbuf ^ 1, sbuf ^ 1);
    } else {
      __syncthreads();
      fill(sbuf, 0);
      if (t + 1 < t_hi) load_slots(tile_of(t + 1), sbuf ^ 1);
      vm_wait<0>();
      __syncthreads();
    }
    const int kv0 = tile_of(t) * LKB + kgrp * 32;  // the wave's first key of the tile
    if (!wave_live || kv0 > w_last || (kv0 + KBN * 32 - 1 < w_lo && kv0 >= a.keep)) continue;
    Ks += kgrp * 32 * LROWB, Vs += kgrp * 32 * LROWB;

    f32x16 s[KBN];
#pragma unroll
    for (int kb = 0; kb < KBN; ++kb)
#pragma unroll
      for (int i = 0; i < 16; ++i) s[kb][i] = 0.f;
    // the next k-steps' fragments are read while the ones before them are multiplied (left to itself the compiler reads each just ahead of its use)
    constexpr int KST = NKS >= 32 ? 1 : 2;  // (the widest keys have no registers for more)
    bf16x8_t kf[2][KST][KBN];
    auto read_k = [&](int k0, bf16x8_t (&f)[KST][KBN]) {
#pragma unroll
      for (int i = 0; i < KST; ++i)
#pragma unroll
        for (int kb = 0; kb < KBN; ++kb)
          f[i][kb] = lds_read_b128(Ks + ((k0 + i) >> 3) * LIMG + kb * 32 * LROWB, k_row + (k_x ^ (((2 * (k0 + i)) & 15) << 4)));
    };
    read_k(0, kf[0]);
#pragma unroll
    for (int k0 = 0; k0 < NKS; k0 += KST) {
      if (k0 + KST < NKS) read_k(k0 + KST, kf[(k0 / KST + 1) & 1]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < KST; ++i)
#pragma unroll
        for (int kb = 0; kb < KBN; ++kb) s[kb] = mfma32(kf[(k0 / KST) & 1][i][kb], qf[k0 + i], s[kb]);
      __builtin_amdgcn_sched_barrier(0);
    }
    auto hidden = [&](int key) {  // (no branches: 32 of them per tile and lane)
      return !valid | (key > my_pos) | ((key < my_lo) & ((key >= a.keep) | (key < my_c0))) | (key >= ctx);
    };
    bf16x8_t pb[KBN][2];
    if constexpr (SIG) {
      // x (log2 domain) = s * scale - a log2(1 + b (i - j)) + bias; weight = 1 / (1 + 2^-x); hidden keys weigh 0
#pragma unroll
      for (int kb = 0; kb < KBN; ++kb) {
        float p[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int key = kv0 + kb * 32 + acc_row(i, hh);
          const float dist = (float)max(my_pos - key, 0);
          const float x = s[kb][i] * my_scale - pen_a * __log2f(1.0f + pen_b * dist) + sig_b2;
          const float w = __builtin_amdgcn_rcpf(1.0f + fast_exp2(-x));
          p[i] = hidden(key) ? 0.f : w;
        }
        pb[kb][0] = to_bf16x8(p);
        pb[kb][1] = to_bf16x8(p + 8);
      }
    } else {
      float mx = -INFINITY;
      if (kv0 + KBN * 32 - 1 <= w_first && kv0 >= w_lo_last && kv0 + KBN * 32 - 1 < ctx) {
        // every key is visible to every row of this wave: no mask (rows past the portion's end
        // carry finite scores of a repeated row and are never stored)
#pragma unroll
        for (int kb = 0; kb < KBN; ++kb)
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            if constexpr (CAP) s[kb][i] = a.cap_log2 * (1.0f - 2.0f * __builtin_amdgcn_rcpf(1.0f + fast_exp2(s[kb][i] * a.cap_inv2)));
            else s[kb][i] *= my_scale;
            mx = fmaxf(mx, s[kb][i]);
          }
        if (!valid) mx = -INFINITY;  // such a row must not trigger the wave's rescale
      } else {
#pragma unroll
        for (int kb = 0; kb < KBN; ++kb)
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            float x;
            if constexpr (CAP) x = a.cap_log2 * (1.0f - 2.0f * __builtin_amdgcn_rcpf(1.0f + fast_exp2(s[kb][i] * a.cap_inv2)));
            else x = s[kb][i] * my_scale;
            const int key = kv0 + kb * 32 + acc_row(i, hh);
            x = hidden(key) ? -INFINITY : x;
            s[kb][i] = x;
            mx = fmaxf(mx, x);
          }
      }
      mx = xor32_max(mx);
      const bool grow = __builtin_amdgcn_ballot_w64(mx > m_i + kRescaleTh) != 0;
      const float m_raw = grow ? fmaxf(m_i, mx) : m_i;
      const float m_new = m_raw == -INFINITY ? 0.f : m_raw;  // nothing seen yet (a later split, all keys masked)
      float rs = 0.f;
#pragma unroll
      for (int kb = 0; kb < KBN; ++kb) {
        float p[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          p[i] = fast_exp2(s[kb][i] - m_new);
          rs += p[i];
        }
        pb[kb][0] = to_bf16x8(p);
        pb[kb][1] = to_bf16x8(p + 8);
      }
      rs = xor32_add(rs);
      if (grow) {
        const float alpha = fast_exp2(m_i - m_new);
        l_i *= alpha;
#pragma unroll
        for (int d = 0; d < NDB; ++d)
#pragma unroll
          for (int i = 0; i < 16; ++i) o[d][i] *= alpha;
      }
      l_i += rs;
      m_i = m_raw;
    }
#pragma unroll
    for (int kb = 0; kb < KBN; ++kb)
#pragma unroll
      for (int st = 0; st < 2; ++st)
#pragma unroll
        for (int d = 0; d < NDB; ++d) {
          const bf16x8_t vf = tr_frag_at<128>(Vs + (d >> 2) * LIMG, kb * 32 + 16 * st, tr_lo[d & 3], tr_hi[d & 3]);
          o[d] = mfma32(vf, pb[kb][st], o[d]);
        }
  }

  if constexpr (KG2) {  // the second group's results into the first's, through the images (all of whose fills have landed)
    static_assert(4 * 64 * (NDB * 16 + 2) * 4 <= (DB ? 2 : 1) * BUFB, "LDS");
    float* xs = reinterpret_cast<float*>(smem) + wave * 64 * (NDB * 16 + 2) + lane;
    __syncthreads();
    if (kgrp == 1) {
#pragma unroll
      for (int d = 0; d < NDB; ++d)
#pragma unroll
        for (int i = 0; i < 16; ++i) xs[64 * (d * 16 + i)] = o[d][i];
      xs[64 * NDB * 16] = m_i;
      xs[64 * (NDB * 16 + 1)] = l_i;
    }
    __syncthreads();
    if (kgrp == 1) return;
    const float m_o = xs[64 * NDB * 16], l_o = xs[64 * (NDB * 16 + 1)];
    const float m_both = fmaxf(m_i, m_o), m_ref = m_both == -INFINITY ? 0.f : m_both;
    const float f_i = SIG ? 1.f : fast_exp2(m_i - m_ref), f_o = SIG ? 1.f : fast_exp2(m_o - m_ref);
    l_i = l_i * f_i + l_o * f_o;
    m_i = m_both;
#pragma unroll
    for (int d = 0; d < NDB; ++d)
#pragma unroll
      for (int i = 0; i < 16; ++i) o[d][i] = o[d][i] * f_i + xs[64 * (d * 16 + i)] * f_o;
  }

  if (SPLIT && valid && a.nsplit > 1) {
    const long rowi = (long)n * a.H + my_head;
    float* Wp = a.ws_o + (rowi * a.nsplit + split) * a.rk;
#pragma unroll
    for (int d = 0; d < NDB; ++d)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int col = v0 + d * 32 + 8 * g + 4 * hh;
        if (col < a.rk) *reinterpret_cast<float4*>(Wp + col) = make_float4(o[d][4 * g], o[d][4 * g + 1], o[d][4 * g + 2], o[d][4 * g + 3]);
      }
    if (v0 == 0 && hh == 0) {
      a.ws_ml[(rowi * a.nsplit + split) * 2] = m_i;
      a.ws_ml[(rowi * a.nsplit + split) * 2 + 1] = l_i;
    }
  } else if (valid) {
    const float inv = 1.f / l_i;
    unsigned short* Op = a.out + ((long)(q_begin + my_tok) * a.H + my_head) * a.rk;
    // A copy for either, not a branch in each of its stores: a launch without a gate reads no more code than before.  2048 tokens x 16 heads of 128 columns, a gate each:
    // 53.3 us and a pass of 8.5 for the gate, so 58.9; 600 tokens 21.0 and 4.0, so 27.2 (the sigmoids' code is read once, from memory), but a launch less for the host: lenitar, 700 tokens
    // 939 us with the pass, so 915.
    auto store = [&](auto gated_c) __attribute__((always_inline)) {
      constexpr bool GATED = decltype(gated_c)::value;
      // a lane's gates lie in its own row, 8 bytes at a time: all on their way before the first is used, but for the widest turned values, whose loop stays one (an array that it
      // indexes would lie in scratch memory: 1088 bytes a lane for 576, in launches without a gate too)
      constexpr bool AHEAD = !(ROT && NDB > 4);
      const bf16_t* Gp = a.gate + (long)(q_begin + my_tok) * a.gate_st;
      const bool each = a.gate_per == 1;
      float one = 0.f;
      if constexpr (GATED) one = each ? 0.f : ldf(Gp + my_head);
      auto gates = [&](int col) { return each ? ld4(Gp + (long)my_head * a.rk + min(col, a.rk - 4)) : make_float4(one, one, one, one); };
      float4 gt[GATED && AHEAD ? NDB : 1][4];
      if constexpr (GATED && AHEAD) {
#pragma unroll
        for (int d = 0; d < NDB; ++d)
#pragma unroll
          for (int g = 0; g < 4; ++g) gt[d][g] = gates(v0 + d * 32 + 8 * g + 4 * hh);
      }
#pragma unroll
      for (int d = 0; d < NDB; ++d)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const int col = v0 + d * 32 + 8 * g + 4 * hh;
          if (col < a.rk) {
            if constexpr (ROT) {  // turn the neighbour pairs (col, col + 1), (col + 2, col + 3) back
#pragma unroll
              for (int j = 0; j < 4; j += 2) {
                float sn, cs;
                sincosf((float)my_pos * a.ofreq[(col + j) >> 1], &sn, &cs);
                const float u = o[d][4 * g + j], w = o[d][4 * g + j + 1];
                o[d][4 * g + j] = u * cs + w * sn;
                o[d][4 * g + j + 1] = w * cs - u * sn;
              }
            }
            unsigned short w4[4];
            float4 gv;
            if constexpr (GATED) {
              if constexpr (AHEAD) gv = gt[d][g];
              else gv = gates(col);
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              float v = o[d][4 * g + j] * inv;
              if constexpr (GATED) v = gated(v, (&gv.x)[j]);
              w4[j] = __bfloat16_as_ushort(__float2bfloat16(v));
            }
            *reinterpret_cast<uint2*>(Op + col) =
                make_uint2((unsigned)w4[0] | ((unsigned)w4[1] << 16), (unsigned)w4[2] | ((unsigned)w4[3] << 16));
          }
        }
    };
    if (a.gate != nullptr) store(std::true_type{});
    else store(std::false_type{});
  }
}

template <int NKS, bool SPLIT, bool ROT, bool SIG = false, bool CAP = false>
void launch_ncb(const LArgs& a, int ndb, dim3 grid, hipStream_t st) {
  auto go = [&](auto kern, int NDBv) {
    constexpr int NCB = (NKS + 7) / 8;
    const size_t one = (size_t)(NCB + (NDBv + 3) / 4) * LIMG;
    const size_t lds = (2 * one + 1024 <= 160 * 1024 ? 2 * one : one) + 2 * LKB * sizeof(int);
    HYB_CHECK(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) == hipSuccess, "LDS size");
    kern<<<grid, two_key_groups(NKS, NDBv, SPLIT) ? 512 : 256, lds, st>>>(a);
  };
  if (ndb == 2) go(latent_attn_mfma_kernel<NKS, 2, ROT, SIG, CAP, SPLIT>, 2);
  else if (ndb == 4) go(latent_attn_mfma_kernel<NKS, 4, ROT, SIG, CAP, SPLIT>, 4);
  else go(latent_attn_mfma_kernel<NKS, 8, ROT, SIG, CAP, SPLIT>, 8);
}

template <bool SPLIT>
void launch_form(const LArgs& a, int ncb, int ndb, dim3 grid, const RowAttnOpts& x) {
  hipStream_t st = cur_stream();
  if (x.softcap > 0.0) {  // built for keys up to 256 wide, plain softmax form (the caller checks)
    HYB_CHECK(x.hscale == nullptr && ncb <= 2, "capped scores: no per-head factor, keys up to 256 wide");
    if (ncb == 1) launch_ncb<8, SPLIT, false, false, true>(a, ndb, grid, st);
    else launch_ncb<16, SPLIT, false, false, true>(a, ndb, grid, st);
  } else if (x.sig_bias != nullptr) {  // built for keys up to 256 wide (latent_attn_mfma_ok)
    if (ncb == 1) launch_ncb<8, SPLIT, false, true>(a, ndb, grid, st);
    else launch_ncb<16, SPLIT, false, true>(a, ndb, grid, st);
  } else if (x.ofreq != nullptr) {
    if (ncb == 1) launch_ncb<8, SPLIT, true>(a, ndb, grid, st);
    else launch_ncb<16, SPLIT, true>(a, ndb, grid, st);
  } else {
    switch (ncb) {
      case 1: launch_ncb<8, SPLIT, false>(a, ndb, grid, st); break;
      case 2:
        if (!SPLIT && a.R <= 192) launch_ncb<12, false, false>(a, ndb, grid, st);
        else launch_ncb<16, SPLIT, false>(a, ndb, grid, st);
        break;
      case 3: launch_ncb<24, SPLIT, false>(a, ndb, grid, st); break;
      case 4: launch_ncb<32, SPLIT, false>(a, ndb, grid, st); break;
      default: launch_ncb<40, SPLIT, false>(a, ndb, grid, st); break;
    }
  }
}

// The cut of a call: column blocks of the keys and value tiles, heads and tokens of a workgroup's 128 rows.
struct Cut {
  int ncb, ndb, nvt, HB, hpg;
  Cut(int64_t R, int64_t rk, int64_t P, bool heads) {
    ncb = (int)((R + 127) / 128);
    ndb = rk <= 64 ? 2 : (rk <= 128 ? 4 : 8);
    nvt = (int)((rk + ndb * 32 - 1) / (ndb * 32));
    HB = 1;
    while (heads && HB < P && HB < 128) HB *= 2;
    hpg = (int)((P + HB - 1) / HB);
  }
};

LArgs make_args(const at::Tensor& qa, const at::Tensor& cache, const at::Tensor& bt, const int* cu, const at::Tensor& ctx, int64_t window, const float* sink,
                double scale, int64_t rk, at::Tensor& out, const RowAttnOpts& x, const Cut& c) {
  LArgs a = {};
  a.qa = reinterpret_cast<const unsigned short*>(qa.data_ptr()), a.cache = reinterpret_cast<const unsigned short*>(cache.data_ptr());
  a.out = reinterpret_cast<unsigned short*>(out.data_ptr());
  a.bt = bt.data_ptr<int>(), a.cu = cu, a.ctx = ctx.data_ptr<int>();
  a.sink = sink, a.hscale = x.hscale, a.ofreq = x.ofreq, a.dist_a = x.dist_a, a.dist_b = x.dist_b, a.sig_bias = x.sig_bias;
  a.H = (int)qa.size(1), a.R = (int)qa.size(2), a.rk = (int)rk, a.bs = (int)cache.size(1), a.maxb = (int)bt.size(1), a.window = (int)window;
  a.HB = c.HB, a.nvt = c.nvt, a.G = (int)x.groups, a.rs = (int)(cache.size(2) / x.groups), a.koff = (int)x.koff, a.chunk = (int)x.chunk, a.hpg = c.hpg;
  a.keep = (int)x.keep_first;
  a.scale_log2 = (float)(scale * 1.4426950408889634), a.cap_log2 = (float)(x.softcap * 1.4426950408889634);
  a.cap_inv2 = x.softcap > 0.0 ? (float)(2.0 * 1.4426950408889634 * scale / x.softcap) : 0.f;
  a.nsplit = 1;
  a.gate = x.gate, a.gate_st = x.gate_st, a.gate_per = x.gate_per;
  return a;
}
}  // namespace

// turn_back: the output is to be turned back (RowAttnOpts::ofreq) or the weights are sigmoids
// (RowAttnOpts::sig_bias); those forms are built for keys up to 256 wide
bool latent_attn_mfma_ok(const at::Tensor& qa, int64_t rk, int64_t rs, int64_t koff, bool turn_back) {
  const int64_t R = qa.size(2);
  return qa.scalar_type() == at::kBFloat16 && R % 8 == 0 && rk % 8 == 0 && rs % 8 == 0 && koff % 8 == 0 && R <= (turn_back ? 256 : 640) && qa.size(1) >= 1;
}

// ``x`` carries the optional parts (see RowAttnOpts).
void latent_attn_mfma(const at::Tensor& qa, const at::Tensor& cache, const at::Tensor& bt, const at::Tensor& cu, const at::Tensor& ctx,
                      int64_t window, const float* sink, double scale, int64_t rk, int64_t max_q, at::Tensor& out, const RowAttnOpts& x) {
  const int64_t ns = ctx.numel();
  const Cut c(qa.size(2), rk, qa.size(1) / x.groups, max_q < 64);
  const int TB = 128 / c.HB, z = (int)x.groups * c.hpg * c.nvt;
  HYB_CHECK(ns <= 65535 && z <= 65535, "grid too large");
  LArgs a = make_args(qa, cache, bt, cu.data_ptr<int>(), ctx, window, sink, scale, rk, out, x, c);
  a.xcd = z % 8 == 0 ? 1 : 0;
  launch_form<false>(a, c.ncb, c.ndb, dim3((unsigned)((max_q + TB - 1) / TB), (unsigned)ns, (unsigned)z), x);
}

void row_merge(const at::Tensor& ws_o, const at::Tensor& ws_ml, at::Tensor& out, const at::Tensor& ctx, const RowAttnOpts& x);  // row_decode.hip

// The decode form's cut: the visible key tiles are split over workgroups until the launch has a few hundred of them.  ``images``: 128-column
// images of a tile's keys and values in LDS.
DecodeCut tile_cut(int64_t ns, int64_t H, int64_t R, int64_t rk, int64_t window, const RowAttnOpts& x, int* images) {
  const Cut c(R, rk, H / x.groups, true);
  *images = c.ncb + (c.ndb + 3) / 4;
  const int64_t span = std::min<int64_t>(std::min<int64_t>(window, x.chunk), x.max_ctx > 0 ? x.max_ctx : (int64_t)1 << 30);
  DecodeCut d = {ns * x.groups * c.hpg * c.nvt, 1, std::min<int64_t>((span + LKB - 1) / LKB + 1 + (x.keep_first + LKB - 1) / LKB, 1 << 20)};
  while (d.nsplit < d.steps && d.nsplit < 32 && d.groups * d.nsplit < 512) d.nsplit *= 2;
  return d;
}

// Decode rows: up to 128 heads of a kv group in one tile.
void latent_attn_mfma_decode(const at::Tensor& qa, const at::Tensor& cache, const at::Tensor& bt, const at::Tensor& ctx, int64_t window, const float* sink,
                             double scale, int64_t rk, at::Tensor& out, const RowAttnOpts& x) {
  const int64_t H = qa.size(1), ns = ctx.numel();
  const Cut c(qa.size(2), rk, H / x.groups, true);
  const int z = (int)x.groups * c.hpg * c.nvt;
  HYB_CHECK(ns <= 65535 && z <= 65535, "grid too large");
  LArgs a = make_args(qa, cache, bt, nullptr, ctx, window, sink, scale, rk, out, x, c);
  int images;
  a.nsplit = (int)tile_cut(ns, H, qa.size(2), rk, window, x, &images).nsplit;
  at::Tensor ws_o, ws_ml;
  if (a.nsplit > 1) {
    ws_o = at::empty({ns * H, a.nsplit, rk}, qa.options().dtype(at::kFloat));
    ws_ml = at::empty({ns * H, a.nsplit, 2}, qa.options().dtype(at::kFloat));
    a.ws_o = ws_o.data_ptr<float>(), a.ws_ml = ws_ml.data_ptr<float>();
  }
  launch_form<true>(a, c.ncb, c.ndb, dim3((unsigned)a.nsplit, (unsigned)ns, (unsigned)z), x);
  if (a.nsplit > 1) row_merge(ws_o, ws_ml, out, ctx, x);
}

}  // namespace llmctl_hybrid
