// Attention of decode rows over a paged row cache (bf16; MFMA 16x16x32), with all the options of latent_attn.hip: one query
// row per sequence, up to 16 query heads of one kv group per workgroup.
//
// The prompt kernel (latent_attn_mfma.hip) tiles 128 query rows over its four waves; a decode row fills 4 to 16 of them, so one
// wave multiplied while three waited, over images filled behind two barriers per 64 keys.  Here a workgroup takes 64 keys at a
// time and every wave has a quarter of both products:
//   * scores of 16 keys per wave: the K rows come straight from the cache as MFMA row operands (all column steps in flight), the
//     query fragments stay in registers; the scores meet in LDS (two buffers, so one barrier per 64 keys);
//   * every wave then reads all 64 scores of its lanes' heads in the order of the second product's operand (keys 4 g .. 4 g + 3
//     of two 16-key blocks: any order will do as long as V follows it) and runs the same softmax, so nothing is merged
//     inside a workgroup;
//   * V^T for a quarter of the value columns per wave: those columns of the value rows go to a wave-private LDS image by DMA at the
//     start of the step and come back through transposing reads; 32-byte segments are swizzled by the row (no bank conflicts);
//   * only visible keys are addressed (kept first keys, then the window), so nothing is masked but the last step's tail.
// The key steps of a sequence are spread over ``nsplit`` workgroups; row_merge_kernel joins them.
//
// Bound: the cache stream for many sequences, else the chain slot -> rows -> product -> merge launch.  Measured, kernel and merge, us,
// one MI355X (before: the prompt kernel with one row per tile), 16 query heads:
//   key / value width, kv groups   sequences x context:  4 x 128       16 x 1024     16 x 4096     64 x 4096
//   576 / 512, 1                                         12.4 (21.5)   18.0 (55.2)   35.1 (97.3)   87.5 (259, 3.5 TB/s now)
//   256 / 256, 2                                          8.3 (13.7)   13.7 (33.5)   33.2 (60.9)   106 (156, 5.1 TB/s now)
//   128 / 128, 4                                          7.1 (9.0)    11.9 (22.0)   30.6 (48.3)   99.6 (146, 5.4 TB/s now)
// (The form for keys of 257 to 576 columns fills its 256 registers and spills one vector and eleven scalar registers, 8 bytes of scratch a lane; the
// first row was measured with that.)
#include "attn_common.h"
#include "hybrid_common.h"

namespace llmctl_hybrid {
using namespace llmctl::attn;

namespace {
using facc = __attribute__((ext_vector_type(4))) float;
constexpr float kLog2e = 1.4426950408889634f;
constexpr int KEYS = 64;  // keys of a step
constexpr int WAVES = 4;

struct RArgs {
  const unsigned short* qa;  // [ns, H, R]
  const unsigned short* cache;
  unsigned short* out;       // [ns, H, rk]
  const int* bt;
  const int* ctx;
  const float* sink;
  const float* hscale;
  const float* ofreq;
  const float* dist_a;
  const float* dist_b;
  const float* sig_bias;
  int H, R, rk, bs, bs_shift, maxb, window, chunk, keep, G, rs, koff, htiles, nvt, nsplit;
  float scale_log2, cap_log2, cap_inv2;
  float* ws_o;   // [ns * H, nsplit, rk]
  float* ws_ml;  // [ns * H, nsplit, 2]
};

__device__ __forceinline__ facc mfma16(bf16x8_t a, bf16x8_t b, facc c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }

// Turn neighbour pairs (c, c + 1) of four columns from c on back by -pos * freq.
__device__ __forceinline__ void turn_back(float (&v)[4], const float* ofreq, float pos, int c) {
#pragma unroll
  for (int j = 0; j < 4; j += 2) {
    float sn, cs;
    sincosf(pos * ofreq[(c + j) >> 1], &sn, &cs);
    const float u = v[j], w = v[j + 1];
    v[j] = u * cs + w * sn;
    v[j + 1] = w * cs - u * sn;
  }
}

__device__ __forceinline__ void gate4(float (&v)[4], const bf16_t* row, int per, int head, int rk, int c) {
  const float4 g = per == 1 ? ld4(row + (long)head * rk + c) : make_float4(ldf(row + head), 0.f, 0.f, 0.f);
#pragma unroll
  for (int j = 0; j < 4; ++j) v[j] = gated(v[j], per == 1 ? (&g.x)[j] : g.x);
}

__device__ __forceinline__ void store4(unsigned short* p, const float (&v)[4]) {
  unsigned short h[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) h[j] = __bfloat16_as_ushort(__float2bfloat16(v[j]));
  *reinterpret_cast<uint2*>(p) = make_uint2(h[0] | ((unsigned)h[1] << 16), h[2] | ((unsigned)h[3] << 16));
}

// NK 32-column steps of the key (R <= 32 NK), NV tiles of 16 value columns (wider values: tiles over blockIdx.z)
template <int NK, int NV>
__global__ __launch_bounds__(WAVES * 64, NK > 18 ? 1 : 2) void row_decode_kernel(RArgs a) {
  constexpr int VW = NV * 16 / WAVES;     // value columns of a wave
  constexpr int VT = VW / 16;             // ... in tiles of 16 (32-byte segments of an image row): 2, 4 or 8
  constexpr int RB = VW * 2, IMG = KEYS * RB, RPI = 1024 / RB;  // bytes of an image row and of the image, rows per DMA instruction
  constexpr int SLD = KEYS + 4;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  float* const sbuf = reinterpret_cast<float*>(smem + WAVES * IMG);  // [2][16 heads][SLD]
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int n = blockIdx.y, split = blockIdx.x;
  const int v0 = (int)(blockIdx.z % a.nvt) * (NV * 16) + wave * VW, vcols = min(VW, a.rk - v0);  // this wave's value columns (maybe none)
  const int ht = blockIdx.z / a.nvt, grp = ht / a.htiles, h0 = (ht % a.htiles) * 16;
  const int P = a.H / a.G;                            // query heads per kv group
  const int heads = min(16, P - h0);
  const int head = grp * P + h0 + min(r, heads - 1);  // (columns past the last head repeat it and are never stored)
  const int ctx = a.ctx[n], pos = ctx - 1;
  const int* btn = a.bt + (long)n * a.maxb;
  // the visible keys: [c0, c0 + n_kept) that the window spares, then [lo, ctx)
  const int c0 = max((pos / a.chunk) * a.chunk, 0);
  const int lo = max(max(pos - a.window + 1, c0), 0);
  const int n_kept = max(min(a.keep, lo) - c0, 0);
  const int nkeys = n_kept + ctx - lo;
  const int steps = (nkeys + KEYS - 1) / KEYS, per = (steps + a.nsplit - 1) / a.nsplit;
  const int st_end = min(steps, (split + 1) * per);
  auto slot_of = [&](int st) {  // cache row of key ``lane`` of a step (the last key again past the end)
    const int ki = min(st * KEYS + lane, nkeys - 1);
    const int key = ki < n_kept ? c0 + ki : lo + ki - n_kept;
    const int blk = a.bs_shift >= 0 ? key >> a.bs_shift : key / a.bs;
    return btn[blk] * a.bs + (key - blk * a.bs);
  };
  int slot = split * per < st_end ? slot_of(split * per) : 0;

  // column steps: 8 g on from ks * 32, but in the last step and past it, where a lane stays inside the row
  const int klast = (a.R - 1) / 32 * 32, klane = klast + min(8 * g, a.R - 8 - klast);
  auto kcol = [&](const unsigned short* row, const unsigned short* last, int ks) { return gload16(ks * 32 < klast ? row + ks * 32 : last); };
  bf16x8_t qf[NK];
  {
    const unsigned short* Qp = a.qa + ((long)n * a.H + head) * a.R;
    uint4 v[NK];
#pragma unroll
    for (int ks = 0; ks < NK; ++ks) v[ks] = kcol(Qp + 8 * g, Qp + klane, ks);
#pragma unroll
    for (int ks = 0; ks < NK; ++ks) {
      const unsigned live = ks * 32 + 8 * g < a.R ? ~0u : 0u;  // zero past R
      v[ks].x &= live, v[ks].y &= live, v[ks].z &= live, v[ks].w &= live;
      qf[ks] = __builtin_bit_cast(bf16x8_t, v[ks]);
    }
  }
  const bool sig = a.sig_bias != nullptr;
  const float my_scale = a.scale_log2 * (a.hscale != nullptr ? a.hscale[head] : 1.0f);
  const float pen_a = sig && a.dist_a != nullptr ? a.dist_a[head] : 0.f, pen_b = sig && a.dist_a != nullptr ? a.dist_b[head] : 0.f;
  const float sig_b2 = sig ? a.sig_bias[head] * kLog2e : 0.f;
  // running maximum and denominator: the sink is one unit of mass at its own logit, counted by the first split; sigmoid
  // weights are not normalised (m = 0, and l = 1 in the first split)
  float m_i = -INFINITY, l_i = 0.f;
  if (sig) m_i = 0.f, l_i = split == 0 ? 1.f : 0.f;
  else if (a.sink != nullptr && split == 0) m_i = a.sink[head] * kLog2e, l_i = 1.f;
  facc o[VT];
#pragma unroll
  for (int d = 0; d < VT; ++d) o[d] = facc{0.f, 0.f, 0.f, 0.f};

  unsigned char* const mine = smem + wave * IMG;
  const unsigned lds_mine = lds_addr(smem) + (unsigned)(wave * IMG);
  // swizzle: segment s of image row k lies at s ^ turn(k), so that eight rows in turn cover all banks
  auto turn = [](int k) { return (k / (8 / VT)) & (VT - 1); };
  // transposing reads: lane (q, p) of a 16-lane group addresses row 4 g + q of a 16-key block, columns 4 p .. of a segment
  const int trow = 4 * g + (r >> 2), tturn = turn(trow), toff = trow * RB + (r & 3) * 8;
  const int frow = lane / (64 / RPI), fcol = lane % (64 / RPI);  // this lane's row and 16-byte piece in a DMA instruction

  for (int st = split * per; st < st_end; ++st) {
    const int left = nkeys - st * KEYS;  // keys of this step that exist
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the last step's reads of the image
    if (vcols > 0) {
#pragma unroll
      for (int i = 0; i < KEYS / RPI; ++i) {
        const int k = i * RPI + frow;
        const unsigned short* Vp = a.cache + ((long)__shfl(slot, k) * a.G + grp) * a.rs + v0;
        dma16(Vp + min((fcol ^ (turn(k) << 1)) * 8, vcols - 8), lds_mine + (unsigned)(i * 1024));
      }
    }
    {
      const unsigned short* Kp = a.cache + ((long)__shfl(slot, wave * 16 + r) * a.G + grp) * a.rs + a.koff;
      asm volatile("" : "+v"(Kp));  // (cache + column is loop-invariant; hoisted as such it takes two registers per load)
      uint4 kf[NK];
#pragma unroll
      for (int ks = 0; ks < NK; ++ks) kf[ks] = kcol(Kp + 8 * g, Kp + klane, ks);  // (past R: the query is zero there)
      if (st + 1 < st_end) slot = slot_of(st + 1);
      facc s = facc{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < NK; ++ks) s = mfma16(__builtin_bit_cast(bf16x8_t, kf[ks]), qf[ks], s);
      *reinterpret_cast<float4*>(sbuf + ((st & 1) * 16 + r) * SLD + wave * 16 + 4 * g) = make_float4(s[0], s[1], s[2], s[3]);
    }
    __syncthreads();
    float p[KEYS / 4];  // lane: keys b * 16 + 4 g + i of the step, head r
#pragma unroll
    for (int b = 0; b < KEYS / 16; ++b) {
      const float4 x = *reinterpret_cast<const float4*>(sbuf + ((st & 1) * 16 + r) * SLD + b * 16 + 4 * g);
      p[b * 4] = x.x, p[b * 4 + 1] = x.y, p[b * 4 + 2] = x.z, p[b * 4 + 3] = x.w;
    }
    if (sig) {
      const bool pen = a.dist_a != nullptr;
#pragma unroll
      for (int j = 0; j < KEYS / 4; ++j) {
        const int kk = (j >> 2) * 16 + 4 * g + (j & 3), at = st * KEYS + kk;
        const float dist = (float)(pos - (at < n_kept ? c0 + at : lo + at - n_kept));
        const float x = p[j] * my_scale - (pen ? pen_a * __log2f(1.0f + pen_b * fmaxf(dist, 0.f)) : 0.f) + sig_b2;
        p[j] = kk < left ? __builtin_amdgcn_rcpf(1.0f + fast_exp2(-x)) : 0.f;
      }
    } else {
      if (a.cap_log2 > 0.f) {
#pragma unroll
        for (int j = 0; j < KEYS / 4; ++j) p[j] = a.cap_log2 * (1.0f - 2.0f * __builtin_amdgcn_rcpf(1.0f + fast_exp2(p[j] * a.cap_inv2)));
      } else {
#pragma unroll
        for (int j = 0; j < KEYS / 4; ++j) p[j] *= my_scale;
      }
      float mx = -INFINITY;
#pragma unroll
      for (int j = 0; j < KEYS / 4; ++j) {
        float x = p[j];
        if ((j >> 2) * 16 + 4 * g + (j & 3) >= left) x = -INFINITY;
        p[j] = x;
        mx = fmaxf(mx, x);
      }
      mx = fmaxf(mx, __shfl_xor(mx, 16));
      mx = fmaxf(mx, __shfl_xor(mx, 32));
      const float m_new = fmaxf(m_i, mx);  // finite: the step has a key
      const float alpha = fast_exp2(m_i - m_new);
      float sum = 0.f;
#pragma unroll
      for (int j = 0; j < KEYS / 4; ++j) {
        p[j] = fast_exp2(p[j] - m_new);
        sum += p[j];
      }
      sum += __shfl_xor(sum, 16);
      sum += __shfl_xor(sum, 32);
      l_i = l_i * alpha + sum;
      m_i = m_new;
#pragma unroll
      for (int d = 0; d < VT; ++d) o[d] *= alpha;
    }
    vm_wait<0>();  // the step's value rows are in LDS
#pragma unroll
    for (int b = 0; b < KEYS / 32; ++b) {
      const float (&p8)[8] = *reinterpret_cast<const float (*)[8]>(p + 8 * b);
      const bf16x8_t pb = to_bf16x8(p8);
#pragma unroll
      for (int d = 0; d < VT; ++d) {
        const unsigned char* at = mine + b * 32 * RB + toff + ((d ^ tturn) << 5);  // (16 and 32 rows on, the turn is the same)
        const s4_t va = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)at);
        const s4_t vb = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(at + 16 * RB));
        const s8_t v = {va[0], va[1], va[2], va[3], vb[0], vb[1], vb[2], vb[3]};
        o[d] = mfma16(__builtin_bit_cast(bf16x8_t, v), pb, o[d]);
      }
    }
  }
  // o[d][i]: value column v0 + 16 d + 4 g + i of head r
  if (r >= heads) return;
  const long row = (long)n * a.H + head;
  const float inv = 1.f / l_i;
#pragma unroll
  for (int d = 0; d < VT; ++d) {
    const int c = d * 16 + 4 * g;
    if (c >= vcols) continue;
    if (a.nsplit > 1) {
      *reinterpret_cast<float4*>(a.ws_o + (row * a.nsplit + split) * a.rk + v0 + c) = make_float4(o[d][0], o[d][1], o[d][2], o[d][3]);
    } else {
      float v[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = o[d][j] * inv;
      if (a.ofreq != nullptr) turn_back(v, a.ofreq, (float)pos, v0 + c);
      store4(a.out + row * a.rk + v0 + c, v);
    }
  }
  if (a.nsplit > 1 && v0 == 0 && g == 0) {
    a.ws_ml[(row * a.nsplit + split) * 2] = m_i;
    a.ws_ml[(row * a.nsplit + split) * 2 + 1] = l_i;
  }
}

// out[row] = sum_s o_s 2^(m_s - M) / sum_s l_s 2^(m_s - M), M = max_s m_s (splits that saw nothing: m = -inf, l = 0).  One workgroup
// per row: the splits' factors once (a lane each), then four columns a thread.
__global__ __launch_bounds__(128) void row_merge_kernel(const float* __restrict__ ws_o, const float* __restrict__ ws_ml, unsigned short* __restrict__ out,
                                                        int nsplit, int rk, const float* __restrict__ ofreq, const int* __restrict__ ctx, int H, const bf16_t* __restrict__ gate,
                                                        long gate_st, int gate_per) {
  __shared__ float fac[64];
  constexpr int B = 8;  // splits asked for at once, the first of them before their factors are there
  const long row = blockIdx.x;
  float4 x[B];
  auto load = [&](int s0, int c) {
#pragma unroll
    for (int u = 0; u < B; ++u)
      if (s0 + u < nsplit && c < rk) x[u] = *reinterpret_cast<const float4*>(ws_o + (row * nsplit + s0 + u) * rk + c);
  };
  load(0, threadIdx.x * 4);
  if (threadIdx.x < 64) {
    const int s = threadIdx.x;
    const float m = s < nsplit ? ws_ml[(row * nsplit + s) * 2] : -INFINITY, l = s < nsplit ? ws_ml[(row * nsplit + s) * 2 + 1] : 0.f;
    const float M = wave_max(m);
    const float f = m == -INFINITY ? 0.f : fast_exp2(m - M);
    const float L = wave_sum(l * f);
    fac[s] = f / L;
  }
  __syncthreads();
  for (int c = threadIdx.x * 4; c < rk; c += 512) {
    float v[4] = {0.f, 0.f, 0.f, 0.f};
    for (int s0 = 0; s0 < nsplit; s0 += B) {  // (a split that saw nothing wrote zeros)
      if (s0 > 0 || c >= 512) load(s0, c);
#pragma unroll
      for (int u = 0; u < B; ++u) {
        if (s0 + u >= nsplit) break;
        const float f = fac[s0 + u];
        v[0] = fmaf(x[u].x, f, v[0]), v[1] = fmaf(x[u].y, f, v[1]), v[2] = fmaf(x[u].z, f, v[2]), v[3] = fmaf(x[u].w, f, v[3]);
      }
    }
    if (ofreq != nullptr) turn_back(v, ofreq, (float)(ctx[row / H] - 1), c);
    if (gate != nullptr) gate4(v, gate + row / H * gate_st, gate_per, (int)(row % H), rk, c);
    store4(out + row * rk + c, v);
  }
}
}  // namespace

// Joins the splits of decode rows: ws_o [ns H, nsplit, rk], ws_ml [ns H, nsplit, 2] -> out [ns, H, rk]; at most 64 splits
void row_merge(const at::Tensor& ws_o, const at::Tensor& ws_ml, at::Tensor& out, const at::Tensor& ctx, const RowAttnOpts& x) {
  row_merge_kernel<<<dim3((unsigned)ws_o.size(0)), 128, 0, cur_stream()>>>(ws_o.data_ptr<float>(), ws_ml.data_ptr<float>(),
                                                                         reinterpret_cast<unsigned short*>(out.data_ptr()), (int)ws_o.size(1), (int)ws_o.size(2), x.ofreq,
                                                                         ctx.data_ptr<int>(), (int)out.size(1), x.gate, (long)x.gate_st, x.gate_per);
}

namespace {
int value_tiles(int64_t R, int64_t rk) { return R <= 128 && rk <= 128 ? 8 : (R <= 256 && rk <= 256 ? 16 : 32); }

// The key steps go to further workgroups until the launch has two per CU: a CU draws about 30 GB/s of a chain of dependent loads,
// and the merge of 64 splits costs 2 to 3 us (unrolled: its loads run together).
DecodeCut row_cut(int64_t ns, int64_t H, int64_t R, int64_t rk, int64_t window, const RowAttnOpts& x) {
  const int64_t nv = value_tiles(R, rk), span = std::min<int64_t>(std::min<int64_t>(window, x.chunk), x.max_ctx > 0 ? x.max_ctx : (int64_t)1 << 30) + x.keep_first;
  DecodeCut d = {ns * x.groups * ((H / x.groups + 15) / 16) * ((rk + nv * 16 - 1) / (nv * 16)), 1, (span + KEYS - 1) / KEYS};
  while (d.nsplit < d.steps && d.nsplit < 64 && d.groups * d.nsplit < 512) d.nsplit *= 2;
  return d;
}
}  // namespace

DecodeCut tile_cut(int64_t ns, int64_t H, int64_t R, int64_t rk, int64_t window, const RowAttnOpts& x, int* images);  // latent_attn_mfma.hip

// Are decode rows faster in tiles of up to 128 heads (latent_attn_mfma_decode) than 16 heads at a time?  More than 32 heads of a kv group read each
// key row three times and more here, which costs more than the tiles' idle rows and longer chain once there are enough keys.  ``most``: keys that a row's block table holds.
// us, here / in tiles, one kv group, 128 heads: 576 / 512 wide, 16 rows x 1000 39 / 59, x 4000 101 / 100, x 32000 735 / 527, 64 x 4000 372 / 289, 256 x 500
// 214 / 152; 128 / 128 wide, 16 x 4000 36 / 21, 64 x 8000 216 / 66; 320 / 256 wide, 64 x 500 49 / 54, 64 x 8000 576 / 199.  64 heads: 576 / 512 64 x 8000 394 / 489, 256 /
// 256 64 x 8000 181 / 145.  Both costs are estimated, us = launches + steps in all (at the rate of a full chip) + the steps of one workgroup + the merge, fitted to
// 896 calls each (1 to 256 rows of 128 to 128000 keys, 40 to 256 heads of 64 to 640 wide keys); the choice is 0.7 % off the faster form on average.
bool decode_tiles_pay(int64_t ns, int64_t H, int64_t R, int64_t rk, int64_t window, const RowAttnOpts& x, int64_t most) {
  if (H / x.groups <= 32) return false;
  int images;
  const DecodeCut r = row_cut(ns, H, R, rk, window, x), t = tile_cut(ns, H, R, rk, window, x, &images);
  const int64_t steps = std::min<int64_t>(r.steps, (most + KEYS - 1) / KEYS);
  const double merge = 2e-6 * (double)(ns * H * rk);  // per split
  const int nv = value_tiles(R, rk);
  double row = nv == 8 ? 7.0 : (nv == 16 ? 9.5 : 13.0);
  row += (nv == 8 ? 0.93 : (nv == 16 ? 2.4 : (R <= 576 ? 3.2 + 0.005 * (double)R : 11.0))) * (double)(r.groups * steps) / 512.0;
  row += (nv == 8 ? 0.65 : 0.0) * (double)((steps + r.nsplit - 1) / r.nsplit) + (r.nsplit > 1 ? merge * (double)r.nsplit : 0.0);
  static const double all[6] = {0.42, 1.5, 2.3, 3.1, 4.1, 5.4}, chain[6] = {1.75, 2.1, 3.2, 3.6, 3.6, 4.2};  // by images, 2 to 7
  const int i = std::min(std::max(images, 2), 7) - 2;
  const double tile = 5.5 + 1.7 * images + all[i] * (double)(t.groups * steps) / 256.0 + chain[i] * (double)((steps + t.nsplit - 1) / t.nsplit) +
                      (t.nsplit > 1 ? merge * (double)t.nsplit : 0.0);
  return row > tile;
}

// Keys up to 640 wide; keys, values, sub-rows and the key offset in multiples of 8 (latent_attn_mfma_ok).  True: the gate, if any, is in the output (the merge applies it;
// rows of one split are left to a pass of its own: the widest form has no registers for it).
bool row_decode(const at::Tensor& qa, const at::Tensor& cache, const at::Tensor& bt, const at::Tensor& ctx, int64_t window, const float* sink,
                double scale, int64_t rk, at::Tensor& out, const RowAttnOpts& x) {
  const int64_t ns = qa.size(0), H = qa.size(1), R = qa.size(2), G = x.groups, P = H / G, rs = cache.size(2) / G;
  const int htiles = (int)((P + 15) / 16);
  const int nv = value_tiles(R, rk);
  const int nvt = (int)((rk + nv * 16 - 1) / (nv * 16));
  HYB_CHECK(ns <= 65535 && G * htiles * nvt <= 65535, "grid too large");
  const int nsplit = (int)row_cut(ns, H, R, rk, window, x).nsplit;
  at::Tensor ws_o, ws_ml;
  if (nsplit > 1) {
    ws_o = at::empty({ns * H, nsplit, rk}, qa.options().dtype(at::kFloat));
    ws_ml = at::empty({ns * H, nsplit, 2}, qa.options().dtype(at::kFloat));
  }
  const int bs = (int)cache.size(1);
  int shift = -1;
  if ((bs & (bs - 1)) == 0) shift = __builtin_ctz((unsigned)bs);
  RArgs a{reinterpret_cast<const unsigned short*>(qa.data_ptr()), reinterpret_cast<const unsigned short*>(cache.data_ptr()),
          reinterpret_cast<unsigned short*>(out.data_ptr()), bt.data_ptr<int>(), ctx.data_ptr<int>(), sink, x.hscale, x.ofreq, x.dist_a, x.dist_b,
          x.sig_bias, (int)H, (int)R, (int)rk, bs, shift, (int)bt.size(1), (int)window, (int)x.chunk, (int)x.keep_first, (int)G, (int)rs, (int)x.koff,
          htiles, nvt, nsplit, (float)(scale * 1.4426950408889634), (float)(x.softcap * 1.4426950408889634),
          x.softcap > 0.0 ? (float)(2.0 * 1.4426950408889634 * scale / x.softcap) : 0.f, nsplit > 1 ? ws_o.data_ptr<float>() : nullptr,
          nsplit > 1 ? ws_ml.data_ptr<float>() : nullptr};
  const dim3 grid((unsigned)nsplit, (unsigned)ns, (unsigned)(G * htiles * nvt));
  const hipStream_t st = cur_stream();
  auto go = [&](auto kern, int nv) {
    const int lds = KEYS * nv * 32 + 2 * 16 * (KEYS + 4) * 4;
    if (lds > 64 * 1024)
      HYB_CHECK(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds) == hipSuccess, "LDS size");
    kern<<<grid, WAVES * 64, lds, st>>>(a);
  };
  if (nv == 8) go(row_decode_kernel<4, 8>, 8);
  else if (nv == 16) go(row_decode_kernel<8, 16>, 16);
  else if (R <= 576) go(row_decode_kernel<18, 32>, 32);
  else go(row_decode_kernel<20, 32>, 32);
  if (nsplit > 1) row_merge(ws_o, ws_ml, out, ctx, x);
  return nsplit > 1;
}

}  // namespace llmctl_hybrid
