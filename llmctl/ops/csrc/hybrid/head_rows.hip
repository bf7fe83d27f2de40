// Per-head products of a decode step's few rows: y[t, h] = x[t, h] W[h] with W [H, K, N] (N contiguous), for latent attention's two absorbed
// projections, each with what surrounds it in the same launch:
//   latent_q_rows    the query to the cache row's layout: x = the heads' plain part, W = W_uk, and the rotary part turned beside it
//   latent_out_rows  the attention's latent outputs to values: x = the latent rows, W = W_uv^T, times the sigmoid gate
//
// Bound: the launch and one round trip to HBM (16 heads of 128 x 512: 2 MB of weights).  A workgroup owns 32 columns of a head (16 x 16 or
// 4 x 16 workgroups at that size); its four waves split K in steps of 32 rows, which go to LDS by DMA and come back through
// transposing reads (32-byte segments swizzled by the row); the sums meet in LDS.
// Measured at 16 rows, 16 heads, in a graph: 5.0 us each; before, a batched product of 12.4 us and the assembly of 10.4, and one of 5.7, a copy of
// 5.1 and the gate of 4.3.  A lenitar decode step of 16 sequences: 567 -> 489 us.
#include "attn_common.h"
#include "hybrid_common.h"

namespace llmctl_hybrid {
using namespace llmctl::attn;

namespace {
using facc = __attribute__((ext_vector_type(4))) float;
constexpr int NC = 32;    // columns of a workgroup
constexpr int BATCH = 4;  // 32-row steps of a wave in flight

struct HRArgs {
  const bf16_t* x;  // row t, head h at x + t x_st + h x_sh
  int64_t x_st, x_sh;
  const bf16_t* w;  // [H, K, N]
  bf16_t* y;        // row t, head h at y + t y_st + h y_sh
  int64_t y_st, y_sh;
  int T, K, N;
  const bf16_t* gate;  // nullptr, or [T, H * N] (rows g_st apart): y = product * sigmoid(gate)
  int64_t g_st;
  // nullptr, or the rotary part: x[K, K + dr) of every row and head, turned, to y[N, N + dr)
  const int* pos;
  const float* inv_freq;
  int dr, rot_dims, inter;
  float amp;
};

__device__ __forceinline__ facc mfma16(bf16x8_t a, bf16x8_t b, facc c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }
__device__ __forceinline__ int turn(int k) { return (k >> 2) & 1; }

template <int MT>  // tiles of 16 rows
__global__ __launch_bounds__(256) void head_rows_kernel(HRArgs a) {
  __shared__ __attribute__((aligned(16))) unsigned char img[4][BATCH][32 * NC * 2];
  __shared__ facc red[4][2 * MT][64];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, g = lane >> 4, h = blockIdx.y, n0 = blockIdx.x * NC;
  const int K = a.K, N = a.N, steps = (K + 31) / 32;
  const bf16_t* W = a.w + (int64_t)h * K * N + n0;
  const bf16_t* xp[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) xp[m] = a.x + (int64_t)min(16 * m + r, a.T - 1) * a.x_st + h * a.x_sh;
  facc acc[2][MT];
#pragma unroll
  for (int d = 0; d < 2; ++d)
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[d][m] = facc{0.f, 0.f, 0.f, 0.f};
  const int krow = lane >> 2, trow = 4 * g + (r >> 2), toff = trow * (NC * 2) + (r & 3) * 8;
  const unsigned lds_mine = lds_addr(img[wave]);
  for (int s0 = wave; s0 < steps; s0 += 4 * BATCH) {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the last batch's reads of the images
    uint2 xv[BATCH][MT][2];
#pragma unroll
    for (int i = 0; i < BATCH; ++i) {
      const int k0 = (s0 + 4 * i) * 32;
      if (s0 + 4 * i >= steps) break;
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        const int kr = 16 * half + krow;
        const int col = min(((lane & 3) ^ (turn(kr) << 1)) * 8, N - n0 - 8);  // (columns past N repeat the last ones and are not stored)
        dma16(W + (int64_t)min(k0 + kr, K - 1) * N + col, lds_mine + (unsigned)(i * 32 * NC * 2 + half * 1024));
      }
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int half = 0; half < 2; ++half) {  // K is a multiple of 4; rows past it meet zeros here
          const int k = k0 + 16 * half + 4 * g;
          const uint2 v = *reinterpret_cast<const uint2*>(xp[m] + min(k, K - 4));
          xv[i][m][half] = k < K ? v : make_uint2(0, 0);
        }
    }
    vm_wait<0>();
#pragma unroll
    for (int i = 0; i < BATCH; ++i) {
      if (s0 + 4 * i >= steps) break;
#pragma unroll
      for (int d = 0; d < 2; ++d) {
        const unsigned char* at = img[wave][i] + toff + ((d ^ turn(trow)) << 5);  // (16 rows on, the turn is the same)
        const s4_t va = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)at);
        const s4_t vb = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(at + 16 * NC * 2));
        const s8_t v = {va[0], va[1], va[2], va[3], vb[0], vb[1], vb[2], vb[3]};
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          const uint4 x4 = make_uint4(xv[i][m][0].x, xv[i][m][0].y, xv[i][m][1].x, xv[i][m][1].y);
          acc[d][m] = mfma16(__builtin_bit_cast(bf16x8_t, v), __builtin_bit_cast(bf16x8_t, x4), acc[d][m]);
        }
      }
    }
  }
#pragma unroll
  for (int d = 0; d < 2; ++d)
#pragma unroll
    for (int m = 0; m < MT; ++m) red[wave][d * MT + m][lane] = acc[d][m];
  __syncthreads();
  for (int i = tid; i < 2 * MT * 64; i += 256) {
    const int t = i >> 6, l = i & 63, row = 16 * (t % MT) + (l & 15), c = n0 + 16 * (t / MT) + 4 * (l >> 4);
    if (row >= a.T || c >= N) continue;
    facc s = red[0][t][l];
#pragma unroll
    for (int v = 1; v < 4; ++v) s += red[v][t][l];
    bf16_t o[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      stf(o + j, s[j]);
      if (a.gate != nullptr) stf(o + j, ldf(o + j) * (1.0f / (1.0f + expf(-ldf(a.gate + row * a.g_st + (int64_t)h * N + c + j)))));
    }
    bf16_t* y = a.y + row * a.y_st + h * a.y_sh + c;
    *reinterpret_cast<uint2*>(y) = *reinterpret_cast<const uint2*>(o);  // N and the strides are multiples of 4
  }
  if (a.pos == nullptr || blockIdx.x != 0) return;
  const int half = a.rot_dims / 2, per = half + a.dr - a.rot_dims;  // pairs, then entries that are not turned
  for (int i = tid; i < a.T * per; i += 256) {
    const int t = i / per, c = i - t * per;
    const bf16_t* x = a.x + t * a.x_st + h * a.x_sh + K;
    bf16_t* y = a.y + t * a.y_st + h * a.y_sh + N;
    if (c < half) {
      float sn, cs;
      sincosf((float)a.pos[t] * a.inv_freq[c], &sn, &cs);
      cs *= a.amp, sn *= a.amp;
      const int i0 = a.inter ? 2 * c : c, i1 = a.inter ? 2 * c + 1 : c + half;
      const float u = ldf(x + i0), v = ldf(x + i1);
      stf(y + i0, u * cs - v * sn);
      stf(y + i1, v * cs + u * sn);
    } else {
      const int e = a.rot_dims + c - half;
      y[e] = x[e];
    }
  }
}

void hr_launch(const HRArgs& a, int64_t H) {
  HYB_CHECK(H <= 65535, "grid too large");
  const dim3 grid((unsigned)((a.N + NC - 1) / NC), (unsigned)H);
  if (a.T <= 16) head_rows_kernel<1><<<grid, 256, 0, cur_stream()>>>(a);
  else head_rows_kernel<2><<<grid, 256, 0, cur_stream()>>>(a);
}

bool aligned(const void* p, int n) { return reinterpret_cast<uintptr_t>(p) % n == 0; }

void check_head_weight(const at::Tensor& w, const at::Tensor& x, int64_t H, int64_t K) {
  HYB_CHECK(w.is_cuda() && w.dim() == 3 && w.is_contiguous() && w.scalar_type() == at::kBFloat16 && w.size(0) == H && w.size(1) == K &&
                w.size(2) % 8 == 0 && w.size(2) >= 8 && aligned(w.data_ptr(), 16),
            "head weights: contiguous bf16 [H, K, N], N a multiple of 8");
  HYB_CHECK(x.scalar_type() == at::kBFloat16 && K % 4 == 0 && K >= 4 && x.stride(0) % 4 == 0 && x.stride(1) % 4 == 0 && aligned(x.data_ptr(), 8),
            "rows: bf16, K and the strides multiples of 4");
}
}  // namespace

// qa [T, H, rk + dr] = [q[.., :dn] W_uk | turned q[.., dn:]], q [T, H, dn + dr] (row-strided), W_uk [H, dn, rk]; at most 32 rows
at::Tensor latent_q_rows(const at::Tensor& q, const at::Tensor& w_uk, const at::Tensor& pos, const at::Tensor& inv_freq, int64_t rot_dims,
                         bool interleaved, double amp) {
  HYB_CHECK(q.is_cuda() && q.dim() == 3 && q.stride(2) == 1 && q.size(0) >= 1 && q.size(0) <= 32 && w_uk.dim() == 3, "q: 1 to 32 rows [T, H, dn + rot]");
  const int64_t T = q.size(0), H = q.size(1), dn = w_uk.size(1), rk = w_uk.size(2), dr = q.size(2) - dn;
  check_head_weight(w_uk, q, H, dn);
  HYB_CHECK(dr >= 0 && rot_dims % 2 == 0 && rot_dims <= dr && (rk + dr) % 4 == 0, "rotary: even dims <= rot part; rows a multiple of 4");
  HYB_CHECK(inv_freq.is_cuda() && inv_freq.is_contiguous() && inv_freq.scalar_type() == at::kFloat && inv_freq.numel() == rot_dims / 2, "frequencies: fp32 [rot_dims / 2]");
  HYB_CHECK(pos.is_cuda() && pos.is_contiguous() && pos.scalar_type() == at::kInt && pos.numel() == T, "pos: int32 [T]");
  c10::DeviceGuard guard(q.device());
  at::Tensor qa = at::empty({T, H, rk + dr}, q.options());
  HRArgs a = {};
  a.x = (const bf16_t*)q.data_ptr(), a.x_st = q.stride(0), a.x_sh = q.stride(1), a.w = (const bf16_t*)w_uk.data_ptr();
  a.y = (bf16_t*)qa.data_ptr(), a.y_st = H * (rk + dr), a.y_sh = rk + dr, a.T = (int)T, a.K = (int)dn, a.N = (int)rk;
  a.pos = pos.data_ptr<int>(), a.inv_freq = inv_freq.data_ptr<float>(), a.dr = (int)dr, a.rot_dims = (int)rot_dims;
  a.inter = interleaved, a.amp = (float)amp;
  hr_launch(a, H);
  return qa;
}

// [T, H * dv] = (o [T, H, rk] W_uv^T) (* sigmoid(gate)), W_uv^T [H, rk, dv], gate [T, H * dv] (row-strided); at most 32 rows
at::Tensor latent_out_rows(const at::Tensor& o, const at::Tensor& w, const c10::optional<at::Tensor>& gate) {
  HYB_CHECK(o.is_cuda() && o.dim() == 3 && o.stride(2) == 1 && o.size(0) >= 1 && o.size(0) <= 32 && w.dim() == 3, "o: 1 to 32 rows [T, H, rank]");
  const int64_t T = o.size(0), H = o.size(1), K = o.size(2), N = w.size(2);
  check_head_weight(w, o, H, K);
  c10::DeviceGuard guard(o.device());
  at::Tensor y = at::empty({T, H * N}, o.options());
  HRArgs a = {};
  a.x = (const bf16_t*)o.data_ptr(), a.x_st = o.stride(0), a.x_sh = o.stride(1), a.w = (const bf16_t*)w.data_ptr();
  a.y = (bf16_t*)y.data_ptr(), a.y_st = H * N, a.y_sh = N, a.T = (int)T, a.K = (int)K, a.N = (int)N;
  if (gate.has_value()) {
    HYB_CHECK(gate->is_cuda() && gate->dim() == 2 && gate->size(0) == T && gate->size(1) == H * N && gate->stride(1) == 1 && gate->scalar_type() == at::kBFloat16,
              "gate: bf16 [T, H * dv] rows");
    a.gate = (const bf16_t*)gate->data_ptr(), a.g_st = gate->stride(0);
  }
  hr_launch(a, H);
  return y;
}

}  // namespace llmctl_hybrid
