// Gradient of an embedding table: g[v] (+)= the sum of dy's rows whose token is v.
//
// Bound: one pass over dy and the rows of g that it meets (8192 x 4096: 134 MB, 27 us at a copy's rate).  Three launches (one for few tokens), no atomics, the same bits
// every time:
//   order  the tokens ranked by (id, position): ids in LDS, every wave counts for two tokens the ids below and the equal ones before and in all.  T^2 compares,
//          four a lane and read; 65536 tokens are the most that is taken here, and of narrow rows fewer pay (embed_grad_pays); a radix sort is five launches.
//   rows   a wave per 8 sorted tokens and 512 columns, all loads in flight; a run of one id inside the 8 is final, a run across an edge leaves a partial row
//   edges  the wave whose 8 a crossing run starts in adds the partial rows in order
// so a token that fills half the batch is summed by as many waves as any other half.
// Measured on one MI355X, us, against the library's (sort, segments, scatter into a dense gradient that is then added), ids drawn evenly / all the same:
// 8192 x 768 into 50304 rows 29.4 / 109 (141 / 329), 8192 x 4096 into 32000 49.7 / 200 (468 / 555), 24576 x 4096 230 / 434 (947 / 1179), 65536 x 4096
// 1011 / 1939 (1495 / 3232), 256 x 256 into 512 3.8 / 7.5 (256 x 64 18.5 / 26); ids drawn as 1 / rank, 8192 x 768 into 50304 47 (152),
// 8192 x 4096 into 32000 103 (451).  16 tokens a wave: 40.8, 75, 283, 1091, 17.3, and less only where most tokens are the
// same (72, 104, 406, 1538, 16): a wave adds to the rows of its ids one after the other.
#include "common.h"

namespace llmctl {
namespace {
constexpr int FEW_IDS = 384;  // tokens of one launch: 256 tokens 50304 x 768, ids drawn evenly / half of them the same / all, 11.1 / 12.9 / 12.0 us in three, so 3.8 / 6.0 / 8.3; 512 of 4096 11.7 / 14.8 / 16.5, so
// 10.3 / 11.9 / 17.8
constexpr int RUN = 8, ORDER_IDS = 16384, ORDER_WAVES = 16;

struct EmbedGradArgs {
  const int64_t* ids;
  const unsigned short* dy;
  void* g;
  int* sid;   // [T] ids in order
  int* perm;  // [T] their positions
  int* end;   // [T] where the run of this id ends
  float* part;  // [chunks][2][H]: the run that enters a chunk, the run that starts in it and leaves
  long dy_ld, V;
  int T, H, add;
};

__global__ __launch_bounds__(64 * ORDER_WAVES) void embed_order_kernel(EmbedGradArgs a) {
  __shared__ __attribute__((aligned(16))) int s[ORDER_IDS];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, T = a.T;
  const int t0 = (blockIdx.x * ORDER_WAVES + w) * 2, t1 = t0 + 1;
  const int v0 = t0 < T ? (int)a.ids[t0] : 0, v1 = t1 < T ? (int)a.ids[t1] : 0;
  int lt0 = 0, lt1 = 0, eq0 = 0, eq1 = 0, all0 = 0, all1 = 0;
  for (int base = 0; base < T; base += ORDER_IDS) {
    const int n = min(ORDER_IDS, T - base), n4 = (n + 3) / 4;
    __syncthreads();
    for (int i = threadIdx.x; i < n4 * 4; i += 64 * ORDER_WAVES) s[i] = i < n ? (int)a.ids[base + i] : 0x7fffffff;  // past every id
    __syncthreads();
#pragma unroll 2
    for (int i = lane; i < n4; i += 64) {
      const int4 q = *reinterpret_cast<const int4*>(s + 4 * i);
      const int x[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int p = base + 4 * i + j;
        lt0 += x[j] < v0;
        lt1 += x[j] < v1;
        all0 += x[j] == v0;
        all1 += x[j] == v1;
        eq0 += x[j] == v0 && p < t0;
        eq1 += x[j] == v1 && p < t1;
      }
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    lt0 += __shfl_xor(lt0, o);
    lt1 += __shfl_xor(lt1, o);
    all0 += __shfl_xor(all0, o);
    all1 += __shfl_xor(all1, o);
    eq0 += __shfl_xor(eq0, o);
    eq1 += __shfl_xor(eq1, o);
  }
  if (lane < 2) {
    const int t = lane ? t1 : t0, at = lane ? lt1 + eq1 : lt0 + eq0;
    if (t < T) {
      a.sid[at] = lane ? v1 : v0;
      a.perm[at] = t;
      a.end[at] = lane ? lt1 + all1 : lt0 + all0;
    }
  }
}

// the finished sum of id's row, 8 columns from c
template <typename G>
__device__ __forceinline__ void put_row(const EmbedGradArgs& a, int id, int c, float* v) {
  if (id < 0 || id >= a.V) return;  // (the forward refuses such ids)
  G* p = static_cast<G*>(a.g) + (long)id * a.H + c;
  if constexpr (sizeof(G) == 2) {
    if (a.add) {
      float old[8];
      load8(p, old);
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] += old[j];
    }
    store8(p, v);
  } else {
#pragma unroll
    for (int j = 0; j < 8; ++j) p[j] = a.add ? p[j] + v[j] : v[j];
  }
}

template <typename G>
__global__ __launch_bounds__(256) void embed_rows_grad_kernel(EmbedGradArgs a) {
  const int c = (blockIdx.y * 64 + (threadIdx.x & 63)) * 8;
  const int p0 = __builtin_amdgcn_readfirstlane((blockIdx.x * 4 + (threadIdx.x >> 6)) * RUN), n = min(RUN, a.T - p0);
  if (n <= 0 || c >= a.H) return;
  uint4 row[RUN];
#pragma unroll
  for (int i = 0; i < RUN; ++i) row[i] = *reinterpret_cast<const uint4*>(a.dy + (long)a.perm[p0 + min(i, n - 1)] * a.dy_ld + c);
  const bool enters = p0 > 0 && a.sid[p0 - 1] == a.sid[p0];
  float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  int start = 0;
#pragma unroll
  for (int i = 0; i < RUN; ++i) {
    if (i >= n) break;
    const unsigned u[4] = {row[i].x, row[i].y, row[i].z, row[i].w};
#pragma unroll
    for (int j = 0; j < 4; ++j) v[2 * j] += bf2f(u[j] & 0xffff), v[2 * j + 1] += bf2f(u[j] >> 16);
    const int id = a.sid[p0 + i], end = a.end[p0 + i];
    if (i < n - 1 && end > p0 + i + 1) continue;
    const bool in = start == 0 && enters, out = end > p0 + i + 1;
    if (in || out) {
      float* q = a.part + ((long)(p0 / RUN) * 2 + (in ? 0 : 1)) * a.H + c;
#pragma unroll
      for (int j = 0; j < 8; j += 4) *reinterpret_cast<float4*>(q + j) = make_float4(v[j], v[j + 1], v[j + 2], v[j + 3]);
    } else {
      put_row<G>(a, id, c, v);
    }
    start = i + 1;
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = 0.f;
  }
}

template <typename G>
__global__ __launch_bounds__(256) void embed_edges_kernel(EmbedGradArgs a) {
  const int c = (blockIdx.y * 64 + (threadIdx.x & 63)) * 8;
  const int k = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6)), p0 = k * RUN, last = p0 + RUN - 1;
  if (last >= a.T || c >= a.H) return;  // (the last chunk's runs all end)
  const int id = a.sid[last], end = a.end[last];
  if (end <= last + 1 || (p0 > 0 && a.sid[p0 - 1] == id)) return;
  float v[8];
  auto take = [&](long part, bool first) {
    const float* q = a.part + part * a.H + c;
#pragma unroll
    for (int j = 0; j < 8; j += 4) {
      const float4 x = *reinterpret_cast<const float4*>(q + j);
      v[j] = first ? x.x : v[j] + x.x;
      v[j + 1] = first ? x.y : v[j + 1] + x.y;
      v[j + 2] = first ? x.z : v[j + 2] + x.z;
      v[j + 3] = first ? x.w : v[j + 3] + x.w;
    }
  };
  take(2L * k + 1, true);
  const int k1 = (end - 1) / RUN;
#pragma unroll 8
  for (int i = k + 1; i <= k1; ++i) take(2L * i, false);
  put_row<G>(a, id, c, v);
}
// Few tokens, one launch: a workgroup per token and 512 columns, ids in LDS; that of an id's first token sums its rows, every wave a quarter of the places, up to
// sixteen rows in flight, in eights (as the three launches do).
template <typename G>
__global__ __launch_bounds__(256) void embed_few_kernel(EmbedGradArgs a) {
  __shared__ int s[FEW_IDS];
  __shared__ __attribute__((aligned(16))) float part[3][64][8];
  const int T = a.T, lane = threadIdx.x & 63, wave = threadIdx.x >> 6, t = blockIdx.x;
  for (int i = threadIdx.x; i < T; i += 256) s[i] = (int)a.ids[i];
  __syncthreads();
  const int id = s[t], c = (blockIdx.y * 64 + lane) * 8, cl = min(c, a.H - 8);
  for (int b = 0; b < t; b += 64)
    if (__ballot(b + lane < t && s[min(b + lane, T - 1)] == id)) return;  // (all waves of the workgroup)
  float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  for (int b = 64 * wave; b < T; b += 256) {
    unsigned long long m = __ballot(b + lane >= t && b + lane < T && s[min(b + lane, T - 1)] == id);
    while (m) {
      uint4 row[16];
      int n = 0;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        row[i] = make_uint4(0, 0, 0, 0);
        if (m) {
          row[i] = *reinterpret_cast<const uint4*>(a.dy + (long)(b + __builtin_ctzll(m)) * a.dy_ld + cl);
          m &= m - 1;
          ++n;
        }
      }
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        if (8 * h >= n) break;
        float w[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 8 * h; i < 8 * h + 8; ++i) {
          if (i >= n) break;
          const unsigned u[4] = {row[i].x, row[i].y, row[i].z, row[i].w};
#pragma unroll
          for (int j = 0; j < 4; ++j) w[2 * j] += bf2f(u[j] & 0xffff), w[2 * j + 1] += bf2f(u[j] >> 16);
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] += w[j];
      }
    }
  }
  if (wave > 0) {
#pragma unroll
    for (int j = 0; j < 8; ++j) part[wave - 1][lane][j] = v[j];
  }
  __syncthreads();
  if (wave > 0 || c >= a.H) return;
#pragma unroll
  for (int k = 0; k < 3; ++k)
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] += part[k][lane][j];
  put_row<G>(a, id, c, v);
}
}  // namespace

// g [V, H] (+)= the rows of dy [T, H] by their ids; without add, g's other rows are left as they are (the caller zeroes them)
void embed_grad_(const at::Tensor& ids, const at::Tensor& dy, at::Tensor g, bool add) {
  LLMCTL_CHECK(dy.is_cuda() && dy.dim() == 2 && dy.scalar_type() == at::kBFloat16 && dy.stride(1) == 1 && dy.stride(0) % 8 == 0 &&
                   (reinterpret_cast<uintptr_t>(dy.data_ptr()) & 15) == 0,
               "embed_grad: bf16 rows of 16 bytes' alignment");
  const long T = dy.size(0), H = dy.size(1);
  LLMCTL_CHECK(ids.is_cuda() && ids.dim() == 1 && ids.is_contiguous() && ids.scalar_type() == at::kLong && ids.numel() == T, "embed_grad: int64 ids [T]");
  LLMCTL_CHECK(g.is_cuda() && g.dim() == 2 && g.is_contiguous() && g.size(1) == H && (g.scalar_type() == at::kBFloat16 || g.scalar_type() == at::kFloat) &&
                   (reinterpret_cast<uintptr_t>(g.data_ptr()) & 15) == 0 && g.size(0) < (1L << 31),
               "embed_grad: a contiguous bf16 or fp32 gradient [V, H]");
  LLMCTL_CHECK(H % 8 == 0 && T <= 65536, "embed_grad: H in 8s, at most 65536 tokens");
  if (T == 0 || H == 0) return;
  const c10::DeviceGuard guard(dy.device());
  if (T <= FEW_IDS) {
    const EmbedGradArgs a{ids.data_ptr<int64_t>(), bf_ptr(dy), g.data_ptr(), nullptr, nullptr, nullptr, nullptr, (long)dy.stride(0), (long)g.size(0), (int)T, (int)H,
                          add};
    const dim3 few((unsigned)T, (unsigned)((H / 8 + 63) / 64));
    if (g.scalar_type() == at::kFloat) hipLaunchKernelGGL(embed_few_kernel<float>, few, dim3(256), 0, stream(), a);
    else hipLaunchKernelGGL(embed_few_kernel<unsigned short>, few, dim3(256), 0, stream(), a);
    return;
  }
  const int chunks = (int)((T + RUN - 1) / RUN);
  auto order = at::empty({3, T}, ids.options().dtype(at::kInt));
  auto part = at::empty({chunks, 2, H}, dy.options().dtype(at::kFloat));
  int* o = order.data_ptr<int>();
  EmbedGradArgs a{ids.data_ptr<int64_t>(), bf_ptr(dy), g.data_ptr(), o, o + T, o + 2 * T, part.data_ptr<float>(), (long)dy.stride(0), (long)g.size(0),
                  (int)T, (int)H, add};
  auto s = stream();
  const dim3 grid((unsigned)((chunks + 3) / 4), (unsigned)((H / 8 + 63) / 64));
  hipLaunchKernelGGL(embed_order_kernel, dim3((unsigned)((T + 2 * ORDER_WAVES - 1) / (2 * ORDER_WAVES))), dim3(64 * ORDER_WAVES), 0, s, a);
  if (g.scalar_type() == at::kFloat) {
    hipLaunchKernelGGL(embed_rows_grad_kernel<float>, grid, dim3(256), 0, s, a);
    hipLaunchKernelGGL(embed_edges_kernel<float>, grid, dim3(256), 0, s, a);
  } else {
    hipLaunchKernelGGL(embed_rows_grad_kernel<unsigned short>, grid, dim3(256), 0, s, a);
    hipLaunchKernelGGL(embed_edges_kernel<unsigned short>, grid, dim3(256), 0, s, a);
  }
}

TORCH_LIBRARY_IMPL(llmctl, CUDA, m) { m.impl("embed_grad_", &embed_grad_); }

}  // namespace llmctl
