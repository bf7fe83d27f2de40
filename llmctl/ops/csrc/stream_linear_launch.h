// The launches of stream_linear.h's workgroups, for the files that own them.
#pragma once
#include "stream_linear.h"

namespace stream_linear {

template <int NT, int MT, int NW, int U>
__global__ __launch_bounds__(NW * 64) void kernel(Args g) {
  __shared__ acc_t red[NW][NT * MT][64];
  const auto &bx = blockIdx.x, &by = blockIdx.y;
#include "stream_linear_body.inc"
}

template <int NT, int MT, int NW, int U>
inline void go(Args g, hipStream_t st, int rows = 16 * NT) {
  g.rows = rows;
  const unsigned parts = g.part > 0 ? (unsigned)((g.K + g.part - 1) / g.part) : 1u;
  kernel<NT, MT, NW, U><<<dim3((unsigned)((g.N + rows - 1) / rows), parts), NW * 64, 0, st>>>(g);
}

inline void launch(const Args& g, hipStream_t st) {
  const Form f = form_of(g.M, g.N, g.K);
  if (f.mt == 2) {
    if (f.nt == 1) go<1, 2, 4, 8>(g, st, f.rows);
    else if (f.nt == 2) go<2, 2, 4, 4>(g, st, f.rows);
    else if (f.nt == 3) go<3, 2, 4, 4>(g, st, f.rows);
    else go<4, 2, 4, 4>(g, st, f.rows);
  } else if (f.nt == 1) {
    if (f.nw == 2) go<1, 1, 2, 8>(g, st, f.rows);
    else go<1, 1, 4, 8>(g, st, f.rows);
  } else if (f.nt == 2) {
    if (f.u == 4) go<2, 1, 4, 4>(g, st, f.rows);
    else go<2, 1, 4, 8>(g, st, f.rows);
  } else if (f.nt == 3) {
    go<3, 1, 4, 4>(g, st, f.rows);
  } else {
    go<4, 1, 4, 4>(g, st, f.rows);
  }
}

// K in ``parts`` ranges, each its own fp32 [M, N], for a reader that adds them: one round of 256 workgroups of at most 64 rows
inline void launch_parts(Args g, int parts, hipStream_t st) {
  g.part = ((g.K + parts - 1) / parts + 31) / 32 * 32;
  g.f32 = 1;
  const int n = (g.K + g.part - 1) / g.part;
  const int rows = ((g.N * n + 255) / 256 + 3) / 4 * 4;
  if (g.M > 16) {
    if (rows <= 16) go<1, 2, 4, 8>(g, st, rows);
    else if (rows <= 32) go<2, 2, 4, 4>(g, st, rows);
    else go<4, 2, 4, 4>(g, st, rows > 64 ? 64 : rows);
  } else if (rows <= 16) {
    go<1, 1, 4, 8>(g, st, rows);
  } else if (rows <= 32) {
    go<2, 1, 4, 8>(g, st, rows);
  } else {
    go<4, 1, 4, 4>(g, st, rows > 64 ? 64 : rows);
  }
}

}  // namespace stream_linear
