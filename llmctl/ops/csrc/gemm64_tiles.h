// 256-row MFMA tiles staged through LDS: half-tile images and their swizzles, LDS-DMA pieces, operand fragments, and the two-MFMA statements that the
// hand-scheduled loops are made of.  Shared by gemm64.hip (256 x 256 tiles) and gemm_tall.hip (256 x 128).
#pragma once
#include "attn_common.h"

namespace llmctl {
using namespace attn;
namespace {

using f32x4_t = __attribute__((ext_vector_type(4))) float;
using s2_t = __attribute__((ext_vector_type(2))) unsigned int;
using i32x4_t = __attribute__((ext_vector_type(4))) int;

constexpr int TM = 256, TN = 256, TK = 64;
constexpr int HALF = 16384;       // bytes per half-tile image
constexpr int BUF = 4 * HALF;     // one K-tile: A_lo, A_hi, B_h0, B_h1
constexpr int NTHR = 512;
enum : int { A_LO = 0, A_HI = 1, B_H0 = 2, B_H1 = 3 };

template <int V>
using K_ = std::integral_constant<int, V>;

__device__ __forceinline__ i32x4_t make_rsrc(const void* base) {
  const unsigned long a = (unsigned long)base;
  i32x4_t r;
  r[0] = __builtin_amdgcn_readfirstlane((int)(a & 0xffffffffu));
  r[1] = __builtin_amdgcn_readfirstlane((int)((a >> 32) & 0xffff));
  r[2] = -1;          // num_records: no clamping (offsets validated on the host)
  r[3] = 0x00020000;  // raw buffer, 32-bit data format
  return r;
}
// range-checked raw buffer: loads at byte offsets >= bytes return 0, stores there are dropped
__device__ __forceinline__ i32x4_t make_rsrc_n(const void* base, unsigned bytes) {
  i32x4_t r = make_rsrc(base);
  r[2] = (int)bytes;
  return r;
}
// one LDS-DMA piece: 64 lanes x 16 B -> LDS [lds_byte, +1024), lane-linear
__device__ __forceinline__ void bdma16(i32x4_t rsrc, unsigned voff, unsigned soff, unsigned lds_byte) {
  asm volatile("s_mov_b32 m0, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds" ::"v"(voff), "s"(rsrc),
               "s"(soff), "s"(lds_byte)
               : "memory");
}

__device__ __forceinline__ void bar() { __builtin_amdgcn_s_barrier(); }
template <int N>
__device__ __forceinline__ void wait_vm() {
  if constexpr (N == 0) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  else if constexpr (N == 4) asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
  else if constexpr (N == 6) asm volatile("s_waitcnt vmcnt(6)" ::: "memory");
  else if constexpr (N == 8) asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
  else if constexpr (N == 40) asm volatile("s_waitcnt vmcnt(40)" ::: "memory");
  else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// ---- half-tile images -----------------------------------------------------------------------
// row image (K-contiguous operand): [128 image rows][64 k], 128-B rows, 16-B chunk c stored at
//   c ^ ((row >> 1) & 7): each ds_read_b128 lane group (16 lanes: rows r..r+15 at two chunks)
//   lands on 16 distinct 16-B bank slots.
// tr image (K-major operand): [64 k][128 image cols], 256-B rows, 32-B segment s stored at
//   s ^ h(k), h(k) = (k & 3) | ((k >> 3) & 1) << 2: the 8 k-rows of a 32-lane
//   ds_read_b64_tr_b16 half hit 8 distinct segments (conflict-free).
__device__ __forceinline__ int swr(int row) { return (row >> 1) & 7; }
__device__ __forceinline__ int swt(int k) { return (k & 3) | (((k >> 3) & 1) << 2); }

// image row/col -> tile row/col of each half-tile kind (both image kinds have 128 positions)
template <int KIND>
__device__ __forceinline__ int tile_pos(int ip) {
  if constexpr (KIND == A_LO) return (ip >> 6) * 128 + (ip & 63);
  else if constexpr (KIND == A_HI) return (ip >> 6) * 128 + 64 + (ip & 63);
  else if constexpr (KIND == B_H0) return ip;
  else return 128 + ip;
}

// per-thread byte offset (relative to the operand's tile origin at k = 0) of DMA piece i
template <bool T, int KIND, int NT = NTHR>
__device__ __forceinline__ unsigned stage_voff(int i, int tid, long ld) {
  const int c = i * NT + tid;  // 16-B chunk index in the half-tile image
  if constexpr (!T) {
    const int ir = c >> 3, pc = c & 7;
    const int row = tile_pos<KIND>(ir);
    return (unsigned)(((long)row * ld + ((pc ^ swr(ir)) << 3)) * 2);
  } else {
    const int k = c >> 4, pc = c & 15;
    const int seg = (pc >> 1) ^ swt(k);
    const int col = tile_pos<KIND>(seg * 16 + (pc & 1) * 8);
    return (unsigned)(((long)k * ld + col) * 2);
  }
}

// MFMA operand fragment (16 positions x 32 k): lane l holds X(p0 + (l & 15), 32 ks + 8 (l >> 4) + j)
template <bool T>
__device__ __forceinline__ bf16x8_t frag(const unsigned char* img, int p0, int ks, int lane) {
  const int g = lane >> 4, i16 = lane & 15;
  if constexpr (!T) {
    const int ir = p0 + i16;
    const int c = ks * 4 + g;
    return *reinterpret_cast<const bf16x8_t*>(img + ir * 128 + ((c ^ swr(ir)) << 4));
  } else {
    const int q = i16 >> 2, p = i16 & 3;
    const int k = ks * 32 + 8 * g + q;
    const int seg = (p0 >> 4) ^ swt(k);
    const int off = k * 256 + seg * 32 + p * 8;
    s4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(img + off));
    s4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(img + off + 4 * 256));
    s8_t v = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    return __builtin_bit_cast(bf16x8_t, v);
  }
}

constexpr int NT4 = 256;
// two MFMAs (acc row i x n-tiles j, j+1, one K-slice) / the same with one LDS-DMA piece between
// them (M0 written ahead of the first MFMA, so the MFMA covers the M0 -> LDS-DMA wait state): the
// K-loop's statements, so each fragment read and each DMA piece gets an MFMA gap of its own.
// Accumulators are pinned to the accumulation registers ("+a"; hipcc's own MFMA selection moved
// them through VGPRs and spilled: 256 accumulators + 160 fragment registers exceed the 256
// VGPRs); the "memory" clobber pins the reads / DMA issues placed between two statements to their
// gap.  Hazards (guide §5.7 item 2): MFMA -> MFMA accumulate chains need no wait states; the
// epilogue's reads are fenced after the loop (g4w_fence).
__device__ __forceinline__ void g4w_pair(f32x4_t& c0, f32x4_t& c1, const bf16x8_t& a, const bf16x8_t& b0,
                                         const bf16x8_t& b1) {
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %3, %2, %0\n\t"
               "v_mfma_f32_16x16x32_bf16 %1, %4, %2, %1"
               : "+a"(c0), "+a"(c1)
               : "v"(a), "v"(b0), "v"(b1)
               : "memory");
}
// the same with C = 0 (an item's first K-slice): the accumulators are defined here, not carried
// from a zeroing through the item loop's back-edge (persistent kernel)
__device__ __forceinline__ void g4w_pair_z(f32x4_t& c0, f32x4_t& c1, const bf16x8_t& a, const bf16x8_t& b0,
                                           const bf16x8_t& b1) {
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %3, %2, 0\n\t"
               "v_mfma_f32_16x16x32_bf16 %1, %4, %2, 0"
               : "=a"(c0), "=a"(c1)
               : "v"(a), "v"(b0), "v"(b1)
               : "memory");
}
__device__ __forceinline__ void g4w_pair_dma(f32x4_t& c0, f32x4_t& c1, const bf16x8_t& a, const bf16x8_t& b0,
                                             const bf16x8_t& b1, unsigned voff, i32x4_t rsrc, unsigned soff,
                                             unsigned lds_byte) {
  asm volatile("s_mov_b32 m0, %8\n\t"
               "v_mfma_f32_16x16x32_bf16 %0, %3, %2, %0\n\t"
               "buffer_load_dwordx4 %5, %6, %7 offen lds\n\t"
               "v_mfma_f32_16x16x32_bf16 %1, %4, %2, %1"
               : "+a"(c0), "+a"(c1)
               : "v"(a), "v"(b0), "v"(b1), "v"(voff), "s"(rsrc), "s"(soff), "s"(lds_byte)
               : "memory");
}


}  // namespace
}  // namespace llmctl
