// The LoRA down-projection of a row that a work-group already holds: t[row, col0 .. col0 + n) = bf16(x[row] . A^T) by 256 threads, of
// which thread i owns the 8-element chunks i, i + 256, ... of the bf16 row x in registers, as the norm and the attention combine leave it.
//
// A decode batch's down-projection as a launch of its own is a launch gap, a round trip for its operands and a reduction: 3.9-5 us, whatever
// its size.  Behind the kernel that produces x it costs the product alone: the row's work-groups (one per group of `nc` adapter columns)
// each form the row, redundantly, from operands that the L2 holds, and ask for their first columns of A before they wait for them.
// What bounds it is the bytes of a work-group ((partial planes + nc * 2) * K at some 110 GB/s per compute unit): row_adapter_cols takes groups
// that give every compute unit one work-group.  Measured: norm_rope.hip (tnx_norm_lora) and attention.hip (tnx_gqa_attn_lora).
#pragma once
#include "common.h"

namespace {

struct RowAdapterArgs {
  const uint16_t* a_t;   // bf16 [R, K]
  int R, nc;             // adapter columns, and how many of them a work-group takes
  uint16_t* t;
  int64_t t_ld;
  int groups, c_shift;   // ceil(R / nc); log2 of the column sets (row_adapter_place)
};
// Which row and which group of columns a work-group takes.  Ids go round-robin to the eight XCDs, and the grid is a multiple of eight wide: XCD x has
// column set x % c and row set x / c (c column sets, 8 / c row sets), so that its L2 fetches a part of the rows and a part of A and no
// more.  (Shifts: with two divisions in front of the first load the gain was a third smaller.)  false: none.
__device__ __forceinline__ bool row_adapter_place(const RowAdapterArgs& g, int64_t M, int& group, int64_t& row) {
  const int x = blockIdx.x;
  row = ((x & 7) >> g.c_shift) + ((int)blockIdx.y << (3 - g.c_shift));
  group = (x & ((1 << g.c_shift) - 1)) + ((x >> 3) << g.c_shift);
  return row < M && group < g.groups;
}
template <int MAXC, int NB>
struct RowAdapter {   // NB: adapter columns of a work-group at most, all asked for at once (NB * MAXC loads of 16 bytes per thread)
  u32x4 a[NB][MAXC];
  int ncols;
  // (columns past the last one repeat it, chunks past the row's end repeat its last one: their products are dropped)
  __device__ __forceinline__ void load(const RowAdapterArgs& g, int group, int64_t K) {
    const int nchunks = (int)(K / 8);
    const uint16_t* base = g.a_t + (int64_t)group * g.nc * K;
    ncols = min(g.nc, g.R - group * g.nc);
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int c = 0; c < MAXC; ++c)
        a[i][c] = *reinterpret_cast<const u32x4*>(base + (int64_t)min(i, ncols - 1) * K + (int64_t)min(c * 256 + (int)threadIdx.x, nchunks - 1) * 8);
  }
  // x: the thread's chunks of the row (zeros past its end); red: 4 * NB floats of LDS
  __device__ __forceinline__ void finish(const RowAdapterArgs& g, int group, int64_t row, const u32x4 (&x)[MAXC], float* red) {
    typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int b = 0; b < NB; b += 8) {
      float v[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        v[i] = 0.f;
#pragma unroll
        for (int c = 0; c < MAXC; ++c)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const uint32_t xq = x[c][q], aq = a[b + i][c][q];   // (a bit cast applied to the vector element itself reads element 0)
            v[i] = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf2, xq), __builtin_bit_cast(bf2, aq), v[i], false);
          }
      }
      const float s = wave_sum8(v, lane);
      if ((lane & 7) == 0) red[wave * NB + b + (lane >> 3)] = s;
    }
    __syncthreads();
    const int i = threadIdx.x;
    if (i < ncols) {
      float s = 0.f;
#pragma unroll
      for (int w = 0; w < 4; ++w) s += red[w * NB + i];
      g.t[row * g.t_ld + (int64_t)group * g.nc + i] = f2bf(s);
    }
  }
};

// The sets for operands of `row_bytes` per row, into g: those with which an XCD fetches least, as long as its 32 compute units have one
// work-group each; and the grid.  (Every XCD with a part of the columns of all rows, as ids fall in a grid of groups x rows, Llama-8B layers of 16 rows
// fetched 2.2 MB per norm and XCD instead of 1.3: the rollout of 16 rows 67.3 ms -> 65.4,
// of Gemma3-1B, 64 rows, 90.2 -> 89.6, of Qwen3-MoE layers 27.4 -> 27.0; column sets alone 68.3, 96.4 and 27.8.)
inline dim3 row_adapter_grid(RowAdapterArgs& g, int64_t M, int64_t K, int64_t row_bytes) {
  g.groups = (int)cdiv(g.R, g.nc);
  g.c_shift = 3;
  int64_t least = -1;
  for (int sh = 3; sh >= 0; --sh) {
    const int64_t sets = 8 >> sh, bytes = M * row_bytes / sets + (int64_t)g.R * K * 2 * sets / 8;
    if (cdiv(M, sets) * cdiv(g.groups, 1 << sh) <= 32 && (least < 0 || bytes < least)) {
      g.c_shift = sh;
      least = bytes;
    }
  }
  return dim3((unsigned)(8 * cdiv(g.groups, 1 << g.c_shift)), (unsigned)cdiv(M, 8 >> g.c_shift));
}

// Columns per work-group: whole batches of eight, as few as leave at most one work-group per compute unit.
inline int row_adapter_cols(int64_t M, int R) {
  const int64_t groups = M >= 256 ? 1 : 256 / M;
  return (int)(cdiv(cdiv(R, groups), 8) * 8);
}

}  // namespace
