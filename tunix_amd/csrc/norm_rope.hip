// Embedding gather, RMSNorm (three dtype flows), per-head q/k norm + RoPE + KV-cache write.
// All of these move a few bytes per decode step compared with the weights and the cache; they
// are written for exact dtype-flow parity and few launches, not for peak bandwidth.
#include <string.h>

#include <type_traits>

#include "common.h"
#include "rope_math.h"
#include "row_adapter.h"

namespace {

// ---- block reductions --------------------------------------------------------------------
__device__ __forceinline__ float block_sum(float v, float* red) {
  v = wave_sum(v);
  const int wave = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
  if (nw == 1) return v;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[wave] = v;
  __syncthreads();
  float s = 0.f;
  for (int w = 0; w < nw; ++w) s += red[w];
  return s;
}

__global__ __launch_bounds__(256) void rmsnorm_kernel(const uint16_t* x, const uint16_t* res_pre,
                                                      uint16_t* h_out, const uint16_t* w,
                                                      const uint16_t* res_post, uint16_t* y,
                                                      int64_t D, float eps, int flavor) {
  __shared__ float red[4];
  extern __shared__ __align__(16) unsigned char smem_dyn[];
  float* hrow = reinterpret_cast<float*>(smem_dyn);  // [D]
  const int64_t row = blockIdx.x;
  const uint16_t* xr = x + row * D;
  float ss = 0.f;
  for (int64_t i = threadIdx.x; i < D; i += blockDim.x) {
    float h = bf2f(xr[i]);
    if (res_pre) h = rbf(h + bf2f(res_pre[row * D + i]));
    if (h_out) h_out[row * D + i] = f2bf(h);
    hrow[i] = h;
    ss += sq_term(h, flavor);
  }
  ss = block_sum(ss, red);
  const float ms = finish_ms(ss, (float)D, flavor);
  for (int64_t i = threadIdx.x; i < D; i += blockDim.x) {
    float v = norm_elem(hrow[i], bf2f(w[i]), ms, eps, flavor);
    if (res_post) v = rbf(v + bf2f(res_post[row * D + i]));
    y[row * D + i] = f2bf(v);
  }
}

// The same op for D % 8 == 0 (every model on the path): 16-byte loads and stores, the row stays
// in registers between the two passes (thread t owns the 8-element chunks t, t + 256, ...).
constexpr int kNormMaxChunks = 8;  // D <= 8 * 256 * 8 = 16384
__device__ __forceinline__ void unpack8(const u32x4& p, float (&f)[8]) {
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    f[2 * j] = bflo(p[j]);
    f[2 * j + 1] = bfhi(p[j]);
  }
}
// The input row, by IN: kNormInRow -- x[row]; kNormInPlanes -- bf16(sum of the split_k fp32 partial
// planes ws[z][row][:]) of a split-k linear, added in split order: the linear's own finishing
// pass folded into the norm; kNormInRoutes -- bf16(sum_j cw[row, j] * x[row * split_k + j]) over
// the split_k routed rows of a token, j ascending: the weighted combine of an MoE layer folded
// into the norm (same arithmetic as moe_combine_vec_kernel); kNormInTable -- the embedding of the row's token, x[id] * scale.
constexpr int kNormInRow = 0, kNormInPlanes = 1, kNormInRoutes = 2, kNormInTable = 3;
// sin / cos of angle = position / timescale[i] for the token in column *col_ptr of row b: the
// values rope_kernel computes for the Llama rotation, once per decode step instead of per layer.
struct RopeTable {
  const int32_t* positions;   // null: none asked for
  int64_t pos_ld, B;
  const float* timescale;
  int half;
  float *sin_out, *cos_out;
};
__device__ __forceinline__ void rope_table_row(const RopeTable& r, int64_t b, int col) {
  for (int i = threadIdx.x; i < r.half; i += blockDim.x) {
    const float ang = __fdiv_rn((float)r.positions[b * r.pos_ld + col], r.timescale[i]);
    r.sin_out[b * r.half + i] = sinf(ang);
    r.cos_out[b * r.half + i] = cosf(ang);
  }
}
struct EmbedSrc {
  const int32_t* ids;
  int64_t ids_ld;
  const int32_t* col_ptr;
  int64_t V;
  uint32_t T;
  float scale_bf;
  RopeTable rope;
  int64_t first_table_row;   // of the grid: its rows (rmsnorm_lora_kernel) or its work-groups from there on have a row of the rope table
};
struct NormRow {
  const uint16_t *x, *res_pre;
  uint16_t* h_out;
  const uint16_t *w, *res_post;
  uint16_t* y;
  int64_t D;
  float eps;
  const float* ws;
  int split_k;
  int64_t plane;
  const uint16_t* w2;
  uint16_t* y2;
  const uint16_t* cw;
  EmbedSrc e;
};
__device__ __forceinline__ int64_t embed_id(const EmbedSrc& e, int64_t row) {
  const uint32_t b = (uint32_t)row / e.T, t = (uint32_t)row - b * e.T;
  const int64_t id = e.ids[b * e.ids_ld + (e.col_ptr ? *e.col_ptr : 0) + t];
  return id < 0 || id >= e.V ? 0 : id;   // pad sentinels outside the vocabulary read row 0 (masked later)
}
// One row: writes it (WRITE) and leaves the thread's chunks of the last norm, packed, in `last` (zeros past the row's end).
// behind(): called once every load of the row has been asked for.
template <int MAXC, int FLAVOR, int IN, class F>
__device__ __forceinline__ void norm_row(const NormRow& n, int64_t row, bool write, float* red, u32x4 (&last)[MAXC], F behind) {
  const uint16_t *x = n.x, *res_pre = n.res_pre, *w = n.w, *res_post = n.res_post, *w2 = n.w2, *cw = n.cw;
  uint16_t *h_out = n.h_out, *y = n.y, *y2 = n.y2;
  const float* ws = n.ws;
  const int64_t D = n.D, plane = n.plane;
  const float eps = n.eps;
  const int split_k = n.split_k;
  constexpr bool PLANES = IN == kNormInPlanes, ROUTES = IN == kNormInRoutes, TABLE = IN == kNormInTable;
  const int nchunks = (int)(D / 8);
  float h[MAXC][8];
#pragma unroll
  for (int c = 0; c < MAXC; ++c) last[c] = u32x4{0, 0, 0, 0};
  float ss = 0.f;
  // The norm weights and the post-norm residual do not depend on the row: they are asked for ahead of its planes (a launch is a
  // few round trips to memory long, and one that starts behind the sums adds a whole one: 16 rows of 4096 from
  // eight planes 6.2 -> 5.7 us), or, for rows of more than 4096,
  // whose registers do not hold them that long, before the reduction.
  u32x4 wpre[MAXC], rpost[MAXC], w2pre[MAXC];
  auto fetch_weights = [&]() {
#pragma unroll
    for (int c = 0; c < MAXC; ++c) {
      const int64_t at = (int64_t)min(c * 256 + (int)threadIdx.x, nchunks - 1) * 8;
      wpre[c] = *reinterpret_cast<const u32x4*>(w + at);
      if (w2) w2pre[c] = *reinterpret_cast<const u32x4*>(w2 + at);
      if (res_post && res_post != h_out) rpost[c] = *reinterpret_cast<const u32x4*>(res_post + row * D + at);
    }
  };
  if constexpr (MAXC <= 2) fetch_weights();
  if constexpr (TABLE) x += embed_id(n.e, row) * D;
  // Chunks are taken two at a time with every load of the pair issued before the first sum (up
  // to eight planes per chunk at once, further planes in groups of eight): the kernel is a few
  // dependent memory round trips long, and each group of loads that waits for the previous sum
  // adds one.  The sum itself stays in split order.
  constexpr int CS = MAXC < 2 ? 1 : 2;
#pragma unroll
  for (int c0 = 0; c0 < MAXC; c0 += CS) {
    if (c0 * 256 >= nchunks) break;   // uniform
    f32x4 p0[CS][8], p1[CS][8];
    u32x4 xin[CS], rin[CS], yin[CS][8];
#pragma unroll
    for (int cc = 0; cc < CS; ++cc) {
      const int ch = (c0 + cc) * 256 + threadIdx.x;
      const int64_t o = row * D + (int64_t)min(ch, nchunks - 1) * 8;
      if (PLANES) {
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const int64_t zo = (int64_t)min(u, split_k - 1) * plane + o;
          p0[cc][u] = *reinterpret_cast<const f32x4*>(ws + zo);
          p1[cc][u] = *reinterpret_cast<const f32x4*>(ws + zo + 4);
        }
      } else if (ROUTES) {
#pragma unroll
        for (int u = 0; u < 8; ++u)
          yin[cc][u] = *reinterpret_cast<const u32x4*>(
              x + (row * split_k + min(u, split_k - 1)) * D + (int64_t)min(ch, nchunks - 1) * 8);
      } else {
        xin[cc] = *reinterpret_cast<const u32x4*>(x + (TABLE ? o - row * D : o));
      }
      if (res_pre) rin[cc] = *reinterpret_cast<const u32x4*>(res_pre + o);
    }
    if (c0 + CS >= MAXC || (c0 + CS) * 256 >= nchunks) behind();
#pragma unroll
    for (int cc = 0; cc < CS; ++cc) {
      const int c = c0 + cc;
      const int ch = c * 256 + threadIdx.x;
      if (ch < nchunks) {
        const int64_t o = row * D + (int64_t)ch * 8;
        if (PLANES) {
#pragma unroll
          for (int j = 0; j < 8; ++j) h[c][j] = 0.f;
#pragma unroll
          for (int u = 0; u < 8; ++u)
            if (u < split_k) {
#pragma unroll
              for (int j = 0; j < 4; ++j) {
                h[c][j] += p0[cc][u][j];
                h[c][4 + j] += p1[cc][u][j];
              }
            }
          for (int z0 = 8; z0 < split_k; z0 += 8) {   // more than eight planes: the rest in groups
            f32x4 q0[8], q1[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
              const int64_t zo = (int64_t)min(z0 + u, split_k - 1) * plane + o;
              q0[u] = *reinterpret_cast<const f32x4*>(ws + zo);
              q1[u] = *reinterpret_cast<const f32x4*>(ws + zo + 4);
            }
#pragma unroll
            for (int u = 0; u < 8; ++u)
              if (z0 + u < split_k) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                  h[c][j] += q0[u][j];
                  h[c][4 + j] += q1[u][j];
                }
              }
          }
#pragma unroll
          for (int j = 0; j < 8; ++j) h[c][j] = rbf(h[c][j]);
        } else if (ROUTES) {
#pragma unroll
          for (int j = 0; j < 8; ++j) h[c][j] = 0.f;
#pragma unroll
          for (int u = 0; u < 8; ++u)
            if (u < split_k) {
              const float wt = bf2f(cw[row * split_k + u]);
#pragma unroll
              for (int q = 0; q < 4; ++q) {
                h[c][2 * q] += wt * bflo(yin[cc][u][q]);
                h[c][2 * q + 1] += wt * bfhi(yin[cc][u][q]);
              }
            }
          for (int z0 = 8; z0 < split_k; z0 += 8) {   // more than eight routes per token: the rest in groups
            u32x4 v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u)
              v[u] = *reinterpret_cast<const u32x4*>(x + (row * split_k + min(z0 + u, split_k - 1)) * D + (int64_t)ch * 8);
#pragma unroll
            for (int u = 0; u < 8; ++u)
              if (z0 + u < split_k) {
                const float wt = bf2f(cw[row * split_k + z0 + u]);
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                  h[c][2 * q] += wt * bflo(v[u][q]);
                  h[c][2 * q + 1] += wt * bfhi(v[u][q]);
                }
              }
          }
#pragma unroll
          for (int j = 0; j < 8; ++j) h[c][j] = rbf(h[c][j]);
        } else {
          unpack8(xin[cc], h[c]);
          if (TABLE && n.e.scale_bf != 1.0f) {
#pragma unroll
            for (int j = 0; j < 8; ++j) h[c][j] = rbf(h[c][j] * n.e.scale_bf);
          }
        }
        if (res_pre) {
          float r[8];
          unpack8(rin[cc], r);
#pragma unroll
          for (int j = 0; j < 8; ++j) h[c][j] = rbf(h[c][j] + r[j]);
        }
        if (h_out && write) {
          u32x4 q;
#pragma unroll
          for (int j = 0; j < 4; ++j) q[j] = pack2bf(h[c][2 * j], h[c][2 * j + 1]);
          *reinterpret_cast<u32x4*>(h_out + o) = q;
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) ss += sq_term(h[c][j], FLAVOR);
      }
    }
  }
  if constexpr (MAXC > 2) fetch_weights();
  ss = block_sum(ss, red);
  const float ms = finish_ms(ss, (float)D, FLAVOR);
  float ss2 = 0.f;
#pragma unroll
  for (int c = 0; c < MAXC; ++c) {
    const int ch = c * 256 + threadIdx.x;
    if (ch < nchunks) {
      const int64_t o = row * D + (int64_t)ch * 8;
      float wv[8], v[8];
      unpack8(wpre[c], wv);
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = norm_elem(h[c][j], wv[j], ms, eps, FLAVOR);
      if (res_post) {
        float r[8];
        // (a residual that this launch itself rewrote as h_out is read back here, after the write)
        unpack8(res_post != h_out ? rpost[c] : *reinterpret_cast<const u32x4*>(res_post + o), r);
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = rbf(v[j] + r[j]);
      }
      u32x4 q;
#pragma unroll
      for (int j = 0; j < 4; ++j) q[j] = pack2bf(v[2 * j], v[2 * j + 1]);
      if (write) *reinterpret_cast<u32x4*>(y + o) = q;
      last[c] = q;
      if (w2) {   // the row just written is the input of a second norm: keep it, as rounded
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          h[c][j] = rbf(v[j]);
          ss2 += sq_term(h[c][j], FLAVOR);
        }
      }
    }
  }
  if (!w2) return;
  // y2 = norm(y) with its own weight, the row still in registers (same thread -> chunk map and
  // reduction order as a launch of its own would use: the results are identical)
  ss2 = block_sum(ss2, red);
  const float ms2 = finish_ms(ss2, (float)D, FLAVOR);
#pragma unroll
  for (int c = 0; c < MAXC; ++c) {
    const int ch = c * 256 + threadIdx.x;
    if (ch < nchunks) {
      float wv[8];
      unpack8(w2pre[c], wv);
      u32x4 q;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        q[j] = pack2bf(norm_elem(h[c][2 * j], wv[2 * j], ms2, eps, FLAVOR),
                       norm_elem(h[c][2 * j + 1], wv[2 * j + 1], ms2, eps, FLAVOR));
      if (write) *reinterpret_cast<u32x4*>(y2 + row * D + (int64_t)ch * 8) = q;
      last[c] = q;
    }
  }
}
template <int MAXC, int FLAVOR, int IN>
__global__ __launch_bounds__(256) void rmsnorm_vec_kernel(const NormRow n) {
  __shared__ float red[4];
  u32x4 last[MAXC];
  if constexpr (IN == kNormInTable) {
    if ((int64_t)blockIdx.x >= n.e.first_table_row) {
      rope_table_row(n.e.rope, blockIdx.x - n.e.first_table_row, n.e.col_ptr ? *n.e.col_ptr : 0);
      return;
    }
  }
  norm_row<MAXC, FLAVOR, IN>(n, blockIdx.x, true, red, last, [] {});
}
// The same with the LoRA down-projection of the row behind it (row_adapter.h); the first group of adapter columns writes the row.
template <int MAXC, int FLAVOR, int IN, int NB>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 2))) void rmsnorm_lora_kernel(const NormRow n, int64_t M, const RowAdapterArgs g) {
  __shared__ float red[4], sums[4 * NB];
  u32x4 last[MAXC];
  RowAdapter<MAXC, NB> ad;
  int group;
  int64_t row;
  if constexpr (IN == kNormInTable) {
    if ((int64_t)blockIdx.y >= n.e.first_table_row) {
      const int64_t b = (blockIdx.y - n.e.first_table_row) * gridDim.x + blockIdx.x;
      if (b < n.e.rope.B) rope_table_row(n.e.rope, b, n.e.col_ptr ? *n.e.col_ptr : 0);
      return;
    }
  }
  if (!row_adapter_place(g, M, group, row)) return;
  norm_row<MAXC, FLAVOR, IN>(n, row, group == 0, red, last, [&] { ad.load(g, group, n.D); });
  ad.finish(g, group, row, last, sums);
}

// The kernel is unrolled over its chunks (256 threads x 8 elements each): instantiated for 1, 2, 4
// and 8 chunks per thread so that the common widths (D <= 4096) run the small instances -- the
// code a wave walks through once is fetched cold at every launch.
template <class F>
void with_flavor(int flavor, F f) {
  if (flavor == TNX_NORM_LLAMA) f(std::integral_constant<int, TNX_NORM_LLAMA>{});
  else if (flavor == TNX_NORM_QWEN3) f(std::integral_constant<int, TNX_NORM_QWEN3>{});
  else f(std::integral_constant<int, TNX_NORM_GEMMA3>{});
}
template <class F>
void with_input(int in, F f) {
  if (in == kNormInPlanes) f(std::integral_constant<int, kNormInPlanes>{});
  else if (in == kNormInRoutes) f(std::integral_constant<int, kNormInRoutes>{});
  else if (in == kNormInTable) f(std::integral_constant<int, kNormInTable>{});
  else f(std::integral_constant<int, kNormInRow>{});
}
void launch_rmsnorm_vec(hipStream_t st, int64_t rows, int flavor, int in, const NormRow& given) {
  NormRow n = given;
  n.e.first_table_row = rows;
  const int64_t M = rows + (n.e.rope.positions ? n.e.rope.B : 0);
  with_flavor(flavor, [&](auto f) {
    with_input(in, [&](auto i) {
      constexpr int F = decltype(f)::value, IN = decltype(i)::value;
      if (n.D <= 8 * 256) hipLaunchKernelGGL((rmsnorm_vec_kernel<1, F, IN>), dim3((unsigned)M), dim3(256), 0, st, n);
      else if (n.D <= 8 * 256 * 2) hipLaunchKernelGGL((rmsnorm_vec_kernel<2, F, IN>), dim3((unsigned)M), dim3(256), 0, st, n);
      else if (n.D <= 8 * 256 * 4) hipLaunchKernelGGL((rmsnorm_vec_kernel<4, F, IN>), dim3((unsigned)M), dim3(256), 0, st, n);
      else hipLaunchKernelGGL((rmsnorm_vec_kernel<kNormMaxChunks, F, IN>), dim3((unsigned)M), dim3(256), 0, st, n);
    });
  });
}
// Whether the rows' work-groups take the adapter columns too: as long as there is at most one of them per compute unit.
// us, two launches | one, eight planes: D 4096, 192 columns 1 row 8.6 | 5.8, 8 rows 9.2 | 6.5, 16 rows 9.6 | 8.9, 24 rows (24 columns each) 10.2 | 14;
// D 2048, 128 columns 16 rows 7.3 | 4.8, 64 rows 7.9 | 7.4, 128 rows 9.3 | 11.5; two norms of 1152, 64 columns 64 rows 7.5 | 5.9, 128 rows 7.9 | 6.6.
bool norm_lora_one_launch(int64_t M, int64_t D, int R) {
  if (M > 256 || D > 8 * 256 * 2) return false;
  return D > 8 * 256 ? M <= 16 && row_adapter_cols(M, R) <= 16 : row_adapter_cols(M, R) <= 32;
}
void launch_rmsnorm_lora(hipStream_t st, int64_t M, int flavor, int in, const NormRow& given, RowAdapterArgs g) {
  NormRow n = given;
  dim3 grid = row_adapter_grid(g, M, n.D, n.D * (in == kNormInPlanes ? 4 * n.split_k : in == kNormInRoutes ? 2 * n.split_k : 2));
  n.e.first_table_row = grid.y;
  if (n.e.rope.positions) grid.y += (unsigned)cdiv(n.e.rope.B, grid.x);
  with_flavor(flavor, [&](auto f) {
    with_input(in, [&](auto i) {
      constexpr int F = decltype(f)::value, IN = decltype(i)::value;
      const auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, dim3(256), 0, st, n, M, g); };
      if (n.D > 8 * 256) g.nc <= 8 ? launch(rmsnorm_lora_kernel<2, F, IN, 8>) : launch(rmsnorm_lora_kernel<2, F, IN, 16>);
      else if (g.nc <= 16) g.nc <= 8 ? launch(rmsnorm_lora_kernel<1, F, IN, 8>) : launch(rmsnorm_lora_kernel<1, F, IN, 16>);
      else g.nc <= 24 ? launch(rmsnorm_lora_kernel<1, F, IN, 24>) : launch(rmsnorm_lora_kernel<1, F, IN, 32>);
    });
  });
}

__global__ void embed_kernel(const uint16_t* table, int64_t V, int64_t D, const int32_t* ids,
                             int64_t ids_ld, const int32_t* col_ptr, int64_t T, float scale_bf,
                             uint16_t* out, const PackedRows rows) {
  const int64_t b = blockIdx.x / T, t = blockIdx.x % T;
  if (rows.base && t < rows.starts[b]) return;
  const int64_t row = rows.base ? rows.base[b] + t : blockIdx.x;
  const int col = col_ptr ? *col_ptr : 0;
  int64_t id = ids[b * ids_ld + col + t];
  if (id < 0 || id >= V) id = 0;  // pad sentinels outside the vocabulary read row 0 (masked later)
  const uint16_t* src = table + id * D;
  if (D % 8 == 0) {   // 16 bytes per thread and turn
    for (int64_t i = (int64_t)threadIdx.x * 8; i < D; i += (int64_t)blockDim.x * 8) {
      u32x4 v = *reinterpret_cast<const u32x4*>(src + i);
      if (scale_bf != 1.0f) {
#pragma unroll
        for (int q = 0; q < 4; ++q) v[q] = pack2bf(bflo(v[q]) * scale_bf, bfhi(v[q]) * scale_bf);
      }
      *reinterpret_cast<u32x4*>(out + row * D + i) = v;
    }
    return;
  }
  for (int64_t i = threadIdx.x; i < D; i += blockDim.x) {
    uint16_t v = src[i];
    if (scale_bf != 1.0f) v = f2bf(bf2f(v) * scale_bf);
    out[row * D + i] = v;
  }
}

// grid (B*T, Hq + 2*Hkv); dh/2 threads, rounded up to whole waves (wave_sum): thread i < dh/2 owns elements i and i + dh/2
// of one head; the other threads only take part in the reductions.
// A decode step's launch is a chain of round trips to memory, so everything that needs no other load is asked for at
// once, ahead of the first wait, and the angle is computed while the planes arrive.  64 rows of 4 + 2 heads of 256 from eight planes, us
// per launch 4.5 -> 3.7 alone; 32 + 8 heads of 128 from six 5.2 -> 4.2.
template <bool PLANES>
__global__ void rope_kernel(const RopeArgs a) {
  __shared__ float red[4];
  const uint32_t b = blockIdx.x / (uint32_t)a.T, t = blockIdx.x - b * (uint32_t)a.T;
  if (a.rows.base && (int)t < a.rows.starts[b]) return;
  const uint32_t row = a.rows.base ? (uint32_t)a.rows.base[b] + t : blockIdx.x;
  const int head = blockIdx.y;
  const int half = a.dh / 2, i = threadIdx.x, il = min(i, half - 1);
  const bool live = i < half, is_v = head >= a.Hq + a.Hkv, is_q = head < a.Hq, normed = a.qk_norm >= 0 && !is_v;
  const int col = *a.col_ptr;
  const int ld = (a.Hq + 2 * a.Hkv) * a.dh;
  const int64_t src_off = (int64_t)row * ld + (int64_t)head * a.dh + il;
  // elements i and i + half of this head: from the finished linear output, or as the linear's own finishing
  // pass would produce them, bf16(sum of the split-k planes in split order)
  float x1, x2;
  float p1[8], p2[8];
  uint16_t h1 = 0, h2 = 0;
  const int64_t plane = (a.rows.base ? a.rows.rows : a.B * a.T) * (int64_t)ld;
  if constexpr (PLANES) {
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const float* p = a.ws + (int64_t)min(u, a.split_k - 1) * plane + src_off;
      p1[u] = p[0];
      p2[u] = p[half];
    }
  } else {
    h1 = a.qkv[src_off];
    h2 = a.qkv[src_off + half];
  }
  const uint16_t* wn = is_q ? a.q_norm_w : a.k_norm_w;
  const float ts = a.timescale[il];
  uint16_t w1 = 0, w2 = 0;
  if (normed) {
    w1 = wn[il];
    w2 = wn[il + half];
  }
  const float pos = (float)a.positions[b * a.pos_ld + col + t];
  float sn = 0.f, cs = 0.f;
  if (!is_v) rope_angle(a, pos, ts, sn, cs);
  if constexpr (PLANES) {
    x1 = 0.f;
    x2 = 0.f;
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (u < a.split_k) {
        x1 += p1[u];
        x2 += p2[u];
      }
    for (int z0 = 8; z0 < a.split_k; z0 += 8) {   // eight planes' loads in flight; sum in split order
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const float* p = a.ws + (int64_t)min(z0 + u, a.split_k - 1) * plane + src_off;
        p1[u] = p[0];
        p2[u] = p[half];
      }
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (z0 + u < a.split_k) {
          x1 += p1[u];
          x2 += p2[u];
        }
    }
    x1 = rbf(x1);
    x2 = rbf(x2);
  } else {
    x1 = bf2f(h1);
    x2 = bf2f(h2);
  }
  const int64_t slot = ring_slot((int64_t)col + t, a.S);
  uint16_t* dst;
  if (is_v) {   // V: plain copy into the cache slot
    dst = a.vcache + ((((int64_t)b * a.Hkv + (head - a.Hq - a.Hkv)) * a.S) + slot) * a.dh;
  } else {
    if (normed) {
      const float ss = block_sum(live ? sq_term(x1, a.qk_norm) + sq_term(x2, a.qk_norm) : 0.f, red);
      const float ms = finish_ms(ss, (float)a.dh, a.qk_norm);
      x1 = norm_elem(x1, bf2f(w1), ms, a.norm_eps, a.qk_norm);
      x2 = norm_elem(x2, bf2f(w2), ms, a.norm_eps, a.qk_norm);
    }
    float o1, o2;
    rotate_pair(a, is_q, x1, x2, sn, cs, o1, o2);
    x1 = o1;
    x2 = o2;
    dst = is_q ? a.q_out + ((int64_t)row * a.Hq + head) * a.dh
               : a.kcache + ((((int64_t)b * a.Hkv + (head - a.Hq)) * a.S) + slot) * a.dh;
  }
  if (!live) return;
  dst[i] = f2bf(x1);
  dst[i + half] = f2bf(x2);
}

// Many rows (a prefill or whole-sequence pass): one work-group per token row, 16-byte accesses; the sines and cosines of the
// row's pairs are computed once, a pair per thread, and shared through LDS.  Thread (ch, h0) owns the eight pairs i = 8 ch .. + 7 of
// heads h0, h0 + hstep, ...; a head's sum of squares (NORM) is formed over its dh / 16 neighbouring lanes.  Bound by
// memory: qkv in, q and the cache slots out.  us: 7 x 1023 rows of 32 + 2 x 4 normed heads of 128 136 -> 49 (146 MB; before in rope_kernel, a
// work-group per head), 2 x 6144 rows of 32 + 2 x 8 heads of 128 83 -> 49 (302 MB: 6.2 TB/s; before, sines by every thread for itself).
template <bool NORM>
__global__ __launch_bounds__(256) void rope_rows_kernel(const RopeArgs a) {
  __shared__ float trig[2][256];   // [sine, cosine][pair]: head_dim at most 512
  const uint32_t b = blockIdx.x / (uint32_t)a.T, t = blockIdx.x - b * (uint32_t)a.T;
  if (a.rows.base && (int)t < a.rows.starts[b]) return;   // (uniform)
  const uint32_t row = a.rows.base ? (uint32_t)a.rows.base[b] + t : blockIdx.x;
  const int half = a.dh / 2, CH = half / 8, heads = a.Hq + 2 * a.Hkv;
  const int ch = threadIdx.x % CH, h0 = threadIdx.x / CH, hstep = 256 / CH;
  const int col = *a.col_ptr;
  const int ld = heads * a.dh;
  const int64_t slot = ring_slot((int64_t)col + t, a.S);
  const int i0 = ch * 8;
  u32x4 wq[2], wk[2];
  if constexpr (NORM) {
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      wq[p] = *reinterpret_cast<const u32x4*>(a.q_norm_w + i0 + p * half);
      wk[p] = *reinterpret_cast<const u32x4*>(a.k_norm_w + i0 + p * half);
    }
  }
  if ((int)threadIdx.x < half) {
    const float pos = (float)a.positions[b * a.pos_ld + col + t];
    float sn, cs;
    rope_angle(a, pos, a.timescale[threadIdx.x], sn, cs);
    trig[0][threadIdx.x] = sn;
    trig[1][threadIdx.x] = cs;
  }
  __syncthreads();
  f32x4 sn[2], cs[2];
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    sn[p] = *reinterpret_cast<const f32x4*>(&trig[0][i0 + 4 * p]);
    cs[p] = *reinterpret_cast<const f32x4*>(&trig[1][i0 + 4 * p]);
  }
  for (int head = h0; head < heads; head += hstep) {   // (the lanes of a head stay together: heads differ by whole groups)
    const uint16_t* src = a.qkv + (int64_t)row * ld + (int64_t)head * a.dh + i0;
    const u32x4 v1 = *reinterpret_cast<const u32x4*>(src), v2 = *reinterpret_cast<const u32x4*>(src + half);
    uint16_t* dst;
    if (head >= a.Hq + a.Hkv) {   // V: plain copy into the cache slot
      dst = a.vcache + ((((int64_t)b * a.Hkv + (head - a.Hq - a.Hkv)) * a.S) + slot) * a.dh + i0;
      *reinterpret_cast<u32x4*>(dst) = v1;
      *reinterpret_cast<u32x4*>(dst + half) = v2;
      continue;
    }
    const bool is_q = head < a.Hq;
    float x1[8], x2[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      x1[e] = (e & 1) ? bfhi(v1[e >> 1]) : bflo(v1[e >> 1]);
      x2[e] = (e & 1) ? bfhi(v2[e >> 1]) : bflo(v2[e >> 1]);
    }
    if constexpr (NORM) {
      float ss = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) ss += sq_term(x1[e], a.qk_norm) + sq_term(x2[e], a.qk_norm);
#pragma unroll
      for (int o = 32; o > 0; o >>= 1)
        if (o <= CH / 2) ss += lane_xor(ss, o);
      const float ms = finish_ms(ss, (float)a.dh, a.qk_norm);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const uint32_t w1 = is_q ? wq[0][e >> 1] : wk[0][e >> 1], w2 = is_q ? wq[1][e >> 1] : wk[1][e >> 1];
        x1[e] = norm_elem(x1[e], (e & 1) ? bfhi(w1) : bflo(w1), ms, a.norm_eps, a.qk_norm);
        x2[e] = norm_elem(x2[e], (e & 1) ? bfhi(w2) : bflo(w2), ms, a.norm_eps, a.qk_norm);
      }
    }
    u32x4 o1v, o2v;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float o1[2], o2[2];
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const int e = 2 * r + k;
        rotate_pair(a, is_q, x1[e], x2[e], sn[e >> 2][e & 3], cs[e >> 2][e & 3], o1[k], o2[k]);
      }
      o1v[r] = pack2bf(o1[0], o1[1]);
      o2v[r] = pack2bf(o2[0], o2[1]);
    }
    if (is_q) dst = a.q_out + ((int64_t)row * a.Hq + head) * a.dh + i0;
    else dst = a.kcache + ((((int64_t)b * a.Hkv + (head - a.Hq)) * a.S) + slot) * a.dh + i0;
    *reinterpret_cast<u32x4*>(dst) = o1v;
    *reinterpret_cast<u32x4*>(dst + half) = o2v;
  }
}

__global__ void rope_table_kernel(const RopeTable r, const int32_t* col_ptr) { rope_table_row(r, blockIdx.x, *col_ptr); }

}  // namespace

extern "C" int tnx_embed(void* stream, const uint16_t* table, int64_t V, int64_t D,
                         const int32_t* ids, int64_t ids_ld, const int32_t* col_ptr, int64_t B,
                         int64_t T, float scale, uint16_t* out) {
  TNX_REQUIRE(table && ids && out, "embed: null pointer");
  TNX_REQUIRE(V > 0 && D > 0 && B > 0 && T > 0, "embed: bad shape");
  hipLaunchKernelGGL(embed_kernel, dim3((unsigned)(B * T)), dim3(256), 0, as_stream(stream), table,
                     V, D, ids, ids_ld, col_ptr, T, host_round_bf16(scale), out, kAllRows);
  TNX_CHECK_LAUNCH("embed");
  return TNX_OK;
}

extern "C" int tnx_embed_packed(void* stream, const uint16_t* table, int64_t V, int64_t D, const int32_t* ids, int64_t ids_ld, int64_t B, int64_t T, float scale,
                                const tnx_packed_rows* packed, uint16_t* out) {
  TNX_REQUIRE(table && ids && out, "embed: null pointer");
  TNX_REQUIRE(V > 0 && D > 0 && B > 0 && T > 0, "embed: bad shape");
  PackedRows rows;
  const int rc = packed_args(packed, B, T, rows);
  if (rc) return rc;
  hipLaunchKernelGGL(embed_kernel, dim3((unsigned)(B * T)), dim3(256), 0, as_stream(stream), table, V, D, ids, ids_ld, nullptr, T, host_round_bf16(scale), out, rows);
  TNX_CHECK_LAUNCH("embed_packed");
  return TNX_OK;
}

extern "C" int tnx_rmsnorm(void* stream, const uint16_t* x, const uint16_t* res_pre,
                           uint16_t* h_out, const uint16_t* w, const uint16_t* res_post,
                           uint16_t* y, int64_t M, int64_t D, float eps, int flavor) {
  TNX_REQUIRE(x && w && y, "rmsnorm: null pointer");
  TNX_REQUIRE(M > 0 && D > 0 && D <= 16384, "rmsnorm: D=%lld out of range (1..16384)", (long long)D);
  TNX_REQUIRE(flavor >= TNX_NORM_LLAMA && flavor <= TNX_NORM_GEMMA3, "rmsnorm: bad flavor %d", flavor);
  if (D % 8 == 0 && D <= 8 * 256 * kNormMaxChunks)
    launch_rmsnorm_vec(as_stream(stream), M, flavor, kNormInRow, NormRow{x, res_pre, h_out, w, res_post, y, D, eps});
  else
    hipLaunchKernelGGL(rmsnorm_kernel, dim3((unsigned)M), dim3(256), (size_t)D * sizeof(float),
                       as_stream(stream), x, res_pre, h_out, w, res_post, y, D, eps, flavor);
  TNX_CHECK_LAUNCH("rmsnorm");
  return TNX_OK;
}

extern "C" int tnx_rmsnorm_splitk(void* stream, const float* ws, int split_k, const uint16_t* res_pre,
                                  uint16_t* h_out, const uint16_t* w, const uint16_t* res_post,
                                  uint16_t* y, int64_t M, int64_t D, float eps, int flavor) {
  TNX_REQUIRE(ws && w && y, "rmsnorm_splitk: null pointer");
  TNX_REQUIRE(split_k >= 1, "rmsnorm_splitk: split_k must be >= 1");
  TNX_REQUIRE(M > 0 && D > 0 && D % 8 == 0 && D <= 8 * 256 * kNormMaxChunks,
              "rmsnorm_splitk: D=%lld must be a multiple of 8 and <= 16384", (long long)D);
  TNX_REQUIRE(flavor >= TNX_NORM_LLAMA && flavor <= TNX_NORM_GEMMA3, "rmsnorm_splitk: bad flavor %d", flavor);
  launch_rmsnorm_vec(as_stream(stream), M, flavor, kNormInPlanes,
                     NormRow{nullptr, res_pre, h_out, w, res_post, y, D, eps, ws, split_k, (int64_t)(M * D)});
  TNX_CHECK_LAUNCH("rmsnorm_splitk");
  return TNX_OK;
}

extern "C" int tnx_rmsnorm_moe_combine(void* stream, const uint16_t* y_route, const uint16_t* topk_w, int k,
                                       const uint16_t* res_pre, uint16_t* h_out, const uint16_t* w,
                                       const uint16_t* res_post, uint16_t* y, int64_t M, int64_t D, float eps,
                                       int flavor) {
  TNX_REQUIRE(y_route && topk_w && w && y, "rmsnorm_moe_combine: null pointer");
  TNX_REQUIRE(k >= 1, "rmsnorm_moe_combine: k must be >= 1");
  TNX_REQUIRE(M > 0 && D > 0 && D % 8 == 0 && D <= 8 * 256 * kNormMaxChunks,
              "rmsnorm_moe_combine: D=%lld must be a multiple of 8 and <= 16384", (long long)D);
  TNX_REQUIRE(flavor >= TNX_NORM_LLAMA && flavor <= TNX_NORM_GEMMA3, "rmsnorm_moe_combine: bad flavor %d", flavor);
  launch_rmsnorm_vec(as_stream(stream), M, flavor, kNormInRoutes,
                     NormRow{y_route, res_pre, h_out, w, res_post, y, D, eps, nullptr, k, 0, nullptr, nullptr, topk_w});
  TNX_CHECK_LAUNCH("rmsnorm_moe_combine");
  return TNX_OK;
}

extern "C" int tnx_rmsnorm_pair(void* stream, const uint16_t* x, const float* ws, int split_k,
                                const uint16_t* res_pre, uint16_t* h_out, const uint16_t* w,
                                const uint16_t* res_post, uint16_t* y, const uint16_t* w2, uint16_t* y2,
                                int64_t M, int64_t D, float eps, int flavor) {
  TNX_REQUIRE((x != nullptr) != (ws != nullptr), "rmsnorm_pair: exactly one of x and ws must be given");
  TNX_REQUIRE(w && y && w2 && y2, "rmsnorm_pair: null pointer");
  if (ws) TNX_REQUIRE(split_k >= 1, "rmsnorm_pair: split_k must be >= 1");
  TNX_REQUIRE(M > 0 && D > 0 && D % 8 == 0 && D <= 8 * 256 * kNormMaxChunks,
              "rmsnorm_pair: D=%lld must be a multiple of 8 and <= 16384", (long long)D);
  TNX_REQUIRE(flavor >= TNX_NORM_LLAMA && flavor <= TNX_NORM_GEMMA3, "rmsnorm_pair: bad flavor %d", flavor);
  launch_rmsnorm_vec(as_stream(stream), M, flavor, ws ? kNormInPlanes : kNormInRow,
                     NormRow{x, res_pre, h_out, w, res_post, y, D, eps, ws, ws ? split_k : 0, (int64_t)(M * D), w2, y2});
  TNX_CHECK_LAUNCH("rmsnorm_pair");
  return TNX_OK;
}

// e: the rows come from a table, which `d` names as its x
static int norm_lora(void* stream, const tnx_norm_lora_desc* d, const EmbedSrc* e) {
  TNX_REQUIRE(!d->w2 == !d->y2 && !(d->w2 && d->y_route), "norm_lora: the second norm takes w2 and y2, and rows or planes");
  TNX_REQUIRE(d->w && d->y && (e || d->a_t) && (!d->a_t || d->t), "norm_lora: null pointer");
  const int64_t M = d->M, D = d->D;
  TNX_REQUIRE(M > 0 && D > 0 && D % 32 == 0 && D <= 8 * 256 * kNormMaxChunks, "norm_lora: D=%lld must be a multiple of 32 and <= 16384", (long long)D);
  if (d->a_t) TNX_REQUIRE(d->R > 0 && d->R % 16 == 0 && d->t_ld >= d->R, "norm_lora: R=%d must be a multiple of 16 and <= t_ld", d->R);
  TNX_REQUIRE(d->flavor >= TNX_NORM_LLAMA && d->flavor <= TNX_NORM_GEMMA3, "norm_lora: bad flavor %d", d->flavor);
  if (d->ws) TNX_REQUIRE(d->split_k >= 1, "norm_lora: split_k must be >= 1");
  if (d->y_route) TNX_REQUIRE(d->topk_w && d->k >= 1, "norm_lora: y_route needs topk_w and k >= 1");
  const int in = e ? kNormInTable : d->ws ? kNormInPlanes : d->y_route ? kNormInRoutes : kNormInRow;
  const int parts = d->ws ? d->split_k : d->y_route ? d->k : 0;
  const NormRow n{d->y_route ? d->y_route : d->x, d->res_pre, d->h_out, d->w, d->res_post, d->y, D, d->eps, d->ws, parts, M * D, d->w2, d->y2, d->topk_w,
                  e ? *e : EmbedSrc{}};
  if (!d->a_t) {
    launch_rmsnorm_vec(as_stream(stream), M, d->flavor, in, n);
    TNX_CHECK_LAUNCH("norm_lora");
    return TNX_OK;
  }
  // A row's work-groups read it while the first of them writes it and each writes its adapter columns: no output may lie in an input, and t not
  // in another output either.
  const int64_t row_bytes = M * D * 2, t_bytes = ((M - 1) * d->t_ld + d->R) * 2;
  struct Range { const void* p; int64_t bytes; };
  const Range ins[] = {{d->x, e ? e->V * D * 2 : row_bytes}, {d->ws, 2 * parts * row_bytes}, {d->y_route, parts * row_bytes}, {d->res_pre, row_bytes}, {d->res_post, row_bytes}};
  const Range outs[] = {{d->h_out, row_bytes}, {d->y, row_bytes}, {d->y2, row_bytes}};
  bool separate = apart(d->t, t_bytes, d->topk_w, M * parts * 2) && apart(d->t, t_bytes, d->w, D * 2) && apart(d->t, t_bytes, d->w2, D * 2);
  for (const Range& in : ins) {
    separate = separate && apart(d->t, t_bytes, in.p, in.bytes);
    for (const Range& out : outs) separate = separate && apart(out.p, out.bytes, in.p, in.bytes);
  }
  for (const Range& out : outs) separate = separate && apart(d->t, t_bytes, out.p, out.bytes);
  if (separate && norm_lora_one_launch(M, D, d->R)) {
    launch_rmsnorm_lora(as_stream(stream), M, d->flavor, in, n, RowAdapterArgs{d->a_t, d->R, row_adapter_cols(M, d->R), d->t, d->t_ld, 0, 0});
    TNX_CHECK_LAUNCH("norm_lora");
    return TNX_OK;
  }
  launch_rmsnorm_vec(as_stream(stream), M, d->flavor, in, n);
  TNX_CHECK_LAUNCH("norm_lora");
  return tnx_lora_down(stream, d->w2 ? d->y2 : d->y, M, D, d->a_t, d->R, d->t, d->t_ld);
}

extern "C" int tnx_norm_lora(void* stream, const tnx_norm_lora_desc* d) {
  TNX_REQUIRE(d, "norm_lora: null descriptor");
  TNX_REQUIRE((d->x != nullptr) + (d->ws != nullptr) + (d->y_route != nullptr) == 1, "norm_lora: exactly one of x, ws and y_route must be given");
  return norm_lora(stream, d, nullptr);
}

// A launch less ahead of the first layer, two where the step wants a rope table: 2.8 + 3.9 us of the tiny model's step, 4.6 + 4.6 + 5.2 of 16 rows of 4096.
extern "C" int tnx_embed_norm(void* stream, const tnx_embed_desc* e, const tnx_norm_lora_desc* d) {
  TNX_REQUIRE(e && d, "embed_norm: null descriptor");
  TNX_REQUIRE(e->table && e->ids && d->h_out, "embed_norm: null pointer");
  TNX_REQUIRE(!d->x && !d->ws && !d->y_route && !d->res_pre && !d->res_post && !d->w2, "embed_norm: the rows come from the table, with one norm behind them");
  TNX_REQUIRE(e->V > 0 && e->B > 0 && e->T > 0 && d->M == e->B * e->T && d->M < (1ll << 31), "embed_norm: bad shape");
  RopeTable rope{};
  if (e->sin_out) {
    TNX_REQUIRE(e->positions && e->col_ptr && e->timescale && e->cos_out, "embed_norm: null pointer");
    TNX_REQUIRE(e->dh % 2 == 0 && e->dh >= 2 && e->dh <= 2048, "embed_norm: bad shape");
    rope = RopeTable{e->positions, e->pos_ld, e->B, e->timescale, e->dh / 2, e->sin_out, e->cos_out};
  }
  const EmbedSrc src{e->ids, e->ids_ld, e->col_ptr, e->V, (uint32_t)e->T, host_round_bf16(e->scale), rope, 0};
  tnx_norm_lora_desc rows = *d;
  rows.x = e->table;
  return norm_lora(stream, &rows, &src);
}

extern "C" int tnx_rope_table(void* stream, const int32_t* positions, int64_t pos_ld, const int32_t* col_ptr,
                              int64_t B, const float* timescale, int dh, float* sin_out, float* cos_out) {
  TNX_REQUIRE(positions && col_ptr && timescale && sin_out && cos_out, "rope_table: null pointer");
  TNX_REQUIRE(B > 0 && dh % 2 == 0 && dh >= 2 && dh <= 2048, "rope_table: bad shape");
  hipLaunchKernelGGL(rope_table_kernel, dim3((unsigned)B), dim3((unsigned)(dh / 2 < 64 ? 64 : dh / 2)), 0, as_stream(stream),
                     RopeTable{positions, pos_ld, B, timescale, dh / 2, sin_out, cos_out}, col_ptr);
  TNX_CHECK_LAUNCH("rope_table");
  return TNX_OK;
}

static int qknorm_rope_kvwrite(void* stream, const tnx_rope_desc* d, const tnx_packed_rows* packed) {
  RopeArgs a;
  int rc = rope_args(d, a);
  if (rc == TNX_OK && packed) rc = packed_args(packed, d->B, d->T, a.rows);
  if (rc) return rc;
  // many rows, from the finished linear output: the row kernel.  Its thread groups are a head's dh / 16 lanes, whole ones in a
  // work-group and, where they add up a head's squares, inside a wave and a power of two.
  const int chunks = d->dh / 16;
  const bool norm = d->qk_norm >= 0;
  const bool aligned = (((uintptr_t)d->qkv | (uintptr_t)d->q_out | (uintptr_t)d->kcache | (uintptr_t)d->vcache) & 15) == 0 &&
                       (!norm || (((uintptr_t)d->q_norm_w | (uintptr_t)d->k_norm_w) & 15) == 0);
  TNX_REQUIRE(d->B * d->T < (int64_t)1 << 31, "rope: too many rows");
  // Normed heads: the per-head kernel has a work-group for every head, the row kernel one for a row, whose chain (sines, barrier, loads, the
  // sum over lanes) is the longer; the fewer heads, the more rows it takes until the per-head one has enough of them.  us, per head | per row,
  // 256, 512, 1024 rows: 32 + 2 x 4 heads of 128 6.3 | 8.6, 9.5 | 9.4, 16.1 | 12.0; 8 + 2 x 2 of 64 3.6 | 5.1, 4.4 | 5.4, 6.1 | 5.7;
  // 4 + 2 x 1 of 256 3.7 | 5.5, 4.7 | 6.2, 6.7 | 6.6; 64 + 2 x 8 of 128 9.9 | 11.5, 16.1 | 13.3, 29.1 | 18.2.
  const int64_t from = norm ? 384 + 5120 / (d->Hq + 2 * d->Hkv > 0 ? d->Hq + 2 * d->Hkv : 1) : 256;
  if (!d->qkv_ws && d->B * d->T >= from && d->dh % 16 == 0 && 256 % chunks == 0 && aligned) {
    if (norm) hipLaunchKernelGGL(rope_rows_kernel<true>, dim3((unsigned)(d->B * d->T)), dim3(256), 0, as_stream(stream), a);
    else hipLaunchKernelGGL(rope_rows_kernel<false>, dim3((unsigned)(d->B * d->T)), dim3(256), 0, as_stream(stream), a);
    TNX_CHECK_LAUNCH("qknorm_rope_kvwrite (rows)");
    return TNX_OK;
  }
  dim3 grid((unsigned)(d->B * d->T), (unsigned)(d->Hq + 2 * d->Hkv)), block((unsigned)(cdiv(d->dh / 2, 64) * 64));
  if (d->qkv_ws) hipLaunchKernelGGL(rope_kernel<true>, grid, block, 0, as_stream(stream), a);
  else hipLaunchKernelGGL(rope_kernel<false>, grid, block, 0, as_stream(stream), a);
  TNX_CHECK_LAUNCH("qknorm_rope_kvwrite");
  return TNX_OK;
}
extern "C" int tnx_qknorm_rope_kvwrite(void* stream, const tnx_rope_desc* d) { return qknorm_rope_kvwrite(stream, d, nullptr); }
extern "C" int tnx_qknorm_rope_kvwrite_packed(void* stream, const tnx_rope_desc* d, const tnx_packed_rows* rows) {
  TNX_REQUIRE(rows, "rope: null packed rows");
  return qknorm_rope_kvwrite(stream, d, rows);
}
