// GQA attention over the KV cache with a wavefront-level online softmax.
//
// One wave owns a tile of 16 query vectors that share a (batch row, kv head): the G query
// heads of the group (decode), or G heads x 16/G consecutive positions (prefill).  Scores are
// computed transposed, S^T[key, query] = K . q^T, so that every lane ends up holding the
// probabilities of ONE query column for 8 keys -- exactly the A fragment of the P.V MFMA --
// and the max / sum of the online softmax are per-lane scalars reduced over 4 lanes.  V rows
// are loaded in their natural [key][dh] layout (256 B contiguous per key) and transposed
// inside each lane with v_perm_b32 to form B fragments; keys and values go through LDS only in the work-group form for many positions below.
// In a decode step of up to 512 work-groups four waves share a chunk's keys and merge what they have through LDS (several_waves).
#include <string.h>

#include <mutex>
#include <type_traits>

#include "attn_parts.h"
#include "common.h"
#include "gemm_tile.h"   // dma16, raw_rsrc, tnx_wait_vm
#include "rope_math.h"
#include "row_adapter.h"

// Register stages of the key-block ring (head_dim <= 128).  Two: one block in flight while one is
// computed.  A compute unit draws 21-28 GB/s from memory whatever its waves request, so a
// third stage adds nothing to the stream, and its 72 registers push ring registers into AGPRs,
// whose copies wait on loads in flight (measured: 46.5 / 64.8 us with two stages against
// 47.9 / 67.3 us with three at contexts 528 / 768).
#ifndef TNX_ATTN_NS
#define TNX_ATTN_NS 2
#endif

namespace {

struct AttnArgs {
  int64_t B, T, S;
  int Hq, Hkv, dh, G, Gp;
  int gp_shift;                // Gp = 1 << gp_shift (the query group padded to a power of two)
  unsigned QT;                 // query tiles per row: ceil(T / (16 / Gp))
  unsigned QTG;                // (attn_tiles_kernel) groups of QW query tiles per row
  float scale_bf;  // bf16-rounded scale, 0 = none
  int window;
  int32_t pad_id;
  const uint16_t* q;
  const uint16_t* k;
  const uint16_t* v;
  const int32_t* tokens;       // token ids, or (seg_mode) the segment ids of a packed batch
  int64_t tok_ld;
  int seg_mode;                // 0: a key counts when its token != pad_id; 1: when its segment id equals the query's
  const int32_t* col_ptr;
  int kv_chunk, n_chunks;
  float* ws;
  uint16_t* out;
  // fused RoPE + cache write of the step's own token (decode, T == 1, no q/k norm, Llama
  // rotation): the query, key and value come from the qkv linear's output instead of q / the cache
  const float* qkv_ws;        // split-k partial planes [qkv_split][B][(Hq + 2 Hkv) * dh], or null
  const uint16_t* qkv;        // ... or the finished bf16 output
  int qkv_split;
  const float* rope_sin;      // fp32 [B, dh/2] of this step's positions; non-null switches the mode on
  const float* rope_cos;
  PackedRows rows;             // prompts (T > 1) without their padding
};


// f over the four lanes lm + 16 {0, 1, 2, 3} that share a query, in all of them
template <class F>
__device__ __forceinline__ float across_quarters(float x, F f) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = f(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return f(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

// FUSE: 0 = q comes rotated, keys and values are in the cache; 1 = the fused rotation and cache
// write of a decode step (below), qkv taken from the finished output or from any number of
// partial planes; 2 = the same from at most eight partial planes and at most four query heads per
// kv head (one set of 3 x 64 lanes x 16 bytes per plane), all fetched in one round trip; 3 = any rotation, behind per-head norms or not, from
// at most eight partial planes (RopeArgs), the heads divided among the work-group's waves; 4 = 3, the keys of at most two blocks by one wave.
// W: waves of a work-group.  Of more than one (a decode step: T == 1) each takes an equal share of the key blocks that the work-group's
// chunk of the cache holds by now, and they merge what they have through LDS: the pass that would merge them otherwise is a launch, and its partials
// a round trip to memory.  32 heads on 8, with the o adapter's 64 columns behind it, us before | now: 16 rows x 192 keys 14.0 | 12.7, 700 keys 19.9 |
// 16.9, 8 rows x 1000 18.8 | 15.5, 1 row x 732 15.6 | 13.3, 3 rows x 2940 22.8 | 18.7, 64 rows x 372 27.6 | 23.3; 4 heads of 256 on one, 32 columns:
// 64 rows x 288 14.7 | 12.0, 16 rows x 1200 21.7 | 14.6.
constexpr int kAttnWaves = 4;
template <int DH, int FUSE, bool TOKVEC, int W>
__device__ __forceinline__ void attn_body(const AttnArgs& a, const RopeArgs& r) {
  constexpr bool formed = FUSE >= 3;           // the heads come out of this launch's planes
  // FUSE 4, few keys: one wave takes them all, the step's own among them, in the order and with the roundings of the launch without the
  // rotation, for the same time (4.7 ms for a rollout of 32 steps at 48 columns, either way): divided, other last bits turned near-ties of
  // a routed decoder's experts.
  constexpr bool few = FUSE == 4;
  static_assert(!formed || (W > 1 && DH <= 128), "the heads are divided among waves, a pair of dimensions per lane");
  constexpr int KS = DH / 32;                 // k-steps of the QK product
  constexpr int NH = DH > 128 ? DH / 128 : 1; // 128-column halves of V / O
  constexpr int NS = DH > 128 ? 1 : TNX_ATTN_NS;        // register stages of the key-block pipeline
  const int lane = threadIdx.x & 63, lm = lane & 15, lq = lane >> 4;
  const int wave = W > 1 ? __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)) : 0;
  const int chunk = blockIdx.x, hkv = blockIdx.y;
  // (shifts and one unsigned division: a general integer division costs some forty instructions,
  // and the chain in front of this kernel's first loads had several of them)
  const int PT = 16 >> a.gp_shift;                       // positions per query tile
  const unsigned bz = blockIdx.z;
  const int64_t b = FUSE != 0 ? bz : bz / a.QT;          // (the fused decode step has one query tile per row)
  const int qt = FUSE != 0 ? 0 : (int)(bz - (unsigned)b * a.QT);
  // formed: this wave's first heads of the G + 2 of the (row, kv head), all planes at once, ahead of everything that waits for the column.
  // Lane i has dimensions i and i + DH / 2.
  constexpr int HB = 3, HALF = DH / 2;
  const int il = min(lane, HALF - 1);
  struct HeadPlanes {
    float p1[HB][8], p2[HB][8];
  };
  auto load_heads = [&](int h0, HeadPlanes& hp) {
    const int ld = (a.Hq + 2 * a.Hkv) * DH;
    const int64_t plane = a.B * (int64_t)ld;
#pragma unroll
    for (int u = 0; u < HB; ++u) {
      const int hs = min(h0 + u * W + wave, a.G + 1);
      const int head = hs < a.G ? hkv * a.G + hs : (hs == a.G ? a.Hq + hkv : a.Hq + a.Hkv + hkv);
      const float* src = r.ws + b * (int64_t)ld + (int64_t)head * DH + il;
#pragma unroll
      for (int z = 0; z < 8; ++z) {
        const float* p = src + (int64_t)min(z, r.split_k - 1) * plane;
        hp.p1[u][z] = p[0];
        hp.p2[u][z] = p[HALF];
      }
    }
  };
  HeadPlanes hp;
  float timescale = 1.f;
  uint16_t wq[2] = {0, 0}, wk[2] = {0, 0};
  if constexpr (formed) {
    load_heads(0, hp);
    timescale = r.timescale[il];
    if (r.qk_norm >= 0)
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        wq[e] = r.q_norm_w[il + e * HALF];
        wk[e] = r.k_norm_w[il + e * HALF];
      }
    __builtin_amdgcn_sched_barrier(0);
  }
  const int col0 = *a.col_ptr;

  // query column of this lane (as B-fragment column and as softmax owner)
  const int g = lm & (a.Gp - 1), tq = qt * PT + (lm >> a.gp_shift);
  const bool packed = FUSE == 0 && W == 1 && a.rows.base != nullptr;
  const int start = packed ? a.rows.starts[b] : 0;
  const int64_t row0 = packed ? a.rows.base[b] : b * a.T;   // a row's position 0
  if (packed && qt * PT + PT <= start) return;
  const bool qvalid = g < a.G && tq < a.T && tq >= start;
  const int c_n = col0 + tq;                              // cache slot of the query token
  const int lo_n = a.window > 0 ? max(0, c_n - a.window + 1) : 0;
  const int64_t qvec = (row0 + (qvalid ? tq : a.T - 1)) * a.Hq + hkv * a.G + (qvalid ? g : 0);

  // key range of the tile
  const int t_last = min((int)a.T - 1, qt * PT + PT - 1);
  int k_hi = col0 + t_last;                               // inclusive
  int k_lo = max(start, a.window > 0 ? col0 + qt * PT - a.window + 1 : 0);
  if (a.kv_chunk > 0) {
    k_lo = max(k_lo, chunk * a.kv_chunk);
    k_hi = min(k_hi, chunk * a.kv_chunk + a.kv_chunk - 1);
  }

  constexpr bool fused = FUSE != 0;                         // T == 1: c_n = col0 for every lane
  // the chunk that owns the new token (of its waves the last, which has the fewest blocks)
  const bool writer = fused && col0 >= k_lo && col0 <= k_hi && wave == W - 1;
  if constexpr (W > 1) {
    constexpr int N = few ? 1 : W;
    if (fused && !few) k_hi = min(k_hi, col0 - 1);
    const int first = k_lo & ~31, each = (max(k_hi - first + 32, 0) / 32 + N - 1) / N * 32;
    k_lo = max(k_lo, first + wave * each);
    k_hi = min(k_hi, first + (wave + 1) * each - 1);
  }
  u32x4 qf[KS];
#pragma unroll
  for (int j = 0; j < KS; ++j) {
    qf[j] = u32x4{0, 0, 0, 0};
    if (qvalid && !fused) qf[j] = *reinterpret_cast<const u32x4*>(a.q + qvec * DH + j * 32 + lq * 8);
  }
  // in fused mode the step's own key / value never come from the cache: the loop stops one key
  // short and they are added from registers at the end
  // (of few keys they take the place of what the cache held in their block)
  int key_hi = fused && !few ? c_n - 1 : c_n;
  if (fused && !few) k_hi = min(k_hi, col0 - 1);

  f32x4 O[NH][8];
#pragma unroll
  for (int h = 0; h < NH; ++h)
#pragma unroll
    for (int jj = 0; jj < 8; ++jj) O[h][jj] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m_run = kNegBig, l_run = 0.f;

  const uint16_t* kbase = a.k + ((b * a.Hkv + hkv) * a.S) * DH;
  const uint16_t* vbase = a.v + ((b * a.Hkv + hkv) * a.S) * DH;
  const int32_t* tok = a.tokens + b * a.tok_ld;
  // what a key's id is compared with: the pad id (the key counts when it differs), or, for packed
  // batches, the segment id of this lane's query token (the key counts when it is equal).  The
  // query's id is fetched behind the first key blocks and planes (a load in front of them would
  // hold them back until the step counter it depends on has arrived), in both modes: a branch
  // around a load would make the counted waits behind it inexact.
  int32_t id_ref = a.pad_id;
  const bool id_equal = a.seg_mode != 0;
  auto fetch_query_id = [&]() {
    const int32_t id_q = tok[min((int64_t)c_n, a.tok_ld - 1)];
    id_ref = a.seg_mode ? id_q : a.pad_id;
  };
  const int vcol = (8 * lm) % (DH < 128 ? DH : 128);     // DH=64: upper lanes duplicate
  // TOKVEC: 16-byte token loads; the host chooses them when rows are 16-byte aligned and hold
  // whole groups of four slots (keys beyond the range are masked by the range test anyway).  A
  // compile-time choice: a branch around loads would make every wait behind it assume that the
  // shorter side was taken.

  // NS register stages: the loads of the next key block are in flight while a block is computed, so the memory system is never left idle behind a
  // wave's softmax and MFMAs.  No load of the loop stands behind a branch, so that the number in flight is static and the wait for a stage's data does
  // not drain the younger one; the last one or two blocks have code of their own (below), and none is loaded twice.
  struct Stage {
    u32x4 kf[2][KS];
    u32x4 vf[NH][8];
    int tk[8];
  };
  // K / V of this (row, kv head) and the row's token ids as buffer resources: a lane's byte
  // offset is a per-kernel constant plus the block's first key, so a block costs a handful of
  // address instructions, and keys past the cache (S not a multiple of 32, or a prefetch past
  // the end) read zeros; they are masked by the range test anyway.
  const uint32_t slab_bytes = (uint32_t)a.S * DH * 2u;
  const rsrc_t rk = make_rsrc(kbase, slab_bytes), rv = make_rsrc(vbase, slab_bytes);
  // (the row holds tok_ld ids: slots past them read zeros, and the range test masks them)
  const rsrc_t rtok = make_rsrc(tok, (uint64_t)min(a.S, a.tok_ld) * 4);
  const uint32_t koff = (uint32_t)(lm * DH + lq * 8) * 2u;           // + tt * 16 keys, + j * 64 B
  const uint32_t voff = (uint32_t)(4 * lq * DH + vcol) * 2u;         // + s keys, + 16 keys, + h * 256 B
  auto load_block = [&](int kb, Stage& sg) {
    const uint32_t kb_bytes = (uint32_t)kb * (DH * 2u);
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
      const uint32_t o = koff + kb_bytes + (uint32_t)(tt * 16 * DH * 2);
#pragma unroll
      for (int j = 0; j < KS; ++j) sg.kf[tt][j] = __builtin_amdgcn_raw_buffer_load_b128(rk, o + (uint32_t)(j * 64), 0, kStreamOnce);
    }
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      const uint32_t o = voff + kb_bytes + (uint32_t)(((s < 4 ? s : 12 + s)) * DH * 2);
#pragma unroll
      for (int h = 0; h < NH; ++h) sg.vf[h][s] = __builtin_amdgcn_raw_buffer_load_b128(rv, o + (uint32_t)(h * 256), 0, kStreamOnce);
    }
    // token ids of this lane's 8 keys (two runs of 4 consecutive slots), fetched unconditionally
    // together with K and V: a predicated load per key would serialise eight memory latencies
    if constexpr (TOKVEC) {
      const u32x4 t0 = __builtin_amdgcn_raw_buffer_load_b128(rtok, (uint32_t)(kb + 4 * lq) * 4u, 0, 0);
      const u32x4 t1 = __builtin_amdgcn_raw_buffer_load_b128(rtok, (uint32_t)(kb + 16 + 4 * lq) * 4u, 0, 0);
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        sg.tk[s] = (int)t0[s];
        sg.tk[4 + s] = (int)t1[s];
      }
    } else {
#pragma unroll
      for (int s = 0; s < 8; ++s)
        sg.tk[s] = (int)__builtin_amdgcn_raw_buffer_load_b32(
            rtok, (uint32_t)(kb + (s < 4 ? 4 * lq + s : 16 + 4 * lq + (s - 4))) * 4u, 0, 0);
    }
  };
  __shared__ __align__(16) uint16_t rot[formed ? 18 * DH : 8];   // the rotated heads: queries, key, value
  auto compute_block = [&](int kb, Stage& sg) {
    if constexpr (few) {
      if (kb == (col0 & ~31)) {
#pragma unroll
        for (int tt = 0; tt < 2; ++tt)
          if (kb + tt * 16 + lm == col0)
#pragma unroll
            for (int j = 0; j < KS; ++j) sg.kf[tt][j] = *reinterpret_cast<const u32x4*>(&rot[a.G * DH + j * 32 + lq * 8]);
#pragma unroll
        for (int s = 0; s < 8; ++s)
          if (kb + 4 * lq + (s < 4 ? s : 12 + s) == col0) sg.vf[0][s] = *reinterpret_cast<const u32x4*>(&rot[(a.G + 1) * DH + vcol]);
      }
    }
    bool kvalid[8];
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      const int key = kb + (s < 4 ? 4 * lq + s : 16 + 4 * lq + (s - 4));
      kvalid[s] = qvalid && key >= max(k_lo, lo_n) && key <= min(k_hi, key_hi) && ((sg.tk[s] == id_ref) == id_equal);
    }
    // ---- S^T = K . q^T ----
    f32x4 st[2];
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
      st[tt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < KS; ++j) st[tt] = mfma16(sg.kf[tt][j], qf[j], st[tt]);
    }
    float sv[8];
    float bmax = kNegBig;
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      float x = rbf(st[s >> 2][s & 3]);
      if (a.scale_bf != 0.f) x = rbf(x * a.scale_bf);
      sv[s] = x;
      if (kvalid[s]) bmax = fmaxf(bmax, x);
    }
    const float m_new = fmaxf(m_run, across_quarters(bmax, [](float x, float y) { return fmaxf(x, y); }));
    const float alpha = __expf(m_run - m_new);
    m_run = m_new;
    float p[8], psum = 0.f;
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      p[s] = kvalid[s] ? __expf(sv[s] - m_new) : 0.f;
      psum += p[s];
    }
    l_run = l_run * alpha + psum;
    u32x4 pa;
    pa[0] = pack2bf(p[0], p[1]);
    pa[1] = pack2bf(p[2], p[3]);
    pa[2] = pack2bf(p[4], p[5]);
    pa[3] = pack2bf(p[6], p[7]);
    // ---- O = O * alpha + P . V ----
    // the running maximum settles after a few blocks: rescale O only when some column moved
    if (__builtin_amdgcn_ballot_w64(alpha != 1.0f) != 0) {
      float ar[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) ar[i] = __shfl(alpha, 4 * lq + i, 64);
#pragma unroll
      for (int h = 0; h < NH; ++h)
#pragma unroll
        for (int jj = 0; jj < 8; ++jj)
#pragma unroll
          for (int i = 0; i < 4; ++i) O[h][jj][i] *= ar[i];
    }
#pragma unroll
    for (int h = 0; h < NH; ++h)
#pragma unroll
      for (int jj = 0; jj < 8; ++jj) {
        const uint32_t sel = (jj & 1) ? 0x07060302u : 0x05040100u;
        u32x4 bfrag;
#pragma unroll
        for (int r = 0; r < 4; ++r)
          bfrag[r] = __builtin_amdgcn_perm(sg.vf[h][2 * r + 1][jj >> 1], sg.vf[h][2 * r][jj >> 1], sel);
        O[h][jj] = mfma16(pa, bfrag, O[h][jj]);
      }
  };
  // a wave's staged q / k / v, later its part of the output
  __shared__ __align__(16) float stage[FUSE || W > 1 ? W : 1][FUSE == 1 || FUSE == 2 ? 18 * DH : W > 1 ? 16 * DH : 1];
  {
    Stage sg[NS];
    const int kb0 = k_lo & ~31;
    const int kb_last = k_hi & ~31;
    const bool any = kb0 <= k_hi;
    // (issued even when the key range is empty: a block outside the slab reads zeros, and an
    // unconditional load keeps the counted waits behind it exact)
    auto issue_stage = [&](int u) { load_block(min(kb0 + 32 * u, kb_last), sg[u]); };
    auto issue_ring = [&]() {
#pragma unroll
      for (int u = 0; u < NS - 1; ++u) issue_stage(u);
    };
    // Without the fused rotation the first key blocks are requested right away.  With it the
    // partial planes of this step's q / k / v go first: a wave's loads return in order, so
    // planes requested behind 32 KiB of keys and values would only be usable once those have
    // arrived, and the rotation would start late instead of running while the blocks stream in.
    if constexpr (!fused) {
      issue_ring();
      fetch_query_id();
    }
    // the step's own key / value wait in LDS while the cached keys stream through the registers
    constexpr bool parked = FUSE == 1 || FUSE == 2;
    __shared__ u32x4 park_w[parked ? W : 1][parked ? KS + NH : 1][64];
    auto& park = park_w[parked ? wave : 0];
    if constexpr (formed) {
      const float pos = (float)r.positions[b * r.pos_ld + col0];
      load_block(min(k_lo & ~31, k_hi & ~31), sg[0]);
      fetch_query_id();
      float sn, cs;
      rope_angle(r, pos, timescale, sn, cs);   // (while the planes arrive)
      for (int h0 = 0; h0 < a.G + 2; h0 += HB * W) {
        if (h0 > 0) load_heads(h0, hp);
#pragma unroll
        for (int u = 0; u < HB; ++u) {
          const int hs = h0 + u * W + wave;
          const bool is_v = hs > a.G, is_q = hs < a.G;
          if (hs >= a.G + 2) continue;   // (uniform)
          float x1 = 0.f, x2 = 0.f;
#pragma unroll
          for (int z = 0; z < 8; ++z)
            if (z < r.split_k) {
              x1 += hp.p1[u][z];
              x2 += hp.p2[u][z];
            }
          x1 = rbf(x1);
          x2 = rbf(x2);
          if (!is_v) {
            if (r.qk_norm >= 0) {
              const float ms = finish_ms(wave_sum(lane < HALF ? sq_term(x1, r.qk_norm) + sq_term(x2, r.qk_norm) : 0.f), (float)DH, r.qk_norm);
              x1 = norm_elem(x1, bf2f(is_q ? wq[0] : wk[0]), ms, r.norm_eps, r.qk_norm);
              x2 = norm_elem(x2, bf2f(is_q ? wq[1] : wk[1]), ms, r.norm_eps, r.qk_norm);
            }
            float o1, o2;
            rotate_pair(r, is_q, x1, x2, sn, cs, o1, o2);
            x1 = o1;
            x2 = o2;
          }
          if (lane < HALF) {
            rot[hs * DH + lane] = f2bf(x1);
            rot[hs * DH + lane + HALF] = f2bf(x2);
          }
        }
      }
      __syncthreads();
      const u32x4* heads = reinterpret_cast<const u32x4*>(rot);
#pragma unroll
      for (int j = 0; j < KS; ++j)
        if (qvalid) qf[j] = heads[(g * DH + j * 32 + lq * 8) / 8];
      if (writer) {
        const int64_t slot = ((b * a.Hkv + hkv) * a.S + ring_slot(col0, a.S)) * DH;
        for (int c = lane; c < DH / 8; c += 64) {
          *reinterpret_cast<u32x4*>(const_cast<uint16_t*>(a.k) + slot + c * 8) = heads[a.G * DH / 8 + c];
          *reinterpret_cast<u32x4*>(const_cast<uint16_t*>(a.v) + slot + c * 8) = heads[(a.G + 1) * DH / 8 + c];
        }
      }
    }
    if constexpr (parked) {
      u32x4 kn[KS], vn[NH];
      // ---- this step's q (G heads), k and v of the kv head from the qkv linear's output, RoPE
      // applied as the stand-alone kernel does; the first key blocks are already in flight ----
      const int ld = (a.Hq + 2 * a.Hkv) * DH;
      const int64_t plane = a.B * (int64_t)ld;
      const int64_t rowoff = b * (int64_t)ld;
      // The G query heads, the key head and the value head of this (row, kv head), (G + 2) * DH
      // values, are fetched once by the whole wave (16 bytes per lane and plane, all planes of
      // a group in flight together), summed in split order, rounded to bf16 and staged in LDS,
      // from where every lane picks the elements of its fragments.
      float* xs = stage[wave];
      // sine / cosine of this row's position: a per-step table (tnx_rope_table), computed with
      // the arithmetic of the stand-alone kernel; fetched together with the planes
      float sn[KS / 2][8], cs[KS / 2][8];
      {
        f32x4 s0[KS / 2], s1[KS / 2], c0[KS / 2], c1[KS / 2];
#pragma unroll
        for (int j = 0; j < KS / 2; ++j) {
          const int64_t o = b * (DH / 2) + j * 32 + lq * 8;
          s0[j] = *reinterpret_cast<const f32x4*>(a.rope_sin + o);
          s1[j] = *reinterpret_cast<const f32x4*>(a.rope_sin + o + 4);
          c0[j] = *reinterpret_cast<const f32x4*>(a.rope_cos + o);
          c1[j] = *reinterpret_cast<const f32x4*>(a.rope_cos + o + 4);
        }
        // three turns of 64 lanes x 16 bytes at a time (one turn set covers G = 4), every load of
        // the set issued before the first sum: a set costs one memory round trip, not one per turn
        const int n4 = (a.G + 2) * (DH / 4);
        constexpr bool planes_first = FUSE == 2;   // (the host checks qkv_ws, qkv_split <= 8 and G <= 4)
        // (called inside each of the two paths below, not behind their join: a use of the
        // oldest loads after a join of paths with different load sequences waits for everything)
        auto take_sincos = [&]() {
#pragma unroll
          for (int j = 0; j < KS / 2; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              sn[j][e] = s0[j][e]; sn[j][4 + e] = s1[j][e];
              cs[j][e] = c0[j][e]; cs[j][4 + e] = c1[j][e];
            }
        };
        auto load_planes = [&](int base, f32x4 (&p)[3][8]) {
#pragma unroll
          for (int tsel = 0; tsel < 3; ++tsel) {
            const int i4 = min(base + tsel * 64 + lane, n4 - 1);
            const int hsel = i4 / (DH / 4), d = (i4 % (DH / 4)) * 4;
            const int head = hsel < a.G ? hkv * a.G + hsel : (hsel == a.G ? a.Hq + hkv : a.Hq + a.Hkv + hkv);
            const int64_t o = rowoff + (int64_t)head * DH + d;
#pragma unroll
            for (int u = 0; u < 8; ++u)
              p[tsel][u] = *reinterpret_cast<const f32x4*>(a.qkv_ws + (int64_t)min(u, a.qkv_split - 1) * plane + o);
          }
        };
        auto sum_planes = [&](int base, const f32x4 (&p)[3][8]) {
#pragma unroll
          for (int tsel = 0; tsel < 3; ++tsel) {
            const int i4 = base + tsel * 64 + lane;
            f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int u = 0; u < 8; ++u)
              if (u < a.qkv_split) acc += p[tsel][u];
            if (i4 < n4) *reinterpret_cast<f32x4*>(&xs[i4 * 4]) = f32x4{rbf(acc[0]), rbf(acc[1]), rbf(acc[2]), rbf(acc[3])};
          }
        };
        if constexpr (planes_first) {
          // the plane set, then the first block of the key / value ring, then the sums:
          // straight-line, so that the wait for the planes counts the ring's loads behind them
          // (the second block of the ring follows once the planes' registers are free: with
          // both in flight next to 24 plane vectors the ring would not get the registers it keeps
          // in the loop, and moving a register that is still being loaded waits for the load)
          f32x4 p[3][8];
          load_planes(0, p);
          __builtin_amdgcn_sched_barrier(0);
          issue_stage(0);
          fetch_query_id();
          __builtin_amdgcn_sched_barrier(0);
          sum_planes(0, p);
          take_sincos();
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int u = 1; u < NS - 1; ++u) issue_stage(u);
          __builtin_amdgcn_sched_barrier(0);
        } else {
          issue_ring();
          fetch_query_id();
          take_sincos();
          for (int i4 = lane; i4 < n4; i4 += 64) {
              const int hsel = i4 / (DH / 4), d = (i4 % (DH / 4)) * 4;
              const int head = hsel < a.G ? hkv * a.G + hsel : (hsel == a.G ? a.Hq + hkv : a.Hq + a.Hkv + hkv);
              const int64_t o = rowoff + (int64_t)head * DH + d;
              f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
              if (a.qkv_ws) {
                for (int z0 = 0; z0 < a.qkv_split; z0 += 8) {
                  f32x4 p[8];
#pragma unroll
                  for (int u = 0; u < 8; ++u)
                    p[u] = *reinterpret_cast<const f32x4*>(a.qkv_ws + (int64_t)min(z0 + u, a.qkv_split - 1) * plane + o);
#pragma unroll
                  for (int u = 0; u < 8; ++u)
                    if (z0 + u < a.qkv_split) acc += p[u];
                }
              } else {
                const u32x2 q = *reinterpret_cast<const u32x2*>(a.qkv + o);
                acc = f32x4{bflo(q[0]), bfhi(q[0]), bflo(q[1]), bfhi(q[1])};
              }
              *reinterpret_cast<f32x4*>(&xs[i4 * 4]) = f32x4{rbf(acc[0]), rbf(acc[1]), rbf(acc[2]), rbf(acc[3])};
          }
        }
        // only this wave reads them: LDS executes a wave's accesses in order, so the staged
        // values only need the compiler to keep the reads behind the writes (a work-group
        // barrier would also wait for the key / value loads in flight)
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      }
      auto fetch8 = [&](int hsel, int d, float (&x)[8]) {
        const f32x4 v0 = *reinterpret_cast<const f32x4*>(&xs[hsel * DH + d]);
        const f32x4 v1 = *reinterpret_cast<const f32x4*>(&xs[hsel * DH + d + 4]);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          x[e] = v0[e];
          x[4 + e] = v1[e];
        }
      };
      // rotate the head whose first column is `col`: pairs (d, d + DH/2) sit in k-steps j, j + KS/2
      auto rotated = [&](int hsel, u32x4 (&dst)[KS]) {
        float x[KS][8];
#pragma unroll
        for (int j = 0; j < KS; ++j) fetch8(hsel, j * 32 + lq * 8, x[j]);
#pragma unroll
        for (int j = 0; j < KS / 2; ++j) {
          float o1[8], o2[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float x1 = x[j][e], x2 = x[j + KS / 2][e];
            o1[e] = rbf(__fsub_rn(__fmul_rn(x1, cs[j][e]), __fmul_rn(x2, sn[j][e])));
            o2[e] = rbf(__fadd_rn(__fmul_rn(x2, cs[j][e]), __fmul_rn(x1, sn[j][e])));
          }
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            dst[j][e] = pack2bf(o1[2 * e], o1[2 * e + 1]);
            dst[j + KS / 2][e] = pack2bf(o2[2 * e], o2[2 * e + 1]);
          }
        }
      };
      if (qvalid) rotated(g, qf);
#pragma unroll
      for (int j = 0; j < KS; ++j) kn[j] = u32x4{0, 0, 0, 0};
#pragma unroll
      for (int h = 0; h < NH; ++h) vn[h] = u32x4{0, 0, 0, 0};
      if (writer) {
        const int64_t slot = ((b * a.Hkv + hkv) * a.S + (col0 % (int)a.S)) * DH;
        if (lm == 0) {   // lanes (0, lq) hold the key as row 0 of an A fragment
          rotated(a.G, kn);
#pragma unroll
          for (int j = 0; j < KS; ++j)
            *reinterpret_cast<u32x4*>(const_cast<uint16_t*>(a.k) + slot + j * 32 + lq * 8) = kn[j];
        }
        if (lq == 0 && 8 * lm < (DH < 128 ? DH : 128)) {   // lanes (lm, 0) hold the value row of key 0
#pragma unroll
          for (int h = 0; h < NH; ++h) {
            float x[8];
            fetch8(a.G + 1, h * 128 + 8 * lm, x);
#pragma unroll
            for (int e = 0; e < 4; ++e) vn[h][e] = pack2bf(x[2 * e], x[2 * e + 1]);
            *reinterpret_cast<u32x4*>(const_cast<uint16_t*>(a.v) + slot + h * 128 + 8 * lm) = vn[h];
          }
        }
      }
#pragma unroll
      for (int j = 0; j < KS; ++j) park[j][lane] = kn[j];
#pragma unroll
      for (int h = 0; h < NH; ++h) park[KS + h][lane] = vn[h];
    }
    if (any) {
      // Whole turns of the ring without a branch inside (an exit in the middle of a turn makes
      // the compiler merge the stages' registers on the exit edges, and a copy of a register
      // that is still being loaded waits for everything in flight), then the last one or two
      // blocks in code of their own: a load of the last block once more, that the turn would make to keep its
      // count, is a block's worth of the memory's time (of two blocks per wave, half as much again).
      const int nblk = ((kb_last - kb0) >> 5) + 1;
      if constexpr (NS == 1) {
        for (int i = 0; i < nblk; ++i) {
          load_block(kb0 + 32 * i, sg[0]);
          __builtin_amdgcn_sched_barrier(0);
          compute_block(kb0 + 32 * i, sg[0]);
        }
      } else {
        static_assert(NS <= 2, "the turns below are of two blocks");
        auto step = [&](int i, Stage& now, Stage& next) {   // computes block i while i + 1 is on its way
          load_block(kb0 + 32 * (i + 1), next);
          __builtin_amdgcn_sched_barrier(0);
          compute_block(kb0 + 32 * i, now);
        };
        int i = 0;
        for (; i + 2 < nblk; i += 2) {
          step(i, sg[0], sg[1]);
          step(i + 1, sg[1], sg[0]);
        }
        if (i + 1 < nblk) {
          step(i, sg[0], sg[1]);
          compute_block(kb0 + 32 * (i + 1), sg[1]);
        } else {
          compute_block(kb0 + 32 * i, sg[0]);
        }
      }
    }
    if (writer && !few) {
      // the step's own key / value as a block of one key (at position col0) from registers
      Stage& one = sg[0];
#pragma unroll
      for (int j = 0; j < KS; ++j) {
        if constexpr (parked) {
          one.kf[0][j] = park[j][lane];
        } else {   // (row 0 of the key fragment)
          one.kf[0][j] = u32x4{0, 0, 0, 0};
          if (lm == 0) one.kf[0][j] = *reinterpret_cast<const u32x4*>(&rot[formed ? a.G * DH + j * 32 + lq * 8 : 0]);
        }
        one.kf[1][j] = u32x4{0, 0, 0, 0};
      }
#pragma unroll
      for (int h = 0; h < NH; ++h) {
#pragma unroll
        for (int sidx = 0; sidx < 8; ++sidx) one.vf[h][sidx] = u32x4{0, 0, 0, 0};
        if constexpr (parked) one.vf[h][0] = park[KS + h][lane];
        else if (lq == 0 && 8 * lm < (DH < 128 ? DH : 128)) one.vf[h][0] = *reinterpret_cast<const u32x4*>(&rot[formed ? (a.G + 1) * DH + h * 128 + 8 * lm : 0]);
      }
      const int own_tok = tok[col0];
#pragma unroll
      for (int sidx = 0; sidx < 8; ++sidx) one.tk[sidx] = own_tok;
      k_lo = min(k_lo, col0);   // (W > 1: a wave's share may lie behind it, with no block in it)
      k_hi = col0;
      key_hi = col0;
      compute_block(col0, one);
    }
  }

  l_run = across_quarters(l_run, [](float x, float y) { return x + y; });

  // O rows are query columns 4*lq + i; columns are d = h*128 + 8*lm + jj.
  const bool dvalid = 8 * lm < (DH < 128 ? DH : 128);
  if constexpr (W > 1) {   // T == 1: the queries are columns 0 .. G - 1
    __shared__ float ml[W][16][2];
    if (lane < 16) {
      ml[wave][lane][0] = m_run;
      ml[wave][lane][1] = l_run;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int n = 4 * lq + i;
      if (n >= a.G || !dvalid) continue;
#pragma unroll
      for (int h = 0; h < NH; ++h)
#pragma unroll
        for (int jj = 0; jj < 8; jj += 4)
          *reinterpret_cast<f32x4*>(&stage[wave][n * DH + h * 128 + 8 * lm + jj]) = f32x4{O[h][jj][i], O[h][jj + 1][i], O[h][jj + 2][i], O[h][jj + 3][i]};
    }
    __syncthreads();
    for (int e = (int)threadIdx.x * 4; e < a.G * DH; e += 64 * W * 4) {
      const int n = e / DH, d = e - n * DH;
      float M = kNegBig, L = 0.f;
#pragma unroll
      for (int w = 0; w < W; ++w)
        if (ml[w][n][1] != 0.f) M = fmaxf(M, ml[w][n][0]);
      f32x4 o = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w = 0; w < W; ++w) {
        const float l = ml[w][n][1], f = __expf(ml[w][n][0] - M);
        if (l != 0.f) {   // (a wave without a key has 0; a NaN is no such wave)
          L += f * l;
          const f32x4 v = *reinterpret_cast<const f32x4*>(&stage[w][e]);
#pragma unroll
          for (int q = 0; q < 4; ++q) o[q] += f * v[q];
        }
      }
      const int64_t qv = b * a.Hq + hkv * a.G + n;
      if (a.n_chunks == 1) {
        const float inv = L > 0.f ? 1.0f / L : 0.f;
        *reinterpret_cast<u32x2*>(a.out + qv * DH + d) = u32x2{pack2bf(o[0] * inv, o[1] * inv), pack2bf(o[2] * inv, o[3] * inv)};
      } else {
        float* p = a.ws + (qv * a.n_chunks + chunk) * (DH + kPartPad);
        if (d == 0) {
          p[0] = M;
          p[1] = L;
        }
        *reinterpret_cast<f32x4*>(p + kPartPad + d) = o;
      }
    }
    return;
  }
  if (a.kv_chunk <= 0 || a.n_chunks == 1) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int n = 4 * lq + i;
      const float l = __shfl(l_run, n, 64);
      const int gi = n & (a.Gp - 1), ti = qt * PT + (n >> a.gp_shift);
      if (!(gi < a.G && ti < a.T && ti >= start) || !dvalid) continue;
      const float inv = l > 0.f ? 1.0f / l : 0.f;
      uint16_t* o = a.out + ((row0 + ti) * a.Hq + hkv * a.G + gi) * DH;
#pragma unroll
      for (int h = 0; h < NH; ++h) {
        u32x4 w;
#pragma unroll
        for (int r = 0; r < 4; ++r)
          w[r] = pack2bf(O[h][2 * r][i] * inv, O[h][2 * r + 1][i] * inv);
        *reinterpret_cast<u32x4*>(o + h * 128 + 8 * lm) = w;
      }
    }
    return;
  }
  // split: partial (m, l, O[dh]) per (query vector, chunk)
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int n = 4 * lq + i;
    const float l = __shfl(l_run, n, 64);
    const float m = __shfl(m_run, n, 64);
    const int gi = n & (a.Gp - 1), ti = qt * PT + (n >> a.gp_shift);
    if (!(gi < a.G && ti < a.T)) continue;
    const int64_t qv = (b * a.T + ti) * a.Hq + hkv * a.G + gi;
    float* p = a.ws + (qv * a.n_chunks + chunk) * (DH + kPartPad);
    if (lm == 0) {
      p[0] = m;
      p[1] = l;
    }
    if (!dvalid || l <= 0.f) continue;
#pragma unroll
    for (int h = 0; h < NH; ++h)
#pragma unroll
      for (int jj = 0; jj < 8; jj += 4)
        *reinterpret_cast<f32x4*>(p + kPartPad + h * 128 + 8 * lm + jj) = f32x4{O[h][jj][i], O[h][jj + 1][i], O[h][jj + 2][i], O[h][jj + 3][i]};
  }
}

template <int DH, int FUSE, bool TOKVEC, int W>
__global__ __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(DH > 128 || W > 1 ? 2 : 1, DH > 128 || W > 1 ? 2 : 1))) void attn_kernel(const AttnArgs a) {
  attn_body<DH, FUSE, TOKVEC, W>(a, RopeArgs{});
}
// Norms, rotation, the cache write and attention of a decode step in one launch: what it saves is the other one's gap and its trip through memory.
// With the o adapter behind, us in two | one, 32 heads of 128 on 4, 160 keys: 1 row 12.9 | 12.7, 64 rows 16.1 | 14.8, 128 rows 21.7 | 19.0, 1000
// keys 16 rows 18.6 | 18.6, 64 rows 33.2 | 31.8; 8 heads of 64 on 2: 1 row of 48 keys 10.2 | 9.1, 128 rows of 100 11.7 | 10.8.
template <int DH, bool TOKVEC, bool FEW>
__global__ __launch_bounds__(64 * kAttnWaves) __attribute__((amdgpu_waves_per_eu(2, 2))) void attn_rope_kernel(const AttnArgs a, const RopeArgs r) {
  attn_body<DH, FEW ? 4 : 3, TOKVEC, kAttnWaves>(a, r);
}

// Many query positions per row (prefill, whole-sequence log-probability passes): the wave above
// loads 16 KB of keys and values per 32-key block for sixteen MFMAs, i.e. it runs at what a
// compute unit can draw from L2, not at its matrix rate.  This form gives one wave QW
// consecutive query tiles: every loaded block, and the in-lane transposition of its value rows,
// serves QW x 16 query columns.  Each tile sees the same 32-key blocks in the same order with
// the same arithmetic as it would in a wave of its own (a block wholly before a tile's window
// or after its causal limit leaves its running maximum, sum and output untouched: p = 0,
// alpha = exp(0)), so results are bit-identical to the kernel above.  No fused rotation, no key
// split (those are decode modes).
template <int DH, bool TOKVEC, int QW>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(1, 1))) void attn_tiles_kernel(const AttnArgs a) {
  constexpr int KS = DH / 32;
  constexpr int NH = DH > 128 ? DH / 128 : 1;
  constexpr int NS = 2;
  const int lane = threadIdx.x, lm = lane & 15, lq = lane >> 4;
  const int hkv = blockIdx.y;
  const int PT = 16 >> a.gp_shift;
  const unsigned bz = blockIdx.z;
  const int64_t b = bz / a.QTG;
  // (the longest tiles of a row are handed out first: a tile's work grows with its position)
  const int qt0 = ((int)a.QTG - 1 - (int)(bz - (unsigned)b * a.QTG)) * QW;
  const int start = a.rows.base ? a.rows.starts[b] : 0;
  const int64_t row0 = a.rows.base ? a.rows.base[b] : b * a.T;   // a row's position 0
  if ((qt0 + QW) * PT <= start) return;
  const int col0 = *a.col_ptr;
  const int g = lm & (a.Gp - 1);

  int c_n[QW], lo_n[QW];
  bool qvalid[QW];
  u32x4 qf[QW][KS];
#pragma unroll
  for (int w = 0; w < QW; ++w) {
    const int tq = (qt0 + w) * PT + (lm >> a.gp_shift);
    qvalid[w] = g < a.G && tq < a.T && tq >= start;
    c_n[w] = col0 + tq;
    lo_n[w] = a.window > 0 ? max(0, c_n[w] - a.window + 1) : 0;
    const int64_t qvec = (row0 + (qvalid[w] ? tq : a.T - 1)) * a.Hq + hkv * a.G + (qvalid[w] ? g : 0);
#pragma unroll
    for (int j = 0; j < KS; ++j) {
      qf[w][j] = u32x4{0, 0, 0, 0};
      if (qvalid[w]) qf[w][j] = *reinterpret_cast<const u32x4*>(a.q + qvec * DH + j * 32 + lq * 8);
    }
  }
  // key range of the QW tiles together
  const int t_last = min((int)a.T - 1, (qt0 + QW) * PT - 1);
  const int k_hi = col0 + t_last;
  const int k_lo = max(start, a.window > 0 ? col0 + qt0 * PT - a.window + 1 : 0);

  f32x4 O[QW][NH][8];
  float m_run[QW], l_run[QW];
#pragma unroll
  for (int w = 0; w < QW; ++w) {
    m_run[w] = kNegBig;
    l_run[w] = 0.f;
#pragma unroll
    for (int h = 0; h < NH; ++h)
#pragma unroll
      for (int jj = 0; jj < 8; ++jj) O[w][h][jj] = f32x4{0.f, 0.f, 0.f, 0.f};
  }

  const uint16_t* kbase = a.k + ((b * a.Hkv + hkv) * a.S) * DH;
  const uint16_t* vbase = a.v + ((b * a.Hkv + hkv) * a.S) * DH;
  const int32_t* tok = a.tokens + b * a.tok_ld;
  int32_t id_ref[QW];
  const bool id_equal = a.seg_mode != 0;
  const int vcol = (8 * lm) % (DH < 128 ? DH : 128);
  struct Stage {
    u32x4 kf[2][KS];
    u32x4 vf[NH][8];
    int tk[8];
  };
  const uint32_t slab_bytes = (uint32_t)a.S * DH * 2u;
  const rsrc_t rk = make_rsrc(kbase, slab_bytes), rv = make_rsrc(vbase, slab_bytes);
  const rsrc_t rtok = make_rsrc(tok, (uint64_t)min(a.S, a.tok_ld) * 4);
  const uint32_t koff = (uint32_t)(lm * DH + lq * 8) * 2u;
  const uint32_t voff = (uint32_t)(4 * lq * DH + vcol) * 2u;
  // (the blocks are re-read by the waves of the later tiles of this row: default cache policy)
  auto load_block = [&](int kb, Stage& sg) {
    const uint32_t kb_bytes = (uint32_t)kb * (DH * 2u);
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
      const uint32_t o = koff + kb_bytes + (uint32_t)(tt * 16 * DH * 2);
#pragma unroll
      for (int j = 0; j < KS; ++j) sg.kf[tt][j] = __builtin_amdgcn_raw_buffer_load_b128(rk, o + (uint32_t)(j * 64), 0, 0);
    }
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      const uint32_t o = voff + kb_bytes + (uint32_t)(((s < 4 ? s : 12 + s)) * DH * 2);
#pragma unroll
      for (int h = 0; h < NH; ++h) sg.vf[h][s] = __builtin_amdgcn_raw_buffer_load_b128(rv, o + (uint32_t)(h * 256), 0, 0);
    }
    if constexpr (TOKVEC) {
      const u32x4 t0 = __builtin_amdgcn_raw_buffer_load_b128(rtok, (uint32_t)(kb + 4 * lq) * 4u, 0, 0);
      const u32x4 t1 = __builtin_amdgcn_raw_buffer_load_b128(rtok, (uint32_t)(kb + 16 + 4 * lq) * 4u, 0, 0);
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        sg.tk[s] = (int)t0[s];
        sg.tk[4 + s] = (int)t1[s];
      }
    } else {
#pragma unroll
      for (int s = 0; s < 8; ++s)
        sg.tk[s] = (int)__builtin_amdgcn_raw_buffer_load_b32(
            rtok, (uint32_t)(kb + (s < 4 ? 4 * lq + s : 16 + 4 * lq + (s - 4))) * 4u, 0, 0);
    }
  };
  auto compute_block = [&](int kb, const Stage& sg) {
    u32x4 pa[QW];
#pragma unroll
    for (int w = 0; w < QW; ++w) {
      bool kvalid[8];
#pragma unroll
      for (int s = 0; s < 8; ++s) {
        const int key = kb + (s < 4 ? 4 * lq + s : 16 + 4 * lq + (s - 4));
        kvalid[s] = qvalid[w] && key >= max(k_lo, lo_n[w]) && key <= min(k_hi, c_n[w]) &&
                    ((sg.tk[s] == id_ref[w]) == id_equal);
      }
      f32x4 st[2];
#pragma unroll
      for (int tt = 0; tt < 2; ++tt) {
        st[tt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < KS; ++j) st[tt] = mfma16(sg.kf[tt][j], qf[w][j], st[tt]);
      }
      float sv[8];
      float bmax = kNegBig;
#pragma unroll
      for (int s = 0; s < 8; ++s) {
        float x = rbf(st[s >> 2][s & 3]);
        if (a.scale_bf != 0.f) x = rbf(x * a.scale_bf);
        sv[s] = x;
        if (kvalid[s]) bmax = fmaxf(bmax, x);
      }
      bmax = fmaxf(bmax, lane_xor(bmax, 16));
      bmax = fmaxf(bmax, lane_xor(bmax, 32));
      const float m_new = fmaxf(m_run[w], bmax);
      const float alpha = __expf(m_run[w] - m_new);
      m_run[w] = m_new;
      float p[8], psum = 0.f;
#pragma unroll
      for (int s = 0; s < 8; ++s) {
        p[s] = kvalid[s] ? __expf(sv[s] - m_new) : 0.f;
        psum += p[s];
      }
      l_run[w] = l_run[w] * alpha + psum;
      pa[w][0] = pack2bf(p[0], p[1]);
      pa[w][1] = pack2bf(p[2], p[3]);
      pa[w][2] = pack2bf(p[4], p[5]);
      pa[w][3] = pack2bf(p[6], p[7]);
      if (__builtin_amdgcn_ballot_w64(alpha != 1.0f) != 0) {
        float ar[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) ar[i] = __shfl(alpha, 4 * lq + i, 64);
#pragma unroll
        for (int h = 0; h < NH; ++h)
#pragma unroll
          for (int jj = 0; jj < 8; ++jj)
#pragma unroll
            for (int i = 0; i < 4; ++i) O[w][h][jj][i] *= ar[i];
      }
    }
    // O += P . V: a value fragment is transposed once and multiplied with every tile's P
#pragma unroll
    for (int h = 0; h < NH; ++h)
#pragma unroll
      for (int jj = 0; jj < 8; ++jj) {
        const uint32_t sel = (jj & 1) ? 0x07060302u : 0x05040100u;
        u32x4 bfrag;
#pragma unroll
        for (int r = 0; r < 4; ++r)
          bfrag[r] = __builtin_amdgcn_perm(sg.vf[h][2 * r + 1][jj >> 1], sg.vf[h][2 * r][jj >> 1], sel);
#pragma unroll
        for (int w = 0; w < QW; ++w) O[w][h][jj] = mfma16(pa[w], bfrag, O[w][h][jj]);
      }
  };
  {
    Stage sg[NS];
    const int kb0 = k_lo & ~31;
    const int kb_last = k_hi & ~31;
    const bool any = kb0 <= k_hi;
#pragma unroll
    for (int u = 0; u < NS - 1; ++u) load_block(min(kb0 + 32 * u, kb_last), sg[u]);
#pragma unroll
    for (int w = 0; w < QW; ++w) {
      const int32_t id_q = tok[min((int64_t)c_n[w], a.tok_ld - 1)];
      id_ref[w] = a.seg_mode ? id_q : a.pad_id;
    }
    if (any) {
      const int nblk = ((kb_last - kb0) >> 5) + 1;
      int i = 0;
      for (; i + NS <= nblk; i += NS) {
#pragma unroll
        for (int u = 0; u < NS; ++u) {
          const int kbu = kb0 + 32 * (i + u);
          load_block(min(kbu + 32 * (NS - 1), kb_last), sg[(u + NS - 1) % NS]);
          __builtin_amdgcn_sched_barrier(0);
          compute_block(kbu, sg[u]);
        }
      }
#pragma unroll
      for (int u = 0; u < NS - 1; ++u)
        if (i + u < nblk) compute_block(kb0 + 32 * (i + u), sg[u]);
    }
  }
  const bool dvalid = 8 * lm < (DH < 128 ? DH : 128);
#pragma unroll
  for (int w = 0; w < QW; ++w) {
    float lr = l_run[w];
    lr += lane_xor(lr, 16);
    lr += lane_xor(lr, 32);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int n = 4 * lq + i;
      const float l = __shfl(lr, n, 64);
      const int gi = n & (a.Gp - 1), ti = (qt0 + w) * PT + (n >> a.gp_shift);
      if (!(gi < a.G && ti < a.T && ti >= start) || !dvalid) continue;
      const float inv = l > 0.f ? 1.0f / l : 0.f;
      uint16_t* o = a.out + ((row0 + ti) * a.Hq + hkv * a.G + gi) * DH;
#pragma unroll
      for (int h = 0; h < NH; ++h) {
        u32x4 wv;
#pragma unroll
        for (int r = 0; r < 4; ++r)
          wv[r] = pack2bf(O[w][h][2 * r][i] * inv, O[w][h][2 * r + 1][i] * inv);
        *reinterpret_cast<u32x4*>(o + h * 128 + 8 * lm) = wv;
      }
    }
  }
}

// The same for head_dim 128 and 256 with keys and values staged through LDS: a work-group of four waves
// takes 4 x QW consecutive query tiles of one (row, kv head), and every 32-key block is requested
// once per work-group straight into LDS (16 bytes per lane, key rows with their 16-byte chunks
// XOR-swizzled by row so that the fragment reads of 16 rows hit 16 bank groups, value rows by pairs of chunks, which the transposing
// reads take whole; the block's 32 token / segment ids next to them, by the dword: rows of ids need no alignment),
// the next blocks in flight.  Every wave computes exactly the blocks attn_tiles_kernel would give it, in the same order
// with the same arithmetic: outputs are bit-identical.
//
// What bounds it is vector work and the waits between its steps: per score 11 lane-instructions in the straight line of the loop
// (two roundings to bf16 with a scale between them, maximum, exponential, sum, rounding of P; 9 without a scale), 16.7 by counters with masks, rescaling,
// addresses and the two matrix instructions (2 x 6144 positions: the vector unit at work for 72 % of the cycles, the matrix pipe for 32 %).  So the tiles of a wave run through one straight line of
// code, whose chains hide each other's latency, with two such work-groups per compute unit; the values leave LDS transposed
// (ds_read_tr: no packing of rows by the vector unit); maxima cross the lanes in registers (permlane swaps) instead of through LDS; O is kept
// transposed (P.V formed as V^T . P^T: the same operand registers with the operands exchanged), so that a query's rescaling
// factor is already in the lanes that need it; the ids of a block are tested by one read and one ballot, and read key by key only where one
// differs; and head_dim 128 meets at a barrier every second block.
// 32 heads of 128 over 8 kv heads, us before (values rounded in pairs by the vector unit, a barrier per block) and now:
//   2 x 6144 positions 895 -> 826 (691 -> 750 TFLOP/s)   3 x 2900: 337 -> 311   13 x 1024: 221 -> 208   7 x 1023 over 4: 135 -> 132
//   (3 x 2900 inside a pass, under the clock that its GEMMs leave: 434 -> 377 to 407)
//   64 x 256: 119.5 -> 119.5   16 x 128: 16.3 -> 15.6    head_dim 256, 4 heads over 1: 3 x 3000 135 -> 116, 64 x 256 40.8 -> 39.2
// Two blocks in one line of code (both blocks' scores, then both softmaxes, then both blocks' values): 1030 for the first.
typedef uint32_t __attribute__((address_space(3))) lds_word_t;
typedef u32x4 __attribute__((address_space(3))) lds_vec_t;
__device__ __forceinline__ u32x4 attn_lds128(uint32_t addr) {
  return *reinterpret_cast<const lds_vec_t*>(static_cast<uintptr_t>(addr));
}
__device__ __forceinline__ uint32_t attn_lds32(uint32_t addr) { return *reinterpret_cast<const lds_word_t*>(static_cast<uintptr_t>(addr)); }
// Of each 16 lanes, which point at four rows of 16 16-bit elements, 8 bytes a lane (row lane / 4, elements 4 (lane % 4) ..), lane i gets element i of
// the four rows.
typedef short s16x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ u32x2 attn_lds_tr16(uint32_t addr) {
  return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                       (__attribute__((address_space(3))) s16x4*)static_cast<uintptr_t>(addr)));
}
// Maxima of numbers that no operation left as signalling NaNs (fmaxf quiets each operand first, an instruction more).  What a permlane swap reads
// of them is a copy and its source, at least the copy and the distance that the compiler keeps behind it away.
__device__ __forceinline__ float max_plain(float x, float y) {
  float d;
  asm("v_max_f32 %0, %1, %2" : "=v"(d) : "v"(x), "v"(y));
  return d;
}
__device__ __forceinline__ float max3_plain(float x, float y, float z) {
  float d;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(d) : "v"(x), "v"(y), "v"(z));
  return d;
}
// four bytes per lane straight into LDS, at `lds` + 4 * lane (as dma16 of gemm_tile.h)
__device__ __forceinline__ void dma4(uint32_t lds, const u32x4& r, uint32_t voff) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 3\n\tbuffer_load_dword %1, %2, 0 offen lds" ::"s"(lds), "v"(voff), "s"(r) : "memory", "m0");
}
// 32 keys, 32 values, ids
constexpr uint32_t wg_stage_bytes(int dh) { return 32u * (uint32_t)dh * 2u * 2u + 256u; }
// Blocks in LDS, half of them computed and half in flight; what two work-groups per compute unit have room for.
constexpr int wg_stages(int dh) { return dh > 128 ? 2 : 4; }
// Query tiles of a wave: O and the queries of two at head_dim 256 leave room for one wave per SIMD only, and a wave alone does not cover its own
// softmax.
constexpr int wg_tiles_per_wave(int dh) { return dh > 128 ? 1 : 2; }
template <int DH, bool SCALED>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void attn_wg_kernel(const AttnArgs a) {
  constexpr int KS = DH / 32, NH = DH / 128, QW = wg_tiles_per_wave(DH), kWgStages = wg_stages(DH);
  constexpr uint32_t kWgStageBytes = wg_stage_bytes(DH), ROW = DH * 2, PASSES = DH / 64, VAT = 32 * ROW, IAT = 64 * ROW;
  extern __shared__ __align__(16) unsigned char smem_a[];
  const uint32_t lds0 = lds_addr(smem_a);
  const int tid = threadIdx.x, lane = tid & 63, lm = lane & 15, lq = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hkv = blockIdx.y;
  const int PT = 16 >> a.gp_shift;
  const unsigned bz = blockIdx.z;
  const int64_t b = bz / a.QTG;
  // (the longest groups of a row are handed out first: a tile's work grows with its position)
  const int qt_wg = ((int)a.QTG - 1 - (int)(bz - (unsigned)b * a.QTG)) * (4 * QW);
  const int qt0 = qt_wg + wave * QW;
  const int start = a.rows.base ? a.rows.starts[b] : 0;
  const int64_t row0 = a.rows.base ? a.rows.base[b] : b * a.T;   // a row's position 0
  if ((qt_wg + 4 * QW) * PT <= start) return;                   // (the whole work-group)
  const int col0 = *a.col_ptr;
  const int g = lm & (a.Gp - 1);

  int c_n[QW], lo_n[QW];
  bool qvalid[QW];
  u32x4 qf[QW][KS];
#pragma unroll
  for (int w = 0; w < QW; ++w) {
    const int tq = (qt0 + w) * PT + (lm >> a.gp_shift);
    qvalid[w] = g < a.G && tq < a.T && tq >= start;
    c_n[w] = col0 + tq;
    lo_n[w] = a.window > 0 ? max(0, c_n[w] - a.window + 1) : 0;
    const int64_t qvec = (row0 + (qvalid[w] ? tq : a.T - 1)) * a.Hq + hkv * a.G + (qvalid[w] ? g : 0);
#pragma unroll
    for (int j = 0; j < KS; ++j) {
      qf[w][j] = u32x4{0, 0, 0, 0};
      if (qvalid[w]) qf[w][j] = *reinterpret_cast<const u32x4*>(a.q + qvec * DH + j * 32 + lq * 8);
    }
  }
  // key range of this wave's QW tiles (as in attn_tiles_kernel) and of the work-group's 4 QW
  const bool wave_live = qt0 * PT < a.T && (qt0 + QW) * PT > start;
  const int k_hi = col0 + min((int)a.T - 1, (qt0 + QW) * PT - 1);
  const int k_lo = max(start, a.window > 0 ? col0 + qt0 * PT - a.window + 1 : 0);
  const int k_hi_wg = col0 + min((int)a.T - 1, (qt_wg + 4 * QW) * PT - 1);
  const int k_lo_wg = max(start, a.window > 0 ? col0 + qt_wg * PT - a.window + 1 : 0);
  const int kb0_wg = k_lo_wg & ~31;
  const int nblk_wg = (((k_hi_wg & ~31) - kb0_wg) >> 5) + 1;
  const int kb0 = k_lo & ~31, kb_last = k_hi & ~31;
  const bool any = wave_live && kb0 <= k_hi;

  // O^T: lane (query lm, quarter lq) holds dimensions 128 h + 16 jj + 4 lq + i in O[w][8 h + jj][i]
  f32x4 O[QW][8 * NH];
  float m_run[QW], l_run[QW];
#pragma unroll
  for (int w = 0; w < QW; ++w) {
    m_run[w] = kNegBig;
    l_run[w] = 0.f;
#pragma unroll
    for (int jj = 0; jj < 8 * NH; ++jj) O[w][jj] = f32x4{0.f, 0.f, 0.f, 0.f};
  }

  const uint16_t* kbase = a.k + ((b * a.Hkv + hkv) * a.S) * DH;
  const uint16_t* vbase = a.v + ((b * a.Hkv + hkv) * a.S) * DH;
  const int32_t* tok = a.tokens + b * a.tok_ld;
  const bool id_equal = a.seg_mode != 0;
  int32_t id_ref[QW];
#pragma unroll
  for (int w = 0; w < QW; ++w) {
    const int32_t id_q = tok[min((int64_t)c_n[w], a.tok_ld - 1)];
    id_ref[w] = a.seg_mode ? id_q : a.pad_id;
  }
  // A block that lies wholly inside every query's range of all tiles, with no id to mask, takes the
  // same arithmetic without the per-key tests: the bounds of that, uniform over the wave.  In a packed batch the
  // ids that allow it are those of one segment that all queries of the wave belong to.
  int lo_max = -0x7fffffff, hi_min = 0x7fffffff;
  bool full = true;
  const int32_t one_id = __builtin_amdgcn_readfirstlane(id_ref[0]);
#pragma unroll
  for (int w = 0; w < QW; ++w) {
    lo_max = max(lo_max, max(k_lo, lo_n[w]));
    hi_min = min(hi_min, min(k_hi, c_n[w]));
    full = full && __builtin_amdgcn_ballot_w64(qvalid[w] && id_ref[w] == one_id) == ~0ull;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    lo_max = max(lo_max, lane_xor(lo_max, o));
    hi_min = min(hi_min, lane_xor(hi_min, o));
  }
  lo_max = __builtin_amdgcn_readfirstlane(full ? lo_max : 0x7fffffff);
  hi_min = __builtin_amdgcn_readfirstlane(hi_min);
  const uint32_t slab_bytes = (uint32_t)a.S * DH * 2u;
  const u32x4 rk = raw_rsrc(kbase, slab_bytes), rv = raw_rsrc(vbase, slab_bytes);
  const u32x4 rtok = raw_rsrc(tok, (uint64_t)min(a.S, a.tok_ld) * 4);
  // thread t requests, per 4 KB pass over a block (16 rows | 8), the 16 bytes that land at byte 16 t of the pass:
  // row t / 16 | t / 32, and of the key row the chunk (t % 16 | t % 32) ^ (row % 16), of the value row the one whose pair of chunks is that of
  // this place ^ (row % 8)
  constexpr int CH = DH / 8;   // chunks of a row
  const uint32_t krow = (uint32_t)(tid / CH);
  const uint32_t kreq = krow * ROW + ((uint32_t)(tid % CH) ^ krow) * 16u;
  const uint32_t vreq = krow * ROW + ((uint32_t)(tid % CH) ^ ((krow & 7u) * 2u)) * 16u;
  auto request_block = [&](int i) {   // (the ids by every wave: the same bytes)
    const uint32_t base = lds0 + (uint32_t)(i % kWgStages) * kWgStageBytes + (uint32_t)wave * 1024u;
    const uint32_t kb_bytes = (uint32_t)(kb0_wg + 32 * i) * ROW;
#pragma unroll
    for (uint32_t c = 0; c < PASSES; ++c) {   // (rows 8 .. 15 of a block of 512-byte rows come with the odd passes)
      dma16(base + c * 4096u, rk, kb_bytes + c * 4096u + (DH > 128 ? kreq ^ ((c & 1u) * 128u) : kreq), 0);
      dma16(base + VAT + c * 4096u, rv, kb_bytes + c * 4096u + vreq, 0);
    }
    // ids kb .. kb + 63 (the block's 32 and whatever follows them; past the row: zeros)
    dma4(lds0 + (uint32_t)(i % kWgStages) * kWgStageBytes + IAT, rtok, (uint32_t)(kb0_wg + 32 * i + lane) * 4u);
  };
  // this lane's places in a stage: key row lm (+ 16 tt), chunk 4 j + lq; value row 4 lq + lm / 4 (+ 16 tt), 8 bytes lm % 4 of dimensions 16 jj (+ 128 h)
  // .. + 16, jj under XOR; ids 4 lq, and of key lane % 32
  uint32_t kat[KS];
#pragma unroll
  for (int j = 0; j < KS; ++j) kat[j] = (uint32_t)lm * ROW + (((uint32_t)(j * 4 + lq) ^ (uint32_t)lm) * 16u);
  const uint32_t vrow = (uint32_t)(4 * lq + (lm >> 2));
  const uint32_t vat = VAT + vrow * ROW + (vrow & 7u) * 32u + (uint32_t)(lm & 3) * 8u, iat = IAT + (uint32_t)(lq * 16);
  const uint32_t one_at = IAT + (uint32_t)(lane & 31) * 4u;
  auto compute_block = [&](int kb, uint32_t base) {
    u32x4 kf[2][KS];
#pragma unroll
    for (int j = 0; j < KS; ++j) {
      const uint32_t at = base + kat[j];
#pragma unroll
      for (int tt = 0; tt < 2; ++tt) kf[tt][j] = attn_lds128(at + (uint32_t)tt * (16u * ROW));
    }
    // (pad mode: a key counts when its id differs from pad_id; packed: when it is the query's)
    const bool inside = kb >= lo_max && kb + 31 <= hi_min &&
                        __builtin_amdgcn_ballot_w64(((int)attn_lds32(base + one_at) == one_id) == id_equal) == ~0ull;
    f32x4 st[QW][2];
#pragma unroll
    for (int w = 0; w < QW; ++w)
#pragma unroll
      for (int tt = 0; tt < 2; ++tt) st[w][tt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < KS; ++j)
#pragma unroll
      for (int w = 0; w < QW; ++w)
#pragma unroll
        for (int tt = 0; tt < 2; ++tt) st[w][tt] = mfma16(kf[tt][j], qf[w][j], st[w][tt]);
    float sv[QW][8], alpha[QW];
#pragma unroll
    for (int w = 0; w < QW; ++w)
#pragma unroll
      for (int s = 0; s < 8; s += 2) {
        uint32_t u = cvt_pk_bf16(st[w][s >> 2][s & 3], st[w][s >> 2][(s & 3) + 1]);
        if constexpr (SCALED) u = cvt_pk_bf16(bflo(u) * a.scale_bf, bfhi(u) * a.scale_bf);
        sv[w][s] = bflo(u);
        sv[w][s + 1] = bfhi(u);
      }
    if (!inside) {
      asm volatile("");   // (a branch, not selects in every block)
      const u32x4 t0 = attn_lds128(base + iat), t1 = attn_lds128(base + iat + 64u);
#pragma unroll
      for (int w = 0; w < QW; ++w)
#pragma unroll
        for (int s = 0; s < 8; ++s) {
          const int key = kb + (s < 4 ? 4 * lq + s : 16 + 4 * lq + (s - 4));
          const int id = s < 4 ? (int)t0[s & 3] : (int)t1[s & 3];
          const bool ok = qvalid[w] & (key >= max(k_lo, lo_n[w])) & (key <= min(k_hi, c_n[w])) & ((id == id_ref[w]) == id_equal);
          sv[w][s] = ok ? sv[w][s] : -__builtin_inff();
        }
    }
    bool moved = false;
    u32x4 pa[QW];
#pragma unroll
    for (int w = 0; w < QW; ++w) {
      const float m_blk = max3_plain(max3_plain(sv[w][0], sv[w][1], sv[w][2]), max3_plain(sv[w][3], sv[w][4], sv[w][5]), max_plain(sv[w][6], sv[w][7]));
      const float m_new = max_plain(m_run[w], across_quarters(m_blk, [](float x, float y) { return max_plain(x, y); }));
      alpha[w] = __expf(m_run[w] - m_new);
      moved = moved || alpha[w] != 1.0f;
      m_run[w] = m_new;
      float p[8], psum = 0.f;
#pragma unroll
      for (int s = 0; s < 8; ++s) {
        p[s] = __expf(sv[w][s] - m_new);   // (a masked key: exp(-inf) = 0)
        psum += p[s];
      }
      l_run[w] = l_run[w] * alpha[w] + psum;
#pragma unroll
      for (int e = 0; e < 4; ++e) pa[w][e] = cvt_pk_bf16(p[2 * e], p[2 * e + 1]);
    }
    // the running maximum settles after a few blocks: rescale O only when some column moved
    if (__builtin_amdgcn_ballot_w64(moved) != 0) {
#pragma unroll
      for (int w = 0; w < QW; ++w)
#pragma unroll
        for (int jj = 0; jj < 8 * NH; ++jj)
#pragma unroll
          for (int i = 0; i < 4; ++i) O[w][jj][i] *= alpha[w];
    }
    // value fragments come out of LDS transposed, once for all tiles: four keys of a dimension per lane and read
#pragma unroll
    for (int h = 0; h < NH; ++h)
#pragma unroll
      for (int jj = 0; jj < 8; ++jj) {
        const uint32_t at = ((base + vat) ^ (uint32_t)(jj * 32)) + (uint32_t)h * 256u;
        const u32x2 v0 = attn_lds_tr16(at), v1 = attn_lds_tr16(at + 16u * ROW);
        const u32x4 vt = {v0[0], v0[1], v1[0], v1[1]};
#pragma unroll
        for (int w = 0; w < QW; ++w) O[w][8 * h + jj] = mfma16(vt, pa[w], O[w][8 * h + jj]);
      }
  };
  // BATCH blocks behind a barrier; the next ones are on their way meanwhile, into the stages that the ones before were read from.  (A barrier per
  // block: 828 us instead of 815 for 2 x 6144 positions, the rest alike.)
  constexpr int BATCH = kWgStages / 2;
#pragma unroll
  for (int u = 0; u < BATCH; ++u)
    if (u < nblk_wg) request_block(u);
  for (int i = 0; i < nblk_wg; i += BATCH) {
    tnx_wait_vm(0);     // this wave's share of the blocks has landed ...
    __syncthreads();    // ... and everyone's; every wave is also done reading the blocks before
#pragma unroll
    for (int u = 0; u < BATCH; ++u)
      if (i + BATCH + u < nblk_wg) request_block(i + BATCH + u);
#pragma unroll
    for (int u = 0; u < BATCH; ++u) {
      const int kb = kb0_wg + 32 * (i + u);
      if (any && kb >= kb0 && kb <= kb_last) compute_block(kb, lds0 + (uint32_t)((i + u) % kWgStages) * kWgStageBytes);
    }
  }
#pragma unroll
  for (int w = 0; w < QW; ++w) {
    const float l = across_quarters(l_run[w], [](float x, float y) { return x + y; });
    const int ti = (qt0 + w) * PT + (lm >> a.gp_shift);
    if (!qvalid[w]) continue;
    const float inv = l > 0.f ? 1.0f / l : 0.f;
    uint16_t* o = a.out + ((row0 + ti) * a.Hq + hkv * a.G + g) * DH + 4 * lq;
#pragma unroll
    for (int jj = 0; jj < 8 * NH; ++jj)
      *reinterpret_cast<u32x2*>(o + 16 * jj) = u32x2{pack2bf(O[w][jj][0] * inv, O[w][jj][1] * inv), pack2bf(O[w][jj][2] * inv, O[w][jj][3] * inv)};
  }
}

// out[qv, d] = bf16( sum_c e^{m_c - M} O_c[d] / sum_c e^{m_c - M} l_c )
// The (m, l) pairs of all chunks are fetched at once into LDS (one round trip instead of one
// dependent load per chunk and pass); every thread then forms M, the weights and the sums in
// chunk order, with its chunk outputs fetched eight at a time.  (Chunks without a key have
// l = 0 and an O nobody wrote: selected away, never multiplied.  l is a sum of exponentials: 0, positive, or the NaN of a
// query or a key, which has to reach the output.)
__global__ void attn_combine_kernel(const float* ws, int64_t n_qvec, int dh, int n_chunks,
                                    uint16_t* out) {
  extern __shared__ float ml[];   // [n_chunks][2]
  const int64_t qv = blockIdx.x;
  const int d = threadIdx.x;
  const float* p = ws + qv * n_chunks * (dh + kPartPad);
  for (int i = d; i < 2 * n_chunks; i += blockDim.x) ml[i] = p[(i >> 1) * (dh + kPartPad) + (i & 1)];
  __syncthreads();
  if (d >= dh) return;
  float M = kNegBig;
  for (int c = 0; c < n_chunks; ++c)
    if (ml[2 * c + 1] != 0.f) M = fmaxf(M, ml[2 * c]);
  float L = 0.f, o = 0.f;
  for (int c0 = 0; c0 < n_chunks; c0 += 8) {
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = p[min(c0 + u, n_chunks - 1) * (dh + kPartPad) + kPartPad + d];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int c = c0 + u;
      if (c < n_chunks) {
        const float l = ml[2 * c + 1];
        if (l != 0.f) {
          const float w = __expf(ml[2 * c] - M);
          L += w * l;
          o += w * v[u];
        }
      }
    }
  }
  out[qv * dh + d] = f2bf(L != 0.f ? o / L : 0.f);
}

// The same over whole rows of heads, with the LoRA down-projection of the row behind it (row_adapter.h); the first group of adapter columns
// writes the row.  The chunks' (max, sum) pairs of all heads go to LDS; a thread asks for its first eight
// chunks' outputs and its first columns of A ahead of them.
template <int MAXC, int NB, int NCH>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 2))) void attn_combine_lora_kernel(const float* ws, int64_t M, int heads, int dh, int n_chunks, uint16_t* out,
                                                                const RowAdapterArgs g) {
  extern __shared__ float ml[];   // [heads][n_chunks][2]
  __shared__ float sums[4 * NB];
  int group;
  int64_t row;
  if (!row_adapter_place(g, M, group, row)) return;
  const int K = heads * dh, pitch = dh + kPartPad;
  const float* base = ws + row * (int64_t)heads * n_chunks * pitch;
  RowAdapter<MAXC, NB> ad;
  const float* p[MAXC];
  int at[MAXC];
  typedef float f32x2v __attribute__((ext_vector_type(2)));
  f32x4 v[MAXC][NCH][2];
  auto fetch = [&](int c, int c0) {
#pragma unroll
    for (int u = 0; u < NCH; ++u)
#pragma unroll
      for (int q = 0; q < 2; ++q) v[c][u][q] = *reinterpret_cast<const f32x4*>(p[c] + min(c0 + u, n_chunks - 1) * pitch + 4 * q);
  };
  for (int i = threadIdx.x; i < heads * n_chunks; i += 256)
    *reinterpret_cast<f32x2v*>(ml + 2 * i) = *reinterpret_cast<const f32x2v*>(base + (int64_t)i * pitch);
#pragma unroll
  for (int c = 0; c < MAXC; ++c) {
    const int e = min(c * 256 + (int)threadIdx.x, K / 8 - 1) * 8, h = e / dh;
    at[c] = h * n_chunks;
    p[c] = base + (int64_t)h * n_chunks * pitch + kPartPad + (e - h * dh);
    fetch(c, 0);
  }
  ad.load(g, group, K);
  __syncthreads();
  u32x4 x[MAXC];
#pragma unroll
  for (int c = 0; c < MAXC; ++c) {
    x[c] = u32x4{0, 0, 0, 0};
    const float* m = ml + 2 * at[c];
    float M = kNegBig;
    for (int i = 0; i < n_chunks; ++i)
      if (m[2 * i + 1] != 0.f) M = fmaxf(M, m[2 * i]);
    float L = 0.f, o[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int c0 = 0; c0 < n_chunks; c0 += NCH) {
      if (c0 > 0) fetch(c, c0);
#pragma unroll
      for (int u = 0; u < NCH; ++u) {
        const int i = c0 + u;
        if (i < n_chunks) {
          const float l = m[2 * i + 1];
          if (l != 0.f) {   // (a chunk without a key: an O nobody wrote)
            const float w = __expf(m[2 * i] - M);
            L += w * l;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              o[q] += w * v[c][u][0][q];
              o[4 + q] += w * v[c][u][1][q];
            }
          }
        }
      }
    }
    const int ch = c * 256 + threadIdx.x;
    if (ch < K / 8) {
#pragma unroll
      for (int q = 0; q < 4; ++q) x[c][q] = L != 0.f ? pack2bf(o[2 * q] / L, o[2 * q + 1] / L) : 0u;
      if (group == 0) *reinterpret_cast<u32x4*>(out + row * K + (int64_t)ch * 8) = x[c];
    }
  }
  ad.finish(g, group, row, x, sums);
}

// Whether one launch merges the chunks and takes the adapter columns, sixteen per work-group: as long as a row's partials are 64 KB, which every
// group of columns reads again, and every compute unit has at most one work-group (beyond, two share its registers and its reads).  us, attention with two launches |
// one behind it, K and the adapter from memory: 32 heads of 128, 64 columns, 2 chunks 16 rows (64 work-groups) 14.0 | 12.8, 64 rows (256) 22.5 | 20.5, 80 rows (320)
// 30.8 | 34.8; 4 chunks 48 rows 32.6 | 31.0, 100 rows 51.9 | 59.7; 16 heads of 128 80 rows x 8 chunks 42.6 | 47.0.
constexpr int kCombineCols = 16;
bool attn_lora_one_launch(int64_t rows, int64_t K, int n_chunks, int R) {
  return K <= 8 * 256 * 2 && n_chunks * K * 4 <= 64 * 1024 && rows * cdiv(R, kCombineCols) <= 256;
}

int next_pow2(int x) {
  int p = 1;
  while (p < x) p <<= 1;
  return p;
}

}  // namespace

extern "C" size_t tnx_attn_ws_bytes(int64_t B, int64_t T, int64_t S, int Hq, int dh,
                                    int kv_chunk) {
  if (kv_chunk <= 0) return 0;
  const int64_t n_chunks = cdiv(S, kv_chunk);
  return (size_t)(B * T * Hq * n_chunks * (dh + kPartPad)) * sizeof(float);
}

// Whether four waves share each chunk: of more than two key blocks, as long as two work-groups per compute unit hold them all (beyond, waves
// enough of their own: 128 rows x 8 kv heads x 160 keys 21.9 us with one wave, 25.0 with four).
static bool several_waves(const tnx_attn_desc* d, int n_chunks, int64_t keys_over) {
  const int64_t chunk_keys = d->kv_chunk > 0 ? d->kv_chunk : d->S;
  return d->T == 1 && (d->window > 0 ? std::min<int64_t>(chunk_keys, d->window) : chunk_keys) > keys_over && d->B * d->Hkv * n_chunks <= 512;
}

// The attention launch; combine: and, of a split key range, the pass that merges its chunks.  rope: what forms q and writes the step's
// key and value in the same launch (checked by the caller), or null.
static int gqa_attn(void* stream, const tnx_attn_desc* d, bool combine, const RopeArgs* rope = nullptr, const tnx_packed_rows* packed = nullptr) {
  TNX_REQUIRE(d, "attn: null descriptor");
  TNX_REQUIRE(d->B > 0 && d->T > 0 && d->S > 0, "attn: B,T,S must be positive");
  TNX_REQUIRE(d->dh == 64 || d->dh == 128 || d->dh == 256, "attn: head_dim %d not in {64,128,256}", d->dh);
  TNX_REQUIRE(d->Hkv > 0 && d->Hq % d->Hkv == 0, "attn: Hq=%d not a multiple of Hkv=%d", d->Hq, d->Hkv);
  const int G = d->Hq / d->Hkv;
  TNX_REQUIRE(G <= 16, "attn: group size %d > 16 not supported", G);
  TNX_REQUIRE(d->kcache && d->vcache && (d->tokens || d->segment_ids) && d->col_ptr && d->out, "attn: null pointer");
  TNX_REQUIRE(d->kv_chunk >= 0 && d->kv_chunk % 32 == 0, "attn: kv_chunk must be a multiple of 32");
  TNX_REQUIRE(d->tok_ld > 0, "attn: tok_ld=%lld must be positive", (long long)d->tok_ld);
  AttnArgs a;
  a.B = d->B; a.T = d->T; a.S = d->S; a.Hq = d->Hq; a.Hkv = d->Hkv; a.dh = d->dh;
  a.G = G; a.Gp = next_pow2(G);
  a.gp_shift = 0;
  while ((1 << a.gp_shift) < a.Gp) ++a.gp_shift;
  a.QT = (unsigned)cdiv(d->T, 16 / a.Gp);
  a.QTG = 1;
  // bf16(scale), as a weak-typed python float multiplied into a bf16 array
  if (d->scale != 0.f) {
    uint32_t u; float f = d->scale; memcpy(&u, &f, 4);
    u = (u + 0x7fffu + ((u >> 16) & 1u)) & 0xffff0000u;
    memcpy(&a.scale_bf, &u, 4);
  } else {
    a.scale_bf = 0.f;
  }
  a.window = d->window; a.pad_id = d->pad_id;
  a.q = d->q; a.k = d->kcache; a.v = d->vcache; a.tokens = d->segment_ids ? d->segment_ids : d->tokens; a.tok_ld = d->tok_ld;
  a.seg_mode = d->segment_ids ? 1 : 0;
  a.col_ptr = d->col_ptr; a.kv_chunk = d->kv_chunk;
  a.n_chunks = d->kv_chunk > 0 ? (int)cdiv(d->S, d->kv_chunk) : 1;
  a.ws = d->ws; a.out = d->out;
  a.qkv_ws = nullptr; a.qkv = nullptr; a.qkv_split = 0; a.rope_sin = nullptr; a.rope_cos = nullptr; a.rows = kAllRows;
  if (packed) {
    TNX_REQUIRE(d->kv_chunk == 0 && !d->rope_sin && !d->segment_ids, "attn: packed rows take no key chunks, rotation or segments");
    const int rc = packed_args(packed, d->B, d->T, a.rows);
    if (rc) return rc;
  }
  if (d->rope_sin) {
    TNX_REQUIRE(d->T == 1 && d->dh == 128, "attn: the fused RoPE / cache write needs T == 1 and head_dim 128");
    TNX_REQUIRE(d->rope_cos && (d->qkv || d->qkv_ws), "attn: fused RoPE needs the sine / cosine table and the qkv output");
    if (d->qkv_ws) TNX_REQUIRE(d->qkv_split >= 1 && d->qkv_split <= 64, "attn: qkv_split=%d out of range", d->qkv_split);
    a.qkv_ws = d->qkv_ws; a.qkv = d->qkv; a.qkv_split = d->qkv_split;
    a.rope_sin = d->rope_sin; a.rope_cos = d->rope_cos;
  } else {
    TNX_REQUIRE(d->q, "attn: null pointer");
  }
  if (a.n_chunks > 1) TNX_REQUIRE(d->ws, "attn: split key range needs a workspace");
  // (the combine keeps the chunks' (max, sum) pairs in LDS: 8 bytes per chunk)
  TNX_REQUIRE(a.n_chunks <= 4096, "attn: %d key chunks (S / kv_chunk), at most 4096", a.n_chunks);
  const int PT = 16 / a.Gp;
  const int64_t QT = cdiv(d->T, PT);
  TNX_REQUIRE(d->B * QT <= 65535 * 32, "attn: too many query tiles");
  dim3 grid((unsigned)a.n_chunks, (unsigned)d->Hkv, (unsigned)(d->B * QT));
  hipStream_t st = as_stream(stream);
  const bool tv = (d->tok_ld % 4 == 0) && ((reinterpret_cast<uintptr_t>(a.tokens) & 15) == 0) && d->S % 4 == 0;
  auto launch_decode = [&](auto dh_c, auto fuse_c, auto waves_c) {
    constexpr int DH = decltype(dh_c)::value, FUSE = decltype(fuse_c)::value, W = decltype(waves_c)::value;
    if (tv) hipLaunchKernelGGL((attn_kernel<DH, FUSE, true, W>), grid, dim3(64 * W), 0, st, a);
    else hipLaunchKernelGGL((attn_kernel<DH, FUSE, false, W>), grid, dim3(64 * W), 0, st, a);
  };
  const bool waves = !packed && several_waves(d, a.n_chunks, 64);
  auto launch_head_dim = [&](auto dh_c, auto fuse_c) {
    if (waves) launch_decode(dh_c, fuse_c, std::integral_constant<int, kAttnWaves>{});
    else launch_decode(dh_c, fuse_c, std::integral_constant<int, 1>{});
  };
#define TNX_ATTN_LAUNCH(DH, FUSE) launch_head_dim(std::integral_constant<int, DH>{}, std::integral_constant<int, FUSE>{})
  // many query positions at head_dim 128 or 256, no key split, no fused rotation: keys and values through LDS, eight | four query tiles
  // per work-group.  At 256 every wave's own loads of its keys and values are what bounds the other form; us, through LDS | per wave, positions
  // x rows, 4 heads on one: 256 x 64 38.6 | 133.4, 1000 x 16 92 | 335, 3000 x 8 308 | 1334 (window of 512 117 | 490), 3000 x 1 117 | 210; 64 x 64
  // 9.1 | 14.8, 64 x 1 6.7 | 6.1; of fewer tiles, 32 x 64 6.6 | 6.4, 32 x 1 5.5 | 4.6.
  if (!a.rope_sin && a.n_chunks == 1 && d->dh >= 128) {
    auto launch = [&](auto dh_c, auto scaled_c) -> int {
      constexpr int DH = decltype(dh_c)::value;
      constexpr bool SCALED = decltype(scaled_c)::value;
      static std::once_flag wg_once;
      static hipError_t wg_rc = hipSuccess;
      constexpr int kLds = (int)(wg_stages(DH) * wg_stage_bytes(DH));
      std::call_once(wg_once, [] {
        wg_rc = hipFuncSetAttribute(reinterpret_cast<const void*>(&attn_wg_kernel<DH, SCALED>),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
      });
      TNX_REQUIRE(wg_rc == hipSuccess, "attn: cannot raise the dynamic LDS limit");
      hipLaunchKernelGGL((attn_wg_kernel<DH, SCALED>), dim3(1u, (unsigned)d->Hkv, (unsigned)(d->B * a.QTG)), dim3(256), kLds, st, a);
      TNX_CHECK_LAUNCH("gqa_attn (work-group tiles)");
      return TNX_OK;
    };
    const int tiles = 4 * wg_tiles_per_wave(d->dh);   // of a work-group
    if (QT >= 16 && (uint64_t)d->S * d->dh * 2u < (1ull << 32) && d->B * cdiv(QT, tiles) <= 65535) {
      a.QTG = (unsigned)cdiv(QT, tiles);
      const bool scaled = a.scale_bf != 0.f;
      if (d->dh == 128) return scaled ? launch(std::integral_constant<int, 128>{}, std::true_type{}) : launch(std::integral_constant<int, 128>{}, std::false_type{});
      return scaled ? launch(std::integral_constant<int, 256>{}, std::true_type{}) : launch(std::integral_constant<int, 256>{}, std::false_type{});
    }
  }
  // many query positions, no key split, no fused rotation: two query tiles per wave
  constexpr int kTilesPerWave = 2;
  if (!a.rope_sin && a.n_chunks == 1 && d->dh <= 128 && QT >= 2 * kTilesPerWave) {
    a.QTG = (unsigned)cdiv(QT, kTilesPerWave);
    dim3 tgrid(1u, (unsigned)d->Hkv, (unsigned)(d->B * a.QTG));
    if (d->dh == 64) {
      if (tv) hipLaunchKernelGGL((attn_tiles_kernel<64, true, kTilesPerWave>), tgrid, dim3(64), 0, st, a);
      else hipLaunchKernelGGL((attn_tiles_kernel<64, false, kTilesPerWave>), tgrid, dim3(64), 0, st, a);
    } else {
      if (tv) hipLaunchKernelGGL((attn_tiles_kernel<128, true, kTilesPerWave>), tgrid, dim3(64), 0, st, a);
      else hipLaunchKernelGGL((attn_tiles_kernel<128, false, kTilesPerWave>), tgrid, dim3(64), 0, st, a);
    }
    TNX_CHECK_LAUNCH("gqa_attn (tiles)");
    return TNX_OK;
  }
  auto launch_rope = [&](auto dh_c, auto few_c) {
    constexpr int DH = decltype(dh_c)::value;
    constexpr bool FEW = decltype(few_c)::value;
    if (tv) hipLaunchKernelGGL((attn_rope_kernel<DH, true, FEW>), grid, dim3(64 * kAttnWaves), 0, st, a, *rope);
    else hipLaunchKernelGGL((attn_rope_kernel<DH, false, FEW>), grid, dim3(64 * kAttnWaves), 0, st, a, *rope);
  };
  auto launch_rope_keys = [&](auto dh_c) {
    if (waves) launch_rope(dh_c, std::false_type{});
    else launch_rope(dh_c, std::true_type{});
  };
  if (rope) {
    if (d->dh == 64) launch_rope_keys(std::integral_constant<int, 64>{});
    else launch_rope_keys(std::integral_constant<int, 128>{});
  } else switch (d->dh) {
    case 64: TNX_ATTN_LAUNCH(64, 0); break;
    case 128:
      if (a.rope_sin && a.qkv_ws && a.qkv_split <= 8 && G <= 4) TNX_ATTN_LAUNCH(128, 2);
      else if (a.rope_sin) TNX_ATTN_LAUNCH(128, 1);
      else TNX_ATTN_LAUNCH(128, 0);
      break;
    default: TNX_ATTN_LAUNCH(256, 0); break;
  }
#undef TNX_ATTN_LAUNCH
  TNX_CHECK_LAUNCH("gqa_attn");
  if (a.n_chunks > 1 && combine) {
    const int64_t nq = d->B * d->T * d->Hq;
    hipLaunchKernelGGL(attn_combine_kernel, dim3((unsigned)nq), dim3(d->dh), (size_t)a.n_chunks * 2 * sizeof(float), st,
                       a.ws, nq, d->dh, a.n_chunks, a.out);
    TNX_CHECK_LAUNCH("gqa_attn_combine");
  }
  return TNX_OK;
}

extern "C" int tnx_gqa_attn(void* stream, const tnx_attn_desc* d) { return gqa_attn(stream, d, true); }
extern "C" int tnx_gqa_attn_packed(void* stream, const tnx_attn_desc* d, const tnx_packed_rows* rows) {
  TNX_REQUIRE(rows, "attn: null packed rows");
  return gqa_attn(stream, d, true, nullptr, rows);
}

static int gqa_attn_lora(void* stream, const tnx_attn_desc* d, const uint16_t* a_t, int R, uint16_t* t, int64_t t_ld, const RopeArgs* rope) {
  TNX_REQUIRE(d && a_t && t, "attn_lora: null pointer");
  TNX_REQUIRE(R > 0 && R % 16 == 0 && t_ld >= R, "attn_lora: R=%d must be a multiple of 16 and <= t_ld", R);
  const int64_t K = (int64_t)d->Hq * d->dh;
  TNX_REQUIRE(d->B > 0 && d->T > 0 && K > 0 && K % 32 == 0, "attn_lora: bad shape");
  const int n_chunks = d->kv_chunk > 0 ? (int)cdiv(d->S, d->kv_chunk) : 1;
  // (the groups of columns of a row write t while others still read its partials)
  const bool one = d->T == 1 && n_chunks > 1 && attn_lora_one_launch(d->B, K, n_chunks, R) &&
                   apart(t, ((d->B - 1) * t_ld + R) * 2, d->ws, (int64_t)tnx_attn_ws_bytes(d->B, 1, d->S, d->Hq, d->dh, d->kv_chunk));
  const int rc = gqa_attn(stream, d, !one, rope);
  if (rc != TNX_OK) return rc;
  if (!one) return tnx_lora_down(stream, d->out, d->B * d->T, K, a_t, R, t, t_ld);
  RowAdapterArgs g{a_t, R, kCombineCols, t, t_ld, 0, 0};
  const dim3 grid = row_adapter_grid(g, d->B, K, n_chunks * K * 4);
  const size_t lds = (size_t)d->Hq * n_chunks * 2 * sizeof(float);
  auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, dim3(256), lds, as_stream(stream), d->ws, d->B, d->Hq, d->dh, n_chunks, d->out, g); };
  if (K <= 8 * 256) n_chunks <= 4 ? launch(attn_combine_lora_kernel<1, kCombineCols, 4>) : launch(attn_combine_lora_kernel<1, kCombineCols, 8>);
  else n_chunks <= 4 ? launch(attn_combine_lora_kernel<2, kCombineCols, 4>) : launch(attn_combine_lora_kernel<2, kCombineCols, 8>);
  TNX_CHECK_LAUNCH("gqa_attn_combine_lora");
  return TNX_OK;
}

extern "C" int tnx_gqa_attn_lora(void* stream, const tnx_attn_desc* d, const uint16_t* a_t, int R, uint16_t* t, int64_t t_ld) {
  return gqa_attn_lora(stream, d, a_t, R, t, t_ld, nullptr);
}

// combine: see gqa_attn
static int rope_gqa_attn(void* stream, const tnx_rope_desc* r, const tnx_attn_desc* d, const uint16_t* a_t, int R, uint16_t* t, int64_t t_ld, bool combine) {
  TNX_REQUIRE(r && d, "rope_gqa_attn: null descriptor");
  RopeArgs ra;
  int rc = rope_args(r, ra);
  if (rc) return rc;
  TNX_REQUIRE(r->B == d->B && r->T == d->T && r->S == d->S && r->Hq == d->Hq && r->Hkv == d->Hkv && r->dh == d->dh && r->q_out == d->q &&
                  r->kcache == d->kcache && r->vcache == d->vcache && r->col_ptr == d->col_ptr && !d->rope_sin,
              "rope_gqa_attn: the two descriptors name different rows");
  const int n_chunks = d->kv_chunk > 0 ? (int)cdiv(d->S, d->kv_chunk) : 1;
  const bool aligned = (((uintptr_t)r->kcache | (uintptr_t)r->vcache) & 15) == 0;
  // (heads of 256, which three chunks form again each: 1.0 us more per layer than in two launches, Gemma3-1B, 64 rows)
  // The chunks of a head read its planes while the first to end writes its output: neither output may lie in them.
  const int64_t planes = (int64_t)r->split_k * r->B * (r->Hq + 2 * r->Hkv) * r->dh * 4;
  const bool separate = apart(d->out, d->B * d->Hq * d->dh * 2, r->qkv_ws, planes) &&
                        apart(d->ws, (int64_t)tnx_attn_ws_bytes(d->B, 1, d->S, d->Hq, d->dh, d->kv_chunk), r->qkv_ws, planes);
  // Of few keys the heads bound it, three a wave at a time, and a second batch of them pays with many rows of heads of 64 only.  us, two
  // launches | one, 64 keys: 10 + 2 heads of 128 16 rows 11.9 | 12.2; 12 + 2 12.2 | 13.9, 2 x (16 + 2) 13.4 | 15.3, 64 rows 14.3 | 15.7; 4 x (12 + 2)
  // heads of 64 16 rows 12.8 | 13.4, 100 rows 16.0 | 15.2, 4 x (16 + 2) of 128 70 rows 19.1 | 20.2; 90 keys: 12 + 2 of 128 16 rows 15.6 | 13.2.
  const int64_t groups = (int64_t)d->B * d->Hkv;
  const bool heads_fit = d->Hq <= (3 * kAttnWaves - 2) * d->Hkv || (d->dh == 64 && groups > 256) || several_waves(d, n_chunks, 64);
  const bool one = r->qkv_ws && r->split_k <= 8 && aligned && separate && (d->dh == 64 || d->dh == 128) && heads_fit && several_waves(d, n_chunks, 0);
  if (!one) {
    rc = tnx_qknorm_rope_kvwrite(stream, r);
    if (rc) return rc;
  }
  const RopeArgs* rope = one ? &ra : nullptr;
  return a_t ? gqa_attn_lora(stream, d, a_t, R, t, t_ld, rope) : gqa_attn(stream, d, combine, rope);
}

extern "C" int tnx_rope_gqa_attn_lora(void* stream, const tnx_rope_desc* r, const tnx_attn_desc* d, const uint16_t* a_t, int R, uint16_t* t,
                                      int64_t t_ld) {
  return rope_gqa_attn(stream, r, d, a_t, R, t, t_ld, true);
}

extern "C" int tnx_gqa_attn_parts(void* stream, const tnx_rope_desc* r, const tnx_attn_desc* d) {
  TNX_REQUIRE(d && d->T == 1 && d->kv_chunk > 0 && d->S > d->kv_chunk, "gqa_attn_parts: a decode step whose key range is cut into chunks");
  return r ? rope_gqa_attn(stream, r, d, nullptr, 0, nullptr, 0, false) : gqa_attn(stream, d, false);
}
