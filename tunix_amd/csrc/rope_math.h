// Per-head norm and rotation of q and k, and what a norm does to one element: shared by the kernels that do it on its own (norm_rope.hip) and the
// decode attention that does it in front (attention.hip).
#pragma once
#include <string.h>

#include "common.h"
#include "packed_rows.h"

namespace {

// One normalised element, given the row statistics.  `ms` is mean(x^2) (llama/qwen3: fp32 of
// fp32 squares; gemma3: bf16-rounded mean of bf16-rounded squares).
__device__ __forceinline__ float norm_elem(float x, float w, float ms, float eps, int flavor) {
  if (flavor == TNX_NORM_LLAMA) {
    // astype(w * x / rms): w*x is a bf16 product, the division is fp32.
    const float rms = sqrtf(ms + eps);
    return rbf(rbf(w * x) / rms);
  } else if (flavor == TNX_NORM_QWEN3) {
    const float rms = sqrtf(ms + eps);
    return rbf(w * (x / rms));
  } else {
    // gemma3: every op in bf16: x * rsqrt(var + eps) * (1 + scale)
    const float r = rbf(1.0f / sqrtf(rbf(ms + eps)));
    return rbf(rbf(x * r) * rbf(1.0f + w));
  }
}
__device__ __forceinline__ float sq_term(float x, int flavor) {
  return flavor == TNX_NORM_GEMMA3 ? rbf(x * x) : x * x;
}
__device__ __forceinline__ float finish_ms(float ss, float n, int flavor) {
  const float ms = ss / n;
  return flavor == TNX_NORM_GEMMA3 ? rbf(ms) : ms;
}

struct RopeArgs {
  int64_t B, T, S;
  int Hq, Hkv, dh;
  int rope_flavor;
  float rope_scale;
  int qk_norm;
  float norm_eps;
  const uint16_t* q_norm_w;
  const uint16_t* k_norm_w;
  float q_prescale_bf;
  const uint16_t* qkv;
  const int32_t* positions;
  int64_t pos_ld;
  const int32_t* col_ptr;
  const float* timescale;
  uint16_t* q_out;
  uint16_t* kcache;
  uint16_t* vcache;
  const float* ws;   // split-k partial planes of the qkv linear instead of qkv, or null
  int split_k;
  PackedRows rows;
};

// The rotated pair (x1, x2) of a q or k head, as bf16 values.
__device__ __forceinline__ void rotate_pair(const RopeArgs& a, bool is_q, float x1, float x2, float sn, float cs, float& o1, float& o2) {
  if (a.rope_flavor == TNX_ROPE_QWEN3) {
    o1 = rbf(rbf(x1 * cs) - rbf(x2 * sn));
    o2 = rbf(rbf(x2 * cs) + rbf(x1 * sn));
  } else {
    // fp32, one rounding to bf16 at the end; written as the fused forms the compiler makes of such a sum, so that every kernel takes the
    // same one
    o1 = rbf(__builtin_fmaf(x1, cs, -(x2 * sn)));
    o2 = rbf(__builtin_fmaf(x2, cs, x1 * sn));
  }
  if (is_q && a.q_prescale_bf != 0.f) {
    o1 = rbf(o1 * a.q_prescale_bf);
    o2 = rbf(o2 * a.q_prescale_bf);
  }
}
// sine and cosine of one (position, pair), rounded where the flavor rounds them
__device__ __forceinline__ void rope_angle(const RopeArgs& a, float pos, float timescale, float& sn, float& cs) {
  float ang = __fdiv_rn(pos, timescale);
  if (a.rope_flavor == TNX_ROPE_GEMMA3) ang = __fdiv_rn(ang, a.rope_scale);
  sn = sinf(ang);
  cs = cosf(ang);
  if (a.rope_flavor == TNX_ROPE_QWEN3) {
    sn = rbf(sn);
    cs = rbf(cs);
  }
}
// cache slot of the token at column c (the cache is a ring; a division only where it wraps)
__device__ __forceinline__ int64_t ring_slot(int64_t c, int64_t S) { return c < S ? c : c % S; }

inline float host_round_bf16(float f) {
  uint32_t u;
  memcpy(&u, &f, 4);
  u = (u + 0x7fffu + ((u >> 16) & 1u)) & 0xffff0000u;
  memcpy(&f, &u, 4);
  return f;
}

// the kernels' arguments of a checked descriptor
inline int rope_args(const tnx_rope_desc* d, RopeArgs& a) {
  TNX_REQUIRE(d, "rope: null descriptor");
  TNX_REQUIRE(d->B > 0 && d->T > 0 && d->S > 0, "rope: bad shape");
  TNX_REQUIRE(d->dh % 2 == 0 && d->dh >= 2 && d->dh <= 512, "rope: bad head_dim %d", d->dh);
  TNX_REQUIRE((d->qkv || d->qkv_ws) && d->positions && d->col_ptr && d->timescale && d->q_out &&
                  d->kcache && d->vcache,
              "rope: null pointer");
  if (d->qkv_ws) TNX_REQUIRE(d->split_k >= 1 && d->split_k <= 64, "rope: split_k=%d out of range", d->split_k);
  TNX_REQUIRE(d->rope_flavor >= TNX_ROPE_LLAMA && d->rope_flavor <= TNX_ROPE_GEMMA3, "rope: bad flavor");
  TNX_REQUIRE(d->qk_norm >= -1 && d->qk_norm <= TNX_NORM_GEMMA3, "rope: bad qk_norm");
  if (d->qk_norm >= 0) TNX_REQUIRE(d->q_norm_w && d->k_norm_w, "rope: qk_norm weights are null");
  if (d->rope_flavor == TNX_ROPE_GEMMA3)
    TNX_REQUIRE(d->rope_scale >= 1.0f, "rope: scale_factor must be >= 1.0, got %f", d->rope_scale);
  a.B = d->B; a.T = d->T; a.S = d->S; a.Hq = d->Hq; a.Hkv = d->Hkv; a.dh = d->dh;
  a.rope_flavor = d->rope_flavor; a.rope_scale = d->rope_scale; a.qk_norm = d->qk_norm;
  a.norm_eps = d->norm_eps; a.q_norm_w = d->q_norm_w; a.k_norm_w = d->k_norm_w;
  a.q_prescale_bf = d->q_prescale != 0.f ? host_round_bf16(d->q_prescale) : 0.f;
  a.qkv = d->qkv; a.positions = d->positions; a.pos_ld = d->pos_ld; a.col_ptr = d->col_ptr;
  a.timescale = d->timescale; a.q_out = d->q_out; a.kcache = d->kcache; a.vcache = d->vcache;
  a.ws = d->qkv_ws; a.split_k = d->split_k; a.rows = kAllRows;
  return TNX_OK;
}

}  // namespace
