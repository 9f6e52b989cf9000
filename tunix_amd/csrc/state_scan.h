// A matrix state carried token by token in 32 bits, S_t = f_t S_(t-1) + k_t v_t^T and o_t = S_t^T q_t (f a factor per row of S, or one of the
// head), for the head sizes and types that the chunk kernels on MFMAs do not take.
//
// A work-group of four waves has up to 64 columns of a state of up to 4 R rows: a lane one column, a wave R rows, in registers.  q, k, f
// and v come in batches of tokens, through registers into the other half of an LDS buffer while a batch is worked on; the waves' parts of o
// meet once per batch.  Bound by the chain of tokens: 3 R vector instructions and R / 2 broadcast reads each.
#pragma once
#include "decoder.h"

namespace {

constexpr int kScanCols = 64;

// Tokens [t0, T) of one (sequence, head); columns d0 .. of the state S [dk, dv].  fresh: S is taken as zero.
// load(t, i) -> f32x4, what make(raw, q, k, f) forms q_i, k_i (and, FORGET, f_i) of a token from; load_v(t, d); out(t, d, o).
template <int R, bool FORGET, class Load, class Make, class LoadV, class Out>
__device__ __forceinline__ void state_scan(int64_t t0, int64_t T, int dk, int dv, int d0, bool fresh, float decay, float* S, Load load, Make make,
                                           LoadV load_v, Out out) {
  constexpr int DK = 4 * R, TB = R > 32 ? 4 : 8, N = TB * DK / 256, NV = TB * kScanCols / 256;
  __shared__ __align__(16) float qs[2][TB][DK], ks[2][TB][DK], fs[FORGET ? 2 : 1][FORGET ? TB : 1][FORGET ? DK : 1];
  __shared__ float vs[2][TB][kScanCols], part[2][TB][4][kScanCols];
  __shared__ int odd[kScanCols];   // whether a column's v holds an infinity or a NaN
  const int tid = threadIdx.x, lane = tid & 63;
  const int r0 = __builtin_amdgcn_readfirstlane(tid >> 6) * R, wave = r0 / R;
  const int d = d0 + lane;
  const bool mine = d < dv;
  float s[R];
#pragma unroll
  for (int r = 0; r < R; ++r) s[r] = !fresh && mine && r0 + r < dk ? S[(int64_t)(r0 + r) * dv + d] : 0.f;
  f32x4 raw[N];
  float rv[NV];
  auto fetch = [&](int64_t t) {
#pragma unroll
    for (int n = 0; n < N; ++n) {
      const int e = n * 256 + tid, i = e % DK;
      raw[n] = i < dk && t + e / DK < T ? load(t + e / DK, i) : f32x4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int n = 0; n < NV; ++n) {
      const int e = n * 256 + tid, c = d0 + e % kScanCols;
      rv[n] = c < dv && t + e / kScanCols < T ? load_v(t + e / kScanCols, c) : 0.f;
    }
  };
  auto put = [&](int b) {
#pragma unroll
    for (int n = 0; n < N; ++n) {
      const int e = n * 256 + tid, u = e / DK, i = e % DK;
      float q = 0.f, k = 0.f, f = 0.f;
      if (i < dk) make(raw[n], q, k, f);   // (rows past the last: nothing enters them, and they enter nothing)
      qs[b][u][i] = q;
      ks[b][u][i] = k;
      if constexpr (FORGET) fs[b][u][i] = f;
    }
#pragma unroll
    for (int n = 0; n < NV; ++n) {
      // (an infinity would make NaNs of the rows past the last, whose k is zero: it stays out, and its column is formed again in the end)
      const int e = n * 256 + tid;
      const bool finite = fabsf(rv[n]) < __builtin_inff();
      vs[b][e / kScanCols][e % kScanCols] = finite ? rv[n] : 0.f;
      if (!finite) odd[e % kScanCols] = 1;
    }
  };
  if (tid < kScanCols) odd[tid] = 0;
  fetch(t0);
  __syncthreads();
  put(0);
  __syncthreads();
  int b = 0;
  for (int64_t tb = t0; tb < T; tb += TB, b ^= 1) {
    const int nt = (int)min((int64_t)TB, T - tb);
    if (tb + TB < T) fetch(tb + TB);
#pragma unroll 1
    for (int u = 0; u < nt; ++u) {
      const float v = vs[b][u][lane];
      f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int r = 0; r < R; r += 4) {
        const f32x4 q = *reinterpret_cast<const f32x4*>(&qs[b][u][r0 + r]), k = *reinterpret_cast<const f32x4*>(&ks[b][u][r0 + r]);
        f32x4 f = f32x4{decay, decay, decay, decay};
        if constexpr (FORGET) f = *reinterpret_cast<const f32x4*>(&fs[b][u][r0 + r]);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          s[r + e] = __builtin_fmaf(k[e], v, f[e] * s[r + e]);
          acc[e] = __builtin_fmaf(q[e], s[r + e], acc[e]);
        }
      }
      part[b][u][wave][lane] = (acc[0] + acc[1]) + (acc[2] + acc[3]);
    }
    if (tb + TB < T) put(b ^ 1);
    __syncthreads();   // (a batch's parts are read behind it, and written again two batches on)
    for (int e = tid; e < nt * kScanCols; e += 256) {
      const int u = e / kScanCols, c = e % kScanCols;
      if (d0 + c < dv) out(tb + u, d0 + c, (part[b][u][0][c] + part[b][u][1][c]) + (part[b][u][2][c] + part[b][u][3][c]));
    }
  }
#pragma unroll
  for (int r = 0; r < R; ++r)
    if (mine && !odd[lane] && r0 + r < dk) S[(int64_t)(r0 + r) * dv + d] = s[r];
  __syncthreads();   // (every output is written)
  if (tid < kScanCols && mine && odd[lane]) {   // token by token, from the state as it was; the first wave's lane is the column
    bool seen = false;
    for (int64_t t = t0; t < T; ++t) {
      const float v = load_v(t, d);
      seen = seen || !(fabsf(v) < __builtin_inff());
      float acc = 0.f;
      for (int i = 0; i < dk; ++i) {
        float q, k, f = decay;
        make(load(t, i), q, k, f);
        float& at = S[(int64_t)i * dv + d];
        at = __builtin_fmaf(k, v, fresh && t == t0 ? 0.f : f * at);
        acc = __builtin_fmaf(q, at, acc);
      }
      if (seen) out(t, d, acc);
    }
  }
}

}  // namespace
