// What the many-row kernels (qgemm_wide.h, qgemm_pre.h) do with a finished tile of ROWS rows x 256 columns
// that a work-group of 256 threads has staged in LDS as bf16 (from address 0, row stride columns + 8 elements; a gated
// unit's 128 products otherwise): stores it in whole 16-byte chunks, or reduces it to lm_head statistics.
//
// Included by qlinear.hip after qgemm128.h.
#pragma once

namespace {

constexpr int kWideCols = 256;

// Whether an adapter's scale is a power of two near one (1 where alpha is the rank): B times the scale is exact then, and the
// delta is summed onto the accumulators directly.
__host__ __device__ inline bool lora_in_place(float scale) {
  return (__builtin_bit_cast(uint32_t, scale) & 0x007fffffu) == 0u && scale >= 1.0f / 256.0f && scale <= 256.0f;
}

template <int ROWS, bool GROUPED, bool HEAD, bool MUL>
__device__ __forceinline__ void wide_tile_out(const QLArgs& a, const WideHead& h, int ntile, int64_t m0, int rows_here) {
  const int tid = threadIdx.x, lane = tid & 63, wn = __builtin_amdgcn_readfirstlane(tid >> 6);
  constexpr int cols = MUL ? kWideCols / 2 : kWideCols;      // output columns of the work-group
  constexpr int sld = cols + 8;
  constexpr uint32_t stage = 0;
  if (HEAD && h.logits_out != nullptr) {
    // the raw logits (no temperature) as fp32: a wave writes one row of the tile at a time, a
    // lane four columns (1 KB per row, whole lines)
    const int64_t c0 = (int64_t)ntile * kWideCols + lane * 4;
    for (int row = wn; row < rows_here; row += 4) {
      const u32x2 v = *reinterpret_cast<const __attribute__((address_space(3))) u32x2*>(
          static_cast<uintptr_t>(stage + (uint32_t)((row * sld + lane * 4) * 2)));
      float* o = h.logits_out + (m0 + row) * a.N + c0;
      if (c0 + 4 <= a.N) {
        *reinterpret_cast<f32x4*>(o) = f32x4{bflo(v[0]), bfhi(v[0]), bflo(v[1]), bfhi(v[1])};
      } else {
        const float x[4] = {bflo(v[0]), bfhi(v[0]), bflo(v[1]), bfhi(v[1])};
        for (int e = 0; e < 4; ++e)
          if (c0 + e < a.N) o[e] = x[e];
      }
    }
  }
  if constexpr (HEAD) {
    // The whole-vocabulary draw: per column the logit plus the Gumbel noise of element row * N + col of
    // rows_total * N; a block's best (first among equals), its id and its logit go to part_draw.  The noise is a hundred instructions per
    // element, so the tile's (row, half) are spread over all threads: sixteen lanes share one, a 16-byte chunk each, or, where the rows alone
    // occupy the threads and no merging between lanes is needed, two or one take its chunks in turn.  us, one lane | sixteen | as chosen, 70000
    // columns x 512: 16 rows 109 | 39 | 39, 128 rows 92 | 100 | 92; 262144 x 1152: 16 rows 226 | 125 | 124, 256 rows 397 | 398 | 365.
    if (h.part_draw != nullptr) {
      uint32_t ks0 = 0u, ks1 = (uint32_t)(*h.step_ptr);
      threefry2x32(h.key0, h.key1, ks0, ks1);   // fold_in(key, step)
      const uint64_t total = (uint64_t)h.rows_total * (uint64_t)a.N;
      auto draw = [&](auto lanes_c) {
        constexpr int LANES = decltype(lanes_c)::value, STEP = 256 / LANES;
        const int first = tid % LANES;
        for (int p = tid / LANES; p < 2 * rows_here; p += STEP) {
          const int row = p >> 1, hf = p & 1;
          const int64_t pb = (int64_t)ntile * 2 + hf, grow = m0 + row;
          if (pb >= h.nvb) continue;   // (the same for the lanes of a row half)
          float gv = -__builtin_inff(), gl = gv;
          int gi = 0x7fffffff;
#pragma unroll 1
          for (int c = 0; c < 16 / LANES; ++c) {   // (columns ascend: the first among equals of a lane stays)
            const int64_t c0 = pb * 128 + (c * LANES + first) * 8;
            const u32x4 v = lds_ld128(stage + (uint32_t)((row * sld + hf * 128 + (c * LANES + first) * 8) * 2));
#pragma unroll
            for (int q = 0; q < 8; ++q) {
              const int64_t col = c0 + q;
              if (col < a.N) {
                const float raw = (q & 1) ? bfhi(v[q >> 1]) : bflo(v[q >> 1]);
                const float l = __fdiv_rn(raw, h.temperature);
                const float n = l + gumbel_from_bits(random_bits(ks0, ks1, (uint64_t)grow * (uint64_t)a.N + (uint64_t)col, total, h.variant));
                if (n > gv) {
                  gv = n;
                  gi = (int)col;
                  gl = l;
                }
              }
            }
          }
#pragma unroll
          for (int o = LANES / 2; o > 0; o >>= 1) {
            const float ov = lane_xor(gv, o), ol = lane_xor(gl, o);
            const int oi = lane_xor(gi, o);
            if (ov > gv || (ov == gv && oi < gi)) {
              gv = ov;
              gi = oi;
              gl = ol;
            }
          }
          if (first == 0) {
            float* q3 = h.part_draw + (grow * h.nvb + pb) * 3;
            q3[0] = gv;
            q3[1] = __int_as_float(gi);
            q3[2] = gl;
          }
        }
      };
      // (passes of 256 threads, the last one at least seven eighths full)
      const int rest = rows_here & 127;
      if (rows_here >= 112 && (rest == 0 || rest >= 112)) draw(std::integral_constant<int, 1>{});
      else if (rows_here >= 56 && rows_here <= 64) draw(std::integral_constant<int, 2>{});
      else draw(std::integral_constant<int, 16>{});
    }
    // lm_head: thread (row % 128, half) reduces the row's 128 staged logits of column block
    // 2 * ntile + half to (max, first arg-max, sum of exp(l - max), logit of the row's target)
    const int half = tid >> 7;
    const int64_t pb = (int64_t)ntile * 2 + half;
    if (pb >= h.nvb) return;
    for (int row = tid & 127; row < rows_here; row += 128) {
      const int64_t grow = m0 + row, c0 = pb * 128;
      const int tg = h.targets ? h.targets[grow] : -1;
      const uint32_t base = stage + (uint32_t)((row * sld + half * 128) * 2);
      const float ninf = -__builtin_inff();
      float mx = ninf, tgt = ninf, se = 0.f, we = 0.f;
      int idx = (int)c0;
      // The logits are divided by the temperature in fp32, as the reference does.  At temperature 1
      // the division is the identity and is left out: an IEEE division is a dozen instructions, and
      // at two per element it was a seventh of this kernel's time on the log-probability pass.
      auto reduce = [&](auto unit_c) {
        constexpr bool unit = decltype(unit_c)::value;
#pragma unroll 4
        for (int ch = 0; ch < 16; ++ch) {
          const u32x4 v = lds_ld128(base + (uint32_t)(ch * 16));
#pragma unroll
          for (int q = 0; q < 8; ++q) {
            const int64_t col = c0 + ch * 8 + q;
            const float raw = (q & 1) ? bfhi(v[q >> 1]) : bflo(v[q >> 1]);
            const float l = col < a.N ? (unit ? raw : __fdiv_rn(raw, h.temperature)) : ninf;
            if (l > mx) {   // columns ascend: the first maximal index stays
              mx = l;
              idx = (int)col;
            }
            if ((int)col == tg) tgt = l;
          }
        }
        if (mx != ninf) {
#pragma unroll 4
          for (int ch = 0; ch < 16; ++ch) {
            const u32x4 v = lds_ld128(base + (uint32_t)(ch * 16));
#pragma unroll
            for (int q = 0; q < 8; ++q) {
              const int64_t col = c0 + ch * 8 + q;
              const float raw = (q & 1) ? bfhi(v[q >> 1]) : bflo(v[q >> 1]);
              if (col < a.N) {
                const float l = unit ? raw : __fdiv_rn(raw, h.temperature);
                const float e = __expf(l - mx);
                se += e;
                we += e * l;
              }
            }
          }
        }
      };
      // A block that lies wholly inside the vocabulary, no entropy term asked for (every block of a
      // log-probability pass over a head whose width is a multiple of 128): the same arithmetic in
      // the same order without the per-element column tests, and the target's logit is read from its
      // place in the staged row instead of being compared for 128 times.
      auto reduce_full = [&](auto unit_c) {
        constexpr bool unit = decltype(unit_c)::value;
        const int c0i = (int)c0;
        if (tg >= c0i && tg < c0i + 128) {
          const uint32_t w = lds_ld32(base + (uint32_t)((tg - c0i) >> 1) * 4u);
          const float raw = ((tg - c0i) & 1) ? bfhi(w) : bflo(w);
          tgt = unit ? raw : __fdiv_rn(raw, h.temperature);
        }
#pragma unroll 4
        for (int ch = 0; ch < 16; ++ch) {
          const u32x4 v = lds_ld128(base + (uint32_t)(ch * 16));
#pragma unroll
          for (int q = 0; q < 8; ++q) {
            const float raw = (q & 1) ? bfhi(v[q >> 1]) : bflo(v[q >> 1]);
            const float l = unit ? raw : __fdiv_rn(raw, h.temperature);
            if (l > mx) {
              mx = l;
              idx = c0i + ch * 8 + q;
            }
          }
        }
        if (mx != ninf) {
#pragma unroll 4
          for (int ch = 0; ch < 16; ++ch) {
            const u32x4 v = lds_ld128(base + (uint32_t)(ch * 16));
#pragma unroll
            for (int q = 0; q < 8; ++q) {
              const float raw = (q & 1) ? bfhi(v[q >> 1]) : bflo(v[q >> 1]);
              const float l = unit ? raw : __fdiv_rn(raw, h.temperature);
              se += __expf(l - mx);
            }
          }
        }
      };
      const bool plain = c0 + 128 <= a.N && h.part_ent == nullptr;
      if (h.temperature == 1.0f) {
        if (plain) reduce_full(std::true_type{});
        else reduce(std::true_type{});
      } else {
        if (plain) reduce_full(std::false_type{});
        else reduce(std::false_type{});
      }
      float* p = h.part + (grow * h.nvb + pb) * 4;
      p[0] = mx;
      p[1] = __int_as_float(idx);
      p[2] = se;
      p[3] = tgt;
      if (h.part_ent) h.part_ent[grow * h.nvb + pb] = we;
    }
    return;
  }
  if constexpr (!HEAD) {
    const int64_t width = MUL ? a.N / 2 : a.N, ldy = a.ldy > 0 ? a.ldy : width;
    const int64_t col0 = (int64_t)ntile * cols;
    constexpr int chunks = cols / 8;                   // 16-byte chunks per row: 16 | 32
    const int ch = tid % chunks, r0 = tid / chunks, rstep = 256 / chunks;
    uint16_t* y = reinterpret_cast<uint16_t*>(a.y);
    const bool col_ok = col0 + ch * 8 + 8 <= width;
    // The places of all rows at once: y may lie anywhere for all the compiler knows, so that row by row every store stood behind a round trip to the L2
    // of its own (57288 routes of 128 experts, 768 -> 2048, 286 -> 271 us).
    constexpr int PER = ROWS / rstep;
    int route[GROUPED ? PER : 1];
    if constexpr (GROUPED) {
#pragma unroll
      for (int i = 0; i < PER; ++i) route[i] = a.sorted_route[m0 + min(r0 + i * rstep, rows_here - 1)];
    }
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int row = r0 + i * rstep;
      if (row >= rows_here || !col_ok) continue;
      u32x4 v = lds_ld128(stage + (uint32_t)((row * sld + ch * 8) * 2));
      const int64_t orow = GROUPED ? (int64_t)route[GROUPED ? i : 0] : m0 + row;
      const int64_t o = orow * ldy + col0 + ch * 8;
      if (a.epilogue == TNX_EPI_RESIDUAL) {
        const u32x4 res = *reinterpret_cast<const u32x4*>(a.residual + o);
#pragma unroll
        for (int q = 0; q < 4; ++q) v[q] = pack2bf(bflo(v[q]) + bflo(res[q]), bfhi(v[q]) + bfhi(res[q]));
      }
      *reinterpret_cast<u32x4*>(y + o) = v;
    }
  }
}

}  // namespace
