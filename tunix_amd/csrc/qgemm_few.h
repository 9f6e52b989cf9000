// The quantised GEMM over at most 16 rows (a decode batch): one work-group = 8 waves = 16 rows x 128 columns of one k split, no
// barrier between its first and its last load.
//
// What bounds it is the round trip to memory, then the weight stream and the conversion of the codes (two lane-instructions per
// weight).  So nothing is shared between waves that would have to be waited for: of CW x KW = 8 waves, wave (ch, ks) takes 128 / CW
// columns over the k-tiles ks, ks + KW, ..., reads its activation fragments straight from memory (the rows of a decode batch live in the
// L2; rows past M cost nothing), keeps PF k-tiles in flight in registers, and the KW partial sums of a column meet in LDS once,
// at the end.  qgemm128_kernel shares the activations through LDS behind one barrier per k-tile: 24 KB per compute unit in flight and
// its waves in step; here it is 64 to 96 KB, and every wave runs on as its own data arrives.
// CW = 4: fewer sums to exchange, activations read four times over: for up to 8 rows.  CW = 2: twice over, for up to 16 rows and many
// k-tiles.  CW = 1 pays a microsecond for the exchange of 64 KB; at 32 rows the shared form wins everywhere.  Which calls come here:
// few_shape in qlinear.hip.  The planes of a split are stored as they lie in the accumulators and without the non-temporal policy:
// with it the pass that sums them waits longer than this one gains (14336 -> 4096 in 8 splits, 8 rows, with that pass: 16.1 us
// against 17.0, 4096 -> 4096 in 8: 11.6 against 12.5).
//
// Included by qlinear.hip after qgemm128.h.
#pragma once

namespace {

constexpr uint32_t few_out_base(bool int4, int cw) {
  return int4 ? 65536u / (uint32_t)cw : kBigLutBase + (uint32_t)kBigLutBytes;
}
constexpr size_t few_smem_bytes(bool int4, int cw) {
  return few_out_base(int4, cw) + 16 * kRowsActBytes;
}

template <int SPT, bool INT4, int CW>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void qgemm_few_kernel(const QLArgs a) {
  constexpr int CT = 8 / CW, KW = 8 / CW, NT = 2;
  constexpr int UC = CT < 4 ? CT : 4, UH = CT / UC;   // column tiles per unit of conversion, units per k-step
  constexpr int PF = CW == 4 ? 4 : 3;          // k-tiles in flight
  constexpr int SW = SPT / 2;                  // dwords of scales per column and k-tile
  extern __shared__ __align__(16) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6), ch = wv % CW, ks = wv / CW;
  const int lm = lane & 15, lq = lane >> 4;
  // the whole argument block in one batch of scalar loads (left alone, each field is one memory round trip next to its first use)
  asm volatile("" ::"s"(a.M), "s"(a.K), "s"(a.N), "s"(a.x), "s"(a.codes), "s"(a.scales), "s"(a.ktiles_per_split), "s"(a.lora_rank),
               "s"(a.lora_nseg), "s"(a.lora_seg_end[0]), "s"(a.lora_seg_end[1]), "s"(a.lora_seg_end[2]), "s"(a.lora_seg_toff[0]),
               "s"(a.lora_seg_toff[1]), "s"(a.lora_seg_toff[2]), "s"(a.lora_seg_toff[3]));
  asm volatile("" ::"s"(a.t_ld), "s"(a.t), "s"(a.lora_b), "s"(a.lora_scale), "s"(a.epilogue), "s"(a.y), "s"(a.split_k), "s"(a.ws),
               "s"(a.next_a_t), "s"(a.next_rank), "s"(a.next_tpart));
  const uint32_t lane_off = (uint32_t)lane * 4u | kBigLutBase;   // byte 2 = 1: the table's base
  Int4Magic magic;
  if constexpr (INT4) magic.pin<true>();
  const int64_t ntiles = a.N / 16;
  const int ktiles = (int)(a.K / KTILE);
  const int kt_begin = blockIdx.z * a.ktiles_per_split;
  const int kt_end = min(ktiles, kt_begin + a.ktiles_per_split);
  const uint64_t ntk = (uint64_t)ntiles * ktiles;
  const uint32_t xbytes = (uint32_t)a.M * (uint32_t)a.K * 2u;

  // Per-lane offsets (32 bit: the host checks the 4 GiB limits); the k-tile enters as the scalar offset of a load.  Rows past M
  // and column tiles past N start beyond the buffer and read zeros.
  uint32_t coff[CT], soff[CT];
  const uint32_t xoff = ((uint32_t)lm * (uint32_t)a.K + (uint32_t)lq * 8u) * 2u;
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) {
    const uint32_t tile0 = ((uint32_t)blockIdx.y * 8u + (uint32_t)(ch * CT + ct)) * (uint32_t)ktiles;
    coff[ct] = tile0 * 1024u + (uint32_t)lane * 16u;
    soff[ct] = (tile0 * 16u + (uint32_t)lm) * (uint32_t)(SPT * 2);
  }
  u32x4 rc[PF][CT], xf[PF][4];
  uint32_t rs[PF][CT][SW];
  // (a k-tile past the wave's last one is asked of an empty buffer: zeros, and no traffic)
  auto load_w = [&](int d, int kt) {
    const bool live = kt < kt_end;
    const rsrc_t qc = make_rsrc(a.codes, live ? ntk * 1024 : 0);
    const rsrc_t qs = make_rsrc(a.scales, live ? ntk * 16 * SPT * 2 : 0);
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) rc[d][ct] = __builtin_amdgcn_raw_buffer_load_b128(qc, coff[ct], kt * 1024, kStreamOnce);
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
      if constexpr (SW == 1) {
        rs[d][ct][0] = __builtin_amdgcn_raw_buffer_load_b32(qs, soff[ct], kt * (16 * SPT * 2), 0);
      } else {
        const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(qs, soff[ct], kt * (16 * SPT * 2), 0);
        rs[d][ct][0] = v[0];
        rs[d][ct][1] = v[1];
      }
    }
  };
  auto load_x = [&](int d, int j, int kt) {
    const rsrc_t q = make_rsrc(a.x, kt < kt_end ? xbytes : 0);
    xf[d][j] = __builtin_amdgcn_raw_buffer_load_b128(q, xoff + (uint32_t)(j * 64), kt * 256, 0);
  };
  const int kt0 = kt_begin + ks;
#pragma unroll
  for (int d = 0; d < PF; ++d) {
#pragma unroll
    for (int j = 0; j < 4; ++j) load_x(d, j, kt0 + d * KW);
    load_w(d, kt0 + d * KW);
  }
  __builtin_amdgcn_sched_barrier(0);

  // the adapter segment of the two column tiles this wave finishes
  const int wn = wv & 3;
  const int64_t ntile0 = ((int64_t)blockIdx.y * 4 + wn) * NT;
  int toff[NT] = {0, 0};
  if (a.lora_rank > 0) {
    if (a.lora_nseg < 0) {   // interleaved gate / up pair: even tiles segment 0, odd tiles segment 1
      toff[1] = a.lora_rank;
    } else {
      // (N < 2^31: the host checks the 4 GiB limits; opaque copies, or the selects are folded back into loads from the arguments)
      int e0 = (int)a.lora_seg_end[0], e1 = (int)a.lora_seg_end[1], e2 = (int)a.lora_seg_end[2];
      int t0 = a.lora_seg_toff[0], t1 = a.lora_seg_toff[1], t2 = a.lora_seg_toff[2], t3 = a.lora_seg_toff[3];
      asm volatile("" : "+s"(e0), "+s"(e1), "+s"(e2), "+s"(t0), "+s"(t1), "+s"(t2), "+s"(t3));
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        const int col = (int)min(ntile0 + nt, ntiles - 1) * 16;
        int t = t0;
        t = a.lora_nseg > 1 && col >= e0 ? t1 : t;
        t = a.lora_nseg > 2 && col >= e1 ? t2 : t;
        t = a.lora_nseg > 3 && col >= e2 ? t3 : t;
        toff[nt] = t;
      }
    }
  }
  // the adapter's fragments for the rows and columns this wave finishes: asked for here, needed last
  const bool has_rows = wv < 4;
  const bool lora = a.lora_rank > 0 && blockIdx.z == 0 && has_rows, lora_fast = lora && a.lora_rank <= 64;
  u32x4 lb[NT][2], tf[NT][2];
  if (lora_fast) {
    const rsrc_t rb = make_rsrc(a.lora_b, (uint64_t)a.N * a.lora_rank * 2), rt = make_rsrc(a.t, (uint64_t)a.M * a.t_ld * 2);
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const bool on = j * 32 < a.lora_rank;
        const uint32_t ko = (uint32_t)(j * 32 + lq * 8);
        lb[nt][j] = buf_load128(rb, on ? (((uint32_t)(ntile0 + nt) * 16u + (uint32_t)lm) * (uint32_t)a.lora_rank + ko) * 2u : 0xfffffff0u);
        tf[nt][j] = buf_load128(rt, on ? ((uint32_t)lm * (uint32_t)a.t_ld + (uint32_t)toff[nt] + ko) * 2u : 0xfffffff0u);
      }
  }
  if constexpr (!INT4) {
    fill_level_table<512>(kBigLutBase, tid);   // while the first loads are in flight
    __syncthreads();
  }

  f32x4 acc[CT];
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) zero_acc(acc[ct]);
  // one k-tile of ring stage d = four k-steps: the look-ups of the next step are issued before this step's codes are converted
  auto tile = [&](auto Dc, int kt) {
    constexpr int d = decltype(Dc)::value;
    uint32_t lp[2][UC][4];
    auto look = [&](int u) {
#pragma unroll
      for (int c = 0; c < UC; ++c)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const uint32_t w = rc[d][u % UH * UC + c][u / UH];
          if constexpr (INT4) lp[u & 1][c][i] = int4_entry(magic, w, i);
          else lp[u & 1][c][i] = lds_ld32(__builtin_amdgcn_perm(w, lane_off, 0x0c020400u + ((uint32_t)i << 8)));
        }
    };
    look(0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < 4 * UH; ++u) {
      const int j = u / UH;
      if (u + 1 < 4 * UH) look(u + 1);
#pragma unroll
      for (int c = 0; c < UC; ++c) {
        const int ct = u % UH * UC + c;
        const uint32_t sw = rs[d][ct][SPT == 2 ? 0 : j >> 1];
        const float s = (SPT == 2 ? j >> 1 : j & 1) ? bfhi(sw) : bflo(sw);
        u32x4 w;
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          _Float16 l0, l1;
          level_pair<INT4>(lp[u & 1][c], b, l0, l1);
          w[b] = cvt_pk_bf16(__builtin_fmaf((float)l0, s, 0.0f), __builtin_fmaf((float)l1, s, 0.0f));
        }
        acc[ct] = mfma16(xf[d][j], w, acc[ct]);
      }
      __builtin_amdgcn_sched_barrier(0);
      if (u % UH == UH - 1) load_x(d, j, kt + PF * KW);
      __builtin_amdgcn_sched_barrier(0);
    }
    load_w(d, kt + PF * KW);
    __builtin_amdgcn_sched_barrier(0);
  };
  // whole turns of the ring without a branch inside (behind one, the compiler's counted waits would assume that its loads never
  // happened), then the tiles left
  int kt = kt0;
  for (; kt + (PF - 1) * KW < kt_end; kt += PF * KW) {
    tile(ic<0>{}, kt);
    tile(ic<1>{}, kt + KW);
    tile(ic<2>{}, kt + 2 * KW);
    if constexpr (PF > 3) tile(ic<(PF > 3 ? 3 : 0)>{}, kt + 3 * KW);
  }
  if (kt < kt_end) {
    tile(ic<0>{}, kt);
    if (kt + KW < kt_end) {
      tile(ic<1>{}, kt + KW);
      if (PF > 3 && kt + 2 * KW < kt_end) tile(ic<2>{}, kt + 2 * KW);
    }
  }

  // The four k slices of a column meet: every wave leaves its sums, then takes the tiles it finishes from the four waves that hold
  // a share of them.
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) lds_st128((uint32_t)(wv * CT + ct) * 1024u + (uint32_t)lane * 16u, __builtin_bit_cast(u32x4, acc[ct]));
  __syncthreads();
  f32x4 out[1][NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) zero_acc(out[0][nt]);
  if (has_rows) {
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int k = 0; k < KW; ++k) {
        const uint32_t from = (uint32_t)((CW * k + 2 * wn / CT) * CT + (2 * wn) % CT + nt);
        out[0][nt] += __builtin_bit_cast(f32x4, lds_ld128(from * 1024u + (uint32_t)lane * 16u));
      }
  }
  if (lora_fast) {
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      f32x4 part;
      zero_acc(part);
#pragma unroll
      for (int j = 0; j < 2; ++j) part = mfma16(tf[nt][j], lb[nt][j], part);
#pragma unroll
      for (int i = 0; i < 4; ++i) out[0][nt][i] += a.lora_scale * part[i];
    }
  } else if (lora) {
    TileSrc s;
    s.M = a.M; s.K = a.K; s.x = a.x; s.row_index = nullptr; s.row_div = 1; s.x_rows = a.M;
    s.w_bf16 = nullptr; s.codes = a.codes; s.scales = a.scales; s.group = a.group; s.qtype = a.qtype;
    s.ntiles = ntiles; s.lora_rank = a.lora_rank; s.t = a.t; s.t_ld = a.t_ld; s.lora_b = a.lora_b;
    s.lora_scale = a.lora_scale;
    tile_lora<1, NT>(s, 0, ntile0, toff, out);
  }
  quant_rows_out<1, NT, false>(a, out, 0, ntile0, wv, few_out_base(INT4, CW), 0u);
}

}  // namespace
