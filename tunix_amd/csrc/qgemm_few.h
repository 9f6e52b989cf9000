// The quantised GEMM over at most 32 rows, or 64 of a few k-tiles (a decode batch): one work-group = 8 waves = ROWS (8, 16, 32 or 64) rows x 128 columns of one k split, a
// wave a column tile of 16 over the whole of it.
//
// What bounds it is the launch and the round trip to memory, then the conversion of the codes: five instructions per pair of weights and lane
// (address, look-up, two products, rounding; by counters over 4096 -> 28672 and 16 rows 5.1 of the vector unit and 1.3 of
// LDS, the vector unit at work for 49 % of the launch's cycles), of which a compute unit finishes a k-tile (8192 pairs) in 0.36 us or so, looked up, converted and
// multiplied, where vector instructions alone would take 0.28; 4096 -> 28672 has 32 of them per unit, 11.5 of its 18 us, and its 62 MB of codes
// and scales take some 11 us.  So:
//   * the activations, which all waves share, are requested once, as whole kilobytes straight into LDS, ahead of everything else.  (As fragments
//     from memory, 16 bytes of 16 rows a load, they come at a third of that rate and once per wave: the first loads of 4096 -> 28672 over 16 rows
//     took 6 us to be asked for, now 2.)  There is no barrier in the loop as long as LDS holds them, up to 12 to 80 k-tiles by rows and code book;
//   * a wave has a column tile of its own over the whole k range: no sums to exchange, and little code (9 to 10 KB up to 16 rows; a work-group's first pass over its
//     instructions is part of every launch: the same kernel with six k-tiles in flight and a copy of the loop for the tiles left, 22 KB, is
//     0.5 to 1 us slower at every size, with three tiles or two at long contractions 0.2 and 5 us).
// us, before (activations as fragments from memory, or through LDS behind a barrier per k-tile) | now, weights from HBM, NF4 of group 64 with an
// adapter of rank 64, splits without the pass that sums them:
//                                   1 row        8 rows       16 rows       32 rows
//   4096 -> 6144 in 5           8.5 |  6.6    9.1 |  6.7    9.4 |  7.1    9.9 |  8.6
//   4096 -> 4096 in 8           7.5 |  5.4    7.7 |  5.6    7.8 |  5.8    8.3 |  6.9
//   4096 -> 28672 gated        18.8 | 17.8   20.2 | 18.5   20.7 | 18.8   24.7 | 22.5
//   14336 -> 4096 in 8         11.3 |  9.4   12.1 |  9.9   13.2 | 10.2   14.2 | 12.5
//   int4 1152 -> 13824 gated    8.4 |  7.6    9.8 |  7.6    9.9 |  7.8   10.4 |  9.0
//   int4 1024 -> 1152 in 8      5.0 |  3.3    5.2 |  3.7    5.2 |  3.9    5.5 |  4.7
// Over 94 shapes (20 contractions x 5 forms of code book, group and adapter) the geometric mean is 0.80 at 1 to 16 rows and 0.88 at 17 to 32, and
// none is slower but contractions of 64 k-tiles on eight work-groups (8192 -> 1024 unsplit, which the decoder splits: 27.4 | 29.3).  33 to 64 rows:
// few_shape in qlinear.hip.
// Also slower: sixteen waves with half a k-tile each (4096 -> 28672 over one row 23.0 us), column tiles in pairs over half of the k-tiles (the
// sums meet: 4096 -> 4096 in 8 6.1).
//
// Included by qlinear.hip after qgemm128.h.
#pragma once

namespace {

// LDS: the activations of a work-group's k-tiles lie in slots of ROWS * 256 bytes from address 0 on, around the table of the code book (64 KiB to
// 128 KiB; integer codes have none).  Behind the loop the sums of gated columns meet at 128 KiB, the activated tile leaves through the table's place.
constexpr uint32_t kFewLds = 160u << 10, kFewMeet = 0x20000, kFewOut = 0x10000, kFewScratch = 0x14000;

// INNER: the adapter's down-projection t = x . A is formed here (a.inner_a, its fragments in order) instead of ahead of the launch: a work-group
// multiplies the activations it holds with its k range of A (wave (rank tile, half of each k-tile): the fragments of x are there already), and its share
// of t, as a pair of bf16 (to 2^-17 of itself), with B: t is linear, so no sum over the splits has to be waited for, nor is one rounded to bf16 on the
// way (against 64 bits 6e-7 of the result where a rounded t gave 4e-4).  us, down-projection and this kernel in two launches | in one, 16 rows, rank 64:
// 4096 -> 4096 in 8 10.7 | 7.2, 14336 -> 4096 in 8 20.0 | 13.1, int4 1024 -> 1152 in 8 7.6 | 4.4, 2048 -> 4096 unsplit 13.8 | 12.9; 32 rows 11.9 | 8.2,
// 22.5 | 15.8, 8.6 | 5.0, 16.4 | 15.0.  (The fragments of A are 16 KB a k-tile and work-group, from the L2, next to 9 of codes and scales: a pair of
// adapters over a long unsplit range, gate | up's, would be a megabyte for each.)
// SHORT: at most PF k-tiles per split, none of them asked for in vain.  (A load that is not needed still takes its turn in the memory pipe; with the
// adapter's there are twice as many: 1024 -> 1152 in 8, one k-tile each, 5.8 -> 4.1 us with the adapter inside, 4096 -> 4096 in 8 7.7 -> 6.9; without
// it the waits behind the branches cost as much as the loads, 1152 -> 1536 in 5 3.5 | 3.7.)
// WHOLE: rows of x are whole 16-byte pieces, as loads straight into LDS ask for; otherwise they go by way of registers.  (A form of its own: as a branch
// beside those loads it costs every launch 0.2 us, 0.9 % of a rollout of 16 rows.)
typedef uint32_t u32x4_any __attribute__((ext_vector_type(4), aligned(2)));
// MERGE: x is what a decode step's attention left of its key chunks (attn_parts.h), merged here on its way to LDS: a launch less, for a read of the
// partials per column of work-groups and some hundred instructions a wave.  us a layer, with the merging pass | merged here: 32 heads of 128 on 8,
// 4 k-tiles a split: 1 row x 600 keys (5 chunks) 71.0 | 66.1, 2 x 800 (7) 69.2 | 66.9, 3 x 2940 (10) 77.8 | 74.4, 8 x 400 (4) 72.2 | 70.1, 16 x 700 (2) 80.9 | 79.4;
// 4 heads of 256 on one, one k-tile: 1 x 600 (5) 48.4 | 46.4, 16 x 1200 (10) 51.3 | 50.2.  Beyond kMergeBytes of partials a work-group (qlinear.hip) or
// kMergeChunks chunks, which would take a second round trip, nothing is left of it.
constexpr int kMergeChunks = 12;
template <int SPT, bool INT4, int ROWS, bool INNER, bool SHORT, bool WHOLE, bool MERGE>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void qgemm_few_kernel(const QLArgs a) {
  constexpr int MT = (ROWS + 15) / 16;
  constexpr uint32_t SLOT = ROWS * 256;
  constexpr int SLOTS = (int)((kFewLds - (INT4 ? 0u : (uint32_t)kBigLutBytes)) / SLOT);
  constexpr int PF = 4;                        // k-tiles in flight: a turn of the ring
  constexpr int TURNS = SLOTS >= 24 ? 2 : 1, CHUNK = TURNS * PF;   // turns, k-tiles whose slots are filled again together
  constexpr int NB = SLOTS / CHUNK;            // chunks that LDS holds
  static_assert((SHORT ? NB >= 1 : NB >= 2 && NB * CHUNK == SLOTS) && 8 * MT * 1024 <= kFewLds - kFewMeet, "LDS");
  constexpr int SW = SPT / 2;                  // dwords of scales per column and k-tile
  extern __shared__ __align__(16) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
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
  const int kt_end = min(ktiles, kt_begin + a.ktiles_per_split), n = max(kt_end - kt_begin, 0);
  const uint64_t ntk = (uint64_t)ntiles * ktiles;

  // Per-lane offsets (32 bit: the host checks the 4 GiB limits); the k-tile enters as the scalar offset of a load.  Rows past M
  // and column tiles past N start beyond the buffer and read zeros.
  const int64_t my_tile = (int64_t)blockIdx.y * 8 + wv;
  const uint32_t tile0 = (uint32_t)my_tile * (uint32_t)ktiles;
  const uint32_t coff = tile0 * 1024u + (uint32_t)lane * 16u, soff = (tile0 * 16u + (uint32_t)lm) * (uint32_t)(SPT * 2);
  u32x4 rc[PF], ra[PF][2];
  uint32_t rs[PF][SW];
  const int a_tile = wv & 3, a_half = wv >> 2, a_tiles = a.lora_rank / 16;
  const uint32_t aoff = (uint32_t)(a_half * 2 * a_tiles + a_tile) * 1024u + (uint32_t)lane * 16u;
  constexpr int LOADS = INNER ? 4 : 2;   // per k-tile and wave
  // (a k-tile past the last one is asked of an empty buffer: zeros, and no traffic)
  auto load_w = [&](int d, int kt) {
    const bool live = kt < kt_end;
    const rsrc_t qc = make_rsrc(a.codes, live ? ntk * 1024 : 0);
    const rsrc_t qs = make_rsrc(a.scales, live ? ntk * 16 * SPT * 2 : 0);
    rc[d] = __builtin_amdgcn_raw_buffer_load_b128(qc, coff, kt * 1024, kStreamOnce);
    if constexpr (SW == 1) {
      rs[d][0] = __builtin_amdgcn_raw_buffer_load_b32(qs, soff, kt * (16 * SPT * 2), 0);
    } else {
      const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(qs, soff, kt * (16 * SPT * 2), 0);
      rs[d][0] = v[0];
      rs[d][1] = v[1];
    }
    if constexpr (INNER) {
      const rsrc_t qa = make_rsrc(a.inner_a, live && a_tile < a_tiles ? (uint64_t)a.K * a.lora_rank * 2 : 0);
#pragma unroll
      for (int j = 0; j < 2; ++j) ra[d][j] = __builtin_amdgcn_raw_buffer_load_b128(qa, aoff + (uint32_t)(j * a_tiles) * 1024u, kt * 4 * a_tiles * 1024, 0);
    }
  };
  // Activations go from memory straight into LDS, a wave's 64 lanes 1 KB = four rows of a k-tile: chunk p of row r is k-chunk p ^ (r % 16), so
  // that the rows a fragment is read from hit different banks.
  constexpr int QUADS = ROWS / 4, QW = QUADS > 8 ? QUADS / 8 : 1;   // quads of rows per k-tile, and of them per wave
  const u32x4 rx = raw_rsrc(a.x, (uint64_t)a.M * a.K * 2);
  const int quad = wv % QUADS, xrow = quad * 4 + (lane >> 4);
  const uint32_t xvoff = ((uint32_t)xrow * (uint32_t)a.K + (uint32_t)((lane & 15) ^ (xrow & 15)) * 8u) * 2u;
  // k-tiles first .. first + count of this work-group into the slots from `slot` on
  auto request_x = [&](int first, int count, int slot) {
#pragma unroll(WHOLE ? 1 : 4)
    for (int i = wv / QUADS; i < count; i += QW > 1 ? 1 : 8 / QUADS) {
      const uint32_t at = (uint32_t)(slot + i) * SLOT;
#pragma unroll
      for (int q = 0; q < QW; ++q) {
        const uint32_t lds = (INT4 || at < kBigLutBase ? at : at + (uint32_t)kBigLutBytes) + (uint32_t)(quad + 8 * q) * 1024u;
        const uint32_t voff = xvoff + (uint32_t)(32 * q) * (uint32_t)a.K * 2u, koff = (uint32_t)(kt_begin + first + i) * (KTILE * 2);
        if constexpr (WHOLE) {
          dma16(lds, rx, voff, (int)koff);
        } else {
          u32x4 v = {0, 0, 0, 0};
          if (xrow + 32 * q < a.M) v = *reinterpret_cast<const u32x4_any*>(reinterpret_cast<const char*>(a.x) + ((uint64_t)voff + koff));
          lds_st128(lds + (uint32_t)lane * 16u, v);
        }
      }
    }
  };
  // The same from partials: a thread takes eight columns of a row of a k-tile, U such pieces at a time, all of its chunks at once, NC of them at most.  (Vector
  // instructions are what it costs, some 0.3 us per hundred of a wave: few, and no rows or chunks that are not there.)
  auto merge_x = [&](auto Uc, auto NCc) {
    constexpr int U = decltype(Uc)::value, NC = decltype(NCc)::value;
    const uint32_t C = (uint32_t)a.parts_n, dh = 1u << a.parts_shift, pitch = (dh + kPartPad) * 4u, heads = (uint32_t)(a.K >> a.parts_shift);
    const uint32_t pieces = (uint32_t)a.M * (uint32_t)n * 16u;
    const rsrc_t rp = make_rsrc(a.parts, (uint64_t)a.M * heads * C * pitch);
    for (uint32_t e0 = (uint32_t)tid; e0 < pieces; e0 += 512u * U) {
      uint32_t at[U], off[U], to[U];
      u32x2 ml[U][NC];
      u32x4 v[U][NC][2];
#pragma unroll
      for (int k = 0; k < U; ++k) {
        const uint32_t e = e0 + 512u * k, row = n == 1 ? e >> 4 : n == 2 ? e >> 5 : n == 4 ? e >> 6 : e / 48u, i = (e >> 4) - row * (uint32_t)n, p = e & 15u;
        const uint32_t col = ((uint32_t)kt_begin + i) * KTILE + p * 8u;
        at[k] = e < pieces ? (row * heads + (col >> a.parts_shift)) * (C * pitch) : 0xf0000000u;
        off[k] = at[k] + (kPartPad + (col & (dh - 1u))) * 4u;
        const uint32_t slot = i * SLOT;
        to[k] = (INT4 || slot < kBigLutBase ? slot : slot + (uint32_t)kBigLutBytes) + row * 256u + (p ^ (row & 15u)) * 16u;
#pragma unroll
        for (int c = 0; c < NC; ++c)
          if (c < (int)C) {
            ml[k][c] = __builtin_amdgcn_raw_buffer_load_b64(rp, at[k], (int)(c * pitch), 0);
#pragma unroll
            for (int h = 0; h < 2; ++h) v[k][c][h] = __builtin_amdgcn_raw_buffer_load_b128(rp, off[k] + 16u * h, (int)(c * pitch), 0);
          }
      }
#pragma unroll
      for (int k = 0; k < U; ++k) {
        float top = kNegBig, L = 0.0f, o[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = 0.0f;
#pragma unroll
        for (int c = 0; c < NC; ++c)
          if (c < (int)C) top = __uint_as_float(ml[k][c][1]) != 0.0f ? fmaxf(top, __uint_as_float(ml[k][c][0])) : top;
#pragma unroll
        for (int c = 0; c < NC; ++c)
          if (c < (int)C) {
            const float l = __uint_as_float(ml[k][c][1]);
            if (l != 0.0f) {   // (a chunk without a key: an O nobody wrote)
              const float w = __expf(__uint_as_float(ml[k][c][0]) - top);
              L += w * l;
#pragma unroll
              for (int e = 0; e < 8; ++e) o[e] += w * __uint_as_float(v[k][c][e >> 2][e & 3]);
            }
          }
        if (e0 + 512u * k < pieces) {
          // o / L: the quotient by a reciprocal, corrected by its remainder.  An infinite o has none (inf - inf): the maximum makes a finite number of it, and the
          // quotient stays infinite
          const float inv = L != 0.0f ? 1.0f / L : 0.0f;
          u32x4 x;
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float t = o[e] * inv, rest = fmaxf(__builtin_fmaf(-t, L, o[e]), -3.0e38f);
            o[e] = __builtin_fmaf(rest, inv, t);
          }
#pragma unroll
          for (int e = 0; e < 4; ++e) x[e] = pack2bf(o[2 * e], o[2 * e + 1]);
          lds_st128(to[k], x);
        }
      }
    }
  };
  if constexpr (!MERGE) request_x(0, min(n, NB * CHUNK), 0);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int d = 0; d < PF; ++d)
    if (!SHORT || d < n) load_w(d, kt_begin + d);
  __builtin_amdgcn_sched_barrier(0);

  // the adapter segment of this wave's columns
  int toff = 0;
  if (a.lora_rank > 0) {
    if (a.lora_nseg < 0) {   // interleaved gate / up pair: even tiles segment 0, odd tiles segment 1
      toff = (wv & 1) * a.lora_rank;
    } else {
      // (N < 2^31: the host checks the 4 GiB limits; opaque copies, or the selects are folded back into loads from the arguments)
      int e0 = (int)a.lora_seg_end[0], e1 = (int)a.lora_seg_end[1], e2 = (int)a.lora_seg_end[2];
      int t0 = a.lora_seg_toff[0], t1 = a.lora_seg_toff[1], t2 = a.lora_seg_toff[2], t3 = a.lora_seg_toff[3];
      asm volatile("" : "+s"(e0), "+s"(e1), "+s"(e2), "+s"(t0), "+s"(t1), "+s"(t2), "+s"(t3));
      const int col = (int)min(my_tile, ntiles - 1) * 16;
      toff = t0;
      toff = a.lora_nseg > 1 && col >= e0 ? t1 : toff;
      toff = a.lora_nseg > 2 && col >= e1 ? t2 : toff;
      toff = a.lora_nseg > 3 && col >= e2 ? t3 : toff;
    }
  }
  if constexpr (!INT4) fill_level_table<512>(kBigLutBase, tid);   // while the first loads are in flight
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (MERGE) {   // (parts_n <= kMergeChunks: tnx_qlinear_merged_ok)
    static_assert(SHORT && INNER, "all k-tiles in LDS at once");
    if (a.parts_n <= 4 && a.M * n > 32) merge_x(ic<2>{}, ic<4>{});
    else merge_x(ic<1>{}, ic<kMergeChunks>{});
  }
  // the activations, requested ahead of the ring's weights
  if (MERGE) {
    // (they are in registers and stored)
  } else if (!SHORT || n >= 4) tnx_wait_vm(4 * LOADS);
  else if (n == 3) tnx_wait_vm(3 * LOADS);
  else if (n == 2) tnx_wait_vm(2 * LOADS);
  else tnx_wait_vm(LOADS);
  static_assert(PF == 4, "the waits above");
  __syncthreads();
  // the adapter's fragments of this wave's columns, and those of the next linear's adapter: asked for here, needed last
  const bool lora = a.lora_rank > 0 && (INNER || blockIdx.z == 0), lora_fast = lora && a.lora_rank <= 64;
  u32x4 lb[2], tf[MT][2], bn[2];
  if (lora_fast) {
    const rsrc_t rb = make_rsrc(a.lora_b, (uint64_t)a.N * a.lora_rank * 2), rt = make_rsrc(a.t, (uint64_t)a.M * a.t_ld * 2);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const bool on = j * 32 < a.lora_rank;
      const uint32_t ko = (uint32_t)(j * 32 + lq * 8);
      lb[j] = buf_load128(rb, on ? (((uint32_t)my_tile * 16u + (uint32_t)lm) * (uint32_t)a.lora_rank + ko) * 2u : 0xfffffff0u);
#pragma unroll
      for (int m = 0; m < MT; ++m)
        if constexpr (!INNER) tf[m][j] = buf_load128(rt, on ? ((uint32_t)(m * 16 + lm) * (uint32_t)a.t_ld + (uint32_t)toff + ko) * 2u : 0xfffffff0u);
    }
  }
  if (MT == 1 && a.next_tpart && wv < 4) {
    const rsrc_t rn = make_rsrc(a.next_a_t, (uint64_t)a.next_rank * a.N);
#pragma unroll
    for (int j = 0; j < 2; ++j) bn[j] = buf_load128(rn, next_a_off(a, wv, j, lm, lq));
  }
  __builtin_amdgcn_sched_barrier(0);

  f32x4 acc[MT], tacc[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    zero_acc(acc[m]);
    zero_acc(tacc[m]);
  }
  // LDS address of this lane's activation fragment of k-step 0 in a slot; k-step j lies 64 j bytes away under XOR, row tile m 4096 m bytes on.
  // (Rows past the slot's read others: what they give stays in rows past M.)
  const uint32_t xrd = (uint32_t)(lm % ROWS) * 256u + (uint32_t)(lq ^ (lm % ROWS)) * 16u;
  // Entries of the code dwords (four code bytes: eight weights of a column, one k-step) are looked up kAhead dwords before the dword is
  // converted, one at a time between the conversions: the LDS pipe takes an entry in two cycles and gets one of every wave in some
  // sixteen; the counter of LDS accesses tells fifteen apart.
  constexpr int kAhead = 3;
  uint32_t lp[kAhead + 1][4];
  u32x4 xf[2][MT];
  auto entry_addr = [&](uint32_t w, int i) -> uint32_t { return INT4 ? 0u : __builtin_amdgcn_perm(w, lane_off, 0x0c020400u + ((uint32_t)i << 8)); };
  auto entry = [&](uint32_t w, uint32_t at, int i) -> uint32_t {
    if constexpr (INT4) return int4_entry(magic, w, i);
    else return lds_ld32(at);
  };
  auto read_x = [&](u32x4 (&to)[MT], uint32_t slot, int j) {
#pragma unroll
    for (int m = 0; m < MT; ++m) to[m] = lds_ld128(((xrd + slot) ^ (uint32_t)(j * 64)) + (uint32_t)(m * 4096));
  };
  int kt = kt_begin;
  uint32_t here = 0;   // LDS address of the k-tile's slot
  auto tile = [&](auto Dc) {   // one k-tile, of ring stage d
    constexpr int d = decltype(Dc)::value, dn = (d + 1) % PF;
    uint32_t next = here + SLOT;
    if (!INT4) next = next == kBigLutBase ? kBigLutBase + (uint32_t)kBigLutBytes : next;
    next = next == (uint32_t)(NB * CHUNK) * SLOT + (INT4 ? 0u : (uint32_t)kBigLutBytes) ? 0 : next;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t ahead = j + kAhead < 4 ? rc[d][(j + kAhead) & 3] : rc[dn][(j + kAhead) & 3];
      const uint32_t sw = rs[d][SPT == 2 ? 0 : j >> 1];
      const float s = (SPT == 2 ? j >> 1 : j & 1) ? bfhi(sw) : bflo(sw);
      uint32_t (&now)[4] = lp[(j + 4 * d) % (kAhead + 1)], (&later)[4] = lp[(j + 4 * d + kAhead) % (kAhead + 1)];
      u32x4 q;
      // two pairs at a time, an instruction between each and what needs its result
#pragma unroll
      for (int b = 0; b < 4; b += 2) {
        const uint32_t at0 = entry_addr(ahead, b), at1 = entry_addr(ahead, b + 1);
        _Float16 l0, l1, h0, h1;
        level_pair<INT4>(now, b, l0, l1);
        level_pair<INT4>(now, b + 1, h0, h1);
        __builtin_amdgcn_sched_barrier(0);
        const float p0 = __builtin_fmaf((float)l0, s, 0.0f), p1 = __builtin_fmaf((float)l1, s, 0.0f);
        later[b] = entry(ahead, at0, b);
        __builtin_amdgcn_sched_barrier(0);
        const float r0 = __builtin_fmaf((float)h0, s, 0.0f), r1 = __builtin_fmaf((float)h1, s, 0.0f);
        later[b + 1] = entry(ahead, at1, b + 1);
        __builtin_amdgcn_sched_barrier(0);
        if (b == 0) read_x(xf[(j + 1) & 1], j < 3 ? here : next, (j + 1) & 3);
        q[b] = cvt_pk_bf16(p0, p1);
        q[b + 1] = cvt_pk_bf16(r0, r1);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int m = 0; m < MT; ++m) acc[m] = mfma16(xf[j & 1][m], q, acc[m]);
      if (INNER && a_half == j >> 1)
#pragma unroll
        for (int m = 0; m < MT; ++m) tacc[m] = mfma16(xf[j & 1][m], ra[d][j & 1], tacc[m]);
    }
    here = next;
  };
  static_assert(PF * 4 % (kAhead + 1) == 0, "a turn of the ring is whole turns of the look-ups");
  auto turn = [&](auto self, auto Dc) -> void {
    constexpr int d = decltype(Dc)::value;
    if constexpr (d < PF) {
      if (kt < kt_end) tile(Dc);   // (its loads, unconditional, stand behind it: the compiler's counted waits stay exact)
      if constexpr (!SHORT) {
        load_w(d, kt + PF);
        __builtin_amdgcn_sched_barrier(0);
      }
      ++kt;
      self(self, ic<d + 1>{});
    }
  };
  read_x(xf[0], 0, 0);
#pragma unroll
  for (int w = 0; w < kAhead; ++w)
#pragma unroll
    for (int b = 0; b < 4; ++b) lp[w][b] = entry(rc[0][w], entry_addr(rc[0][w], b), b);
  __builtin_amdgcn_sched_barrier(0);
  // Where LDS does not hold the activations of all k-tiles, the end of chunk c frees its slots for those of chunk c + NB, which have NB - 1 chunks
  // to arrive in: the loads of those are the ones that may still be in flight at the wait.
  if constexpr (SHORT) turn(turn, ic<0>{});
  for (int c = 0, into = 0; !SHORT && kt < kt_end; ++c) {
#pragma unroll 1
    for (int t = 0; t < TURNS; ++t) turn(turn, ic<0>{});
    const int left = n - (c + NB) * CHUNK;   // k-tiles behind the chunks that are there
    if (n > NB * CHUNK && (left > 0 || c + 1 >= NB)) {
      constexpr int kYounger = (NB - 1) * CHUNK * LOADS;
      tnx_wait_vm(kYounger < 60 ? kYounger : 60);
      __syncthreads();
      if (left > 0) request_x((c + NB) * CHUNK, min(CHUNK, left), into);
      into = into + CHUNK == NB * CHUNK ? 0 : into + CHUNK;
      read_x(xf[0], here, 0);   // (what the chunk before read may not have been there)
    }
  }
  if constexpr (INNER) {
    // the shares of t meet as rows in LDS, padded by four ranks
    constexpr uint32_t T_LD = 68 * 4, T_HALF = 16 * MT * T_LD, T_AT = 2 * T_HALF <= kFewLds - kFewMeet ? kFewMeet : 0;
    static_assert(2 * T_HALF <= kBigLutBase, "LDS");
    if (T_AT == 0 || (uint32_t)n * SLOT > (INT4 ? kFewMeet : kBigLutBase)) __syncthreads();   // (activations lie there)
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float v = tacc[m][i];
        *reinterpret_cast<lds_u32*>(static_cast<uintptr_t>(T_AT + (uint32_t)a_half * T_HALF + (uint32_t)(m * 16 + lq * 4 + i) * T_LD +
                                                           (uint32_t)(a_tile * 16 + lm) * 4u)) = __float_as_uint(v);
      }
    __syncthreads();
    f32x4 part[MT];
    u32x4 hi[MT][2];
    float all = 0.0f;
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      zero_acc(part[m]);
#pragma unroll
      for (int j = 0; j < 2; ++j) {   // (ranks past the adapter's are zeros: nothing was asked for them, neither of A nor of B)
        const uint32_t at = T_AT + (uint32_t)(m * 16 + lm) * T_LD + (uint32_t)(j * 32 + lq * 8) * 4u;
        u32x4 lo;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const f32x4 v = __builtin_bit_cast(f32x4, lds_ld128(at + h * 16u)) + __builtin_bit_cast(f32x4, lds_ld128(at + T_HALF + h * 16u));
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            hi[m][j][2 * h + i] = cvt_pk_bf16(v[2 * i], v[2 * i + 1]);
            lo[2 * h + i] = cvt_pk_bf16(v[2 * i] - bflo(hi[m][j][2 * h + i]), v[2 * i + 1] - bfhi(hi[m][j][2 * h + i]));
          }
        }
        part[m] = mfma16(lo, lb[j], part[m]);
        part[m] = mfma16(hi[m][j], lb[j], part[m]);
      }
      all += (part[m][0] + part[m][1]) + (part[m][2] + part[m][3]);
    }
    // Where t is infinite, or past the largest bf16, the lower of the pair undoes it (and zeros past 32 ranks, times an infinite x, are none): what
    // came out as no number is then what the uppers give.  (A branch: testing the
    // lowers one by one is 128 instructions a wave at 64 rows, 1.2 % of a rollout of Gemma3-1B where this is 0.5.)
    if (__builtin_amdgcn_ballot_w64(all != all) != 0) {
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        f32x4 upper;
        zero_acc(upper);
        upper = mfma16(hi[m][0], lb[0], upper);
        if (a.lora_rank > 32) upper = mfma16(hi[m][1], lb[1], upper);
#pragma unroll
        for (int i = 0; i < 4; ++i) part[m][i] = part[m][i] != part[m][i] ? upper[i] : part[m][i];
      }
    }
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[m][i] += a.lora_scale * part[m][i];
  } else if (lora_fast) {
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      f32x4 part;
      zero_acc(part);
#pragma unroll
      for (int j = 0; j < 2; ++j) part = mfma16(tf[m][j], lb[j], part);
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[m][i] += a.lora_scale * part[i];
    }
  } else if (lora) {
    TileSrc s;
    s.M = a.M; s.K = a.K; s.x = a.x; s.row_index = nullptr; s.row_div = 1; s.x_rows = a.M;
    s.w_bf16 = nullptr; s.codes = a.codes; s.scales = a.scales; s.group = a.group; s.qtype = a.qtype;
    s.ntiles = ntiles; s.lora_rank = a.lora_rank; s.t = a.t; s.t_ld = a.t_ld; s.lora_b = a.lora_b;
    s.lora_scale = a.lora_scale;
    f32x4 out[MT][1];
#pragma unroll
    for (int m = 0; m < MT; ++m) out[m][0] = acc[m];
    const int toffs[1] = {toff};
    tile_lora<MT, 1>(s, 0, my_tile, toffs, out);
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[m] = out[m][0];
  }
  const bool mul = a.epilogue == TNX_EPI_SILU_MUL || a.epilogue == TNX_EPI_GELU_MUL;
  if (MT < 4 && (!mul || a.split_k > 1)) {
    // The planes of a split are stored as they lie in the accumulators and without the non-temporal policy: with it the pass that sums them waits
    // longer than this one gains (14336 -> 4096 in 8 splits, 8 rows, with that pass: 16.1 us against 17.0, 4096 -> 4096 in 8: 11.6 against 12.5).
    f32x4 out[MT][1];
#pragma unroll
    for (int m = 0; m < MT; ++m) out[m][0] = acc[m];
    store_tile<MT, 1>(a, 0, a.M, my_tile, ntiles, out, [](int64_t r) { return r; });
    return;
  }
  // Gate and up columns meet, and the rows of a plane of many rows (whole lines of 128 bytes instead of four-byte stores: 4096 -> 4096 in 8 over 64 rows
  // 9.5 -> 8.8 us): every wave leaves its sums and takes the two column tiles and the row tiles it finishes.
  __syncthreads();   // (activations and table lie there)
#pragma unroll
  for (int m = 0; m < MT; ++m) lds_st128(kFewMeet + (uint32_t)(wv * MT + m) * 1024u + (uint32_t)lane * 16u, __builtin_bit_cast(u32x4, acc[m]));
  __syncthreads();
  constexpr int HM = (MT + 1) / 2;
  const int wn = wv & 3, rh = wv >> 2;
  f32x4 out[HM][2];
  if (MT > 1 || rh == 0) {
#pragma unroll
    for (int m = 0; m < HM; ++m)
#pragma unroll
      for (int nt = 0; nt < 2; ++nt)
        out[m][nt] = __builtin_bit_cast(f32x4, lds_ld128(kFewMeet + (uint32_t)((2 * wn + nt) * MT + rh * HM + m) * 1024u + (uint32_t)lane * 16u));
  }
  quant_rows_out<MT, 2, (MT >= 4), (MT == 1), 0>(a, out, 0, (int64_t)blockIdx.y * 8 + 2 * wn, wv, kFewOut, kFewScratch, bn);
}

}  // namespace
