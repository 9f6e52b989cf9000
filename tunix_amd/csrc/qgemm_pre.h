// The GEMM for many rows over weights that were converted once (tnx_qw_expand, tnx_dense_expand): output tile
// 16 * RT rows x 256 columns per work-group of four waves, a wave all rows x 64 columns.
//
// What bounds it is power: under MFMA load over random operands the part lowers its clock until its data movement
// and its matrix pipe fit, so the loop is built to move few bytes per multiplication.
//   * 16x16x32 MFMAs: they read and write an accumulator once per 32 k where 32x32x16 does once per 16.  The same
//     loop with 32x32x16 MFMAs kept the matrix pipe 81 % busy at 1.62 GHz, this one 75 % busy at 1.87 GHz: 1390 -> 1470 TFLOP/s
//     (16384 x 4096 -> 28672).  The MFMA is written in assembly with a tied accumulator: the
//     compiler's form gives source and destination registers of their own and spent 720 register copies per k-tile.
//   * RT = 16 (one work-group per compute unit, 256 accumulators): a wave's weights serve 256 rows, half the bytes from L2
//     per row of RT = 8 (two work-groups per unit), which is there for calls with too few tiles to fill the device.
//   * RT = 4 (three work-groups per unit) is for an lm_head over at most 64 rows, which is bound by the stream of its weights: the
//     MFMAs of 64 rows stay below that.  128256 x 4096 at 16 rows 203 -> 172 us
//     (1.05 GB: 6.1 TB/s with the finishing launch), 262144 x 1152 at 64 rows 143 -> 109 us, 151936 x 2048 at 64 rows 150 -> 120 us.
//     With two waves to a SIMD it is the form of all calls with no more tiles of 64 rows than units (launch_qgemm_pre).
//   * activations go from memory straight into LDS, in steps of 64 k (rows of 128 bytes, 16-byte chunks swizzled by row)
//     through four buffers, two steps ahead of their use and spread evenly over the loop: a burst of such loads would
//     stand between a weight fragment and the compiler's wait for it, which does not count them.
//   * weights come as fragments, kPreStages slabs of 32 k in registers.  The copy is laid out for 32x32x16 MFMAs
//     ([column tile][k-tile][wave][column group][16-deep slab][lane] x 16 bytes, lane l: column l % 32 of a group, k-group
//     l / 32 of the slab); a 16x16x32 fragment of columns 16 h .. +15 takes k-group lane / 16 of two slabs: from slab
//     (lane / 16) / 2, lane 32 ((lane / 16) % 2) + 16 h + lane % 16.
//   * products are formed transposed (weights as the A operand): a lane holds four consecutive output columns of one row.
//
// Measured on the Llama-3.1-8B linears with their adapters against the kernel of 32x32x16 MFMAs and 128-row tiles that was here
// before, us: 16384 rows: gate|up 3529 -> 2744, qkv 689 -> 594, o 485 -> 433, down 1553 -> 1347 (1.09-1.24 -> 1.27-1.43 PFLOP/s, without
// adapters up to 1.49; the library's product of the same operands alone 1.53-1.6); 2048 rows: 488 -> 368, 106 -> 86, 71 -> 61, 197 -> 177.
//
// Included by qlinear.hip after wide_out.h.
#pragma once

namespace {

constexpr int kPreStages = 4;
template <int RT>
constexpr uint32_t pre_step_bytes() { return 16 * RT * 128; }
// four step buffers, later the output stage
template <int RT>
constexpr size_t pre_smem_bytes() {
  return std::max<size_t>(4 * pre_step_bytes<RT>(), 16 * RT * (kWideCols + 8) * 2);
}

// (operands that loads have written: the wait for those is all it needs.  The compiler does not know that this is an MFMA and inserts no wait
// states between a copy of an operand and its use: that the built code has no such copy is checked in its listing,
// tests/test_mfma_wait_states.py)
__device__ __forceinline__ void mfma16_acc(u32x4 a, u32x4 b, f32x4& c) {
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
}
// the same for operands that vector instructions may just have written: the two wait states in front of it
__device__ __forceinline__ void mfma16_acc_wait(u32x4 a, u32x4 b, f32x4& c) {
  asm volatile("s_nop 1\n\tv_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
}
// keeps a value that was changed outside the loop in accumulator registers: the whole tile does not fit the others
__device__ __forceinline__ void pin_acc(f32x4& c) { asm volatile("" : "+a"(c)); }
// chunk swizzle of an LDS row: eight consecutive rows spread one k-chunk over all banks
__device__ __forceinline__ uint32_t pre_swizzle(uint32_t row) { return row & 7u; }

// GROUPED: one block of 16 * RT routes of one expert (in expert-sorted order) per work-group: the expert and the block within it
// are found from the expert offsets by a running sum; activation rows are gathered through sorted_route (row =
// route / x_div), output rows are routes.  No adapter, no lm_head statistics then.
// Work-group ids go round-robin to the eight XCDs: XCD x takes the x-th eighth of the tiles, in their order, so that what it
// works on at a time shares rows and columns in its L2 and the XCDs share no more than they must.  -1: no tile.  (With row
// blocks dealt out to the XCDs one by one, a call of 1024 rows had every weight read by all eight: 280 us against 198 for 1024 x
// 4096 -> 28672.)
__device__ __forceinline__ int xcd_tile(int id, int tiles) {
  const int x = id & 7, s = id >> 3, each = tiles >> 3, more = tiles & 7;
  return s < each + (int)(x < more) ? x * each + min(x, more) + s : -1;
}
// KIND, LORA: what happens to the finished tile, an instance each: with the forms as branches of one kernel the code between the
// loops of two tiles took 5 us longer.
enum PreKind { kPreStore, kPreF32, kPreRelu2, kPreSilu, kPreGelu, kPreSiluF32, kPreGeluF32, kPreHead, kPreHeadOnce };
// kPreHeadOnce: a head whose rows are one block: nobody else reads its weights, which are loaded with the non-temporal policy.  us with |
// without it, 128256 x 4096 over 128 rows 181 | 197, 262144 x 1152 123 | 136; with a second block of rows the weights come from L2 and the
// policy loses: 151936 x 2048 over 256 rows 194 | 183.
constexpr bool pre_head(int kind) { return kind == kPreHead || kind == kPreHeadOnce; }
// work-groups per unit, i.e. waves per SIMD
constexpr int pre_waves(int rt, int kind) { return rt == 16 ? 1 : rt == 4 && pre_head(kind) ? 3 : 2; }
constexpr bool pre_mul(int kind) { return kind == kPreSilu || kind == kPreGelu || kind == kPreSiluF32 || kind == kPreGeluF32; }

// LORA: 0 no adapter, kLoraInPlace: its scale is a power of two near one (1 where alpha is the rank): B times the scale is exact, and
// the delta is summed onto the accumulators directly; kLoraScaled: any scale.
constexpr int kLoraInPlace = 1, kLoraScaled = 2;

// sum over the lanes up to and with each one, by DPP: one, two, four, eight lanes on in a row of sixteen, the last lane of each row and of the lower half on
__device__ __forceinline__ int wave_scan(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);
  return v;
}

// The tile of row block mtile and column tile ntile.  CT: 16-column tiles of a wave, four, or two in a last column tile with at most 128
// columns (HALVES), which are divided among all four waves: half the MFMAs and weights of a whole tile, where two waves worked on columns that
// are not there.  us, 14322 rows 6912 -> 1152 214 | 184, 1024 -> 1152 44.1 | 39.5 (448 whole tiles and 112 halves on 512 places); 8000 rows of the
// second 29.9 | 26.4; where all fit in one turn (13000 rows) the same.  (The four waves by two halves of the rows, which reads the
// weights twice: 194.)
template <int RT, bool GROUPED, int KIND, int LORA, int CT>
__device__ __forceinline__ void pre_tile(const QLArgs& a, const WideHead& h, int mtile, int ntile, int expert, int m_from, int m_end) {
  constexpr int ROWS = 16 * RT, S = kPreStages, PASSES = RT / 2, HALF = RT / 4;   // PASSES: LDS loads of a step per thread
  constexpr uint32_t SB = pre_step_bytes<RT>();
  const int tid = threadIdx.x, lane = tid & 63;
  const int wn = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lm = lane & 15, lq = lane >> 4;
  const int tiles_n = (int)((a.N + kWideCols - 1) / kWideCols);
  // first row of the tile (GROUPED: first position in the sorted route list)
  const int64_t m0 = (int64_t)m_from + (int64_t)mtile * ROWS;
  const int rows_here = (int)min((int64_t)ROWS, (GROUPED ? (int64_t)m_end : a.M) - m0);
  const int ktiles = (int)(a.K / KTILE), ksteps = 2 * ktiles;
  const int64_t ntiles = a.N / 16, ntile0 = (int64_t)ntile * 16 + wn * CT;   // first 16-column tile of this wave

  // the activation resource starts at this work-group's first row: offsets stay small whatever M is, and rows past M
  // lie beyond the resource and read zeros (GROUPED: the whole buffer, rows are gathered)
  const u32x4 rx = GROUPED ? raw_rsrc(a.x, (uint64_t)(a.M / a.x_div) * a.K * 2)
                           : raw_rsrc(a.x + m0 * a.K, (uint64_t)rows_here * a.K * 2);
  const rsrc_t re = make_rsrc(a.w_pre + (GROUPED ? (int64_t)expert * tiles_n * ktiles * 32768 : 0),
                              (uint64_t)tiles_n * (uint64_t)ktiles * 65536u);
  // A step's rows in passes of 32: thread t fills chunk t % 8 of row t / 8 + 32 c and fetches for it the k-chunk
  // (t % 8) ^ swizzle(row)
  const uint32_t chs = (uint32_t)(lane & 7) ^ pre_swizzle((uint32_t)(tid >> 3));
  const uint32_t xbase = ((uint32_t)(tid >> 3) * (uint32_t)a.K + chs * 8u) * 2u, xstride = 32u * (uint32_t)a.K * 2u;
  const uint32_t dma_wave = (uint32_t)wn * 1024u;
  uint32_t xrow[GROUPED ? PASSES : 1];   // GROUPED: byte offsets of this thread's rows (rows the block does not have: beyond the buffer)
  if constexpr (GROUPED) {
    const bool whole_shift = (a.x_div & (a.x_div - 1)) == 0;   // (a division is some thirty instructions in front of the first load)
    const int x_shift = __builtin_ctz((uint32_t)a.x_div);
#pragma unroll
    for (int c = 0; c < PASSES; ++c) {
      const int r = (tid >> 3) + 32 * c;
      const uint32_t route = (uint32_t)a.sorted_route[m0 + min(r, rows_here - 1)], src = whole_shift ? route >> x_shift : route / (uint32_t)a.x_div;
      xrow[c] = r < rows_here ? (src * (uint32_t)a.K + chs * 8u) * 2u : 0xfffff000u;
    }
  }
  // (dma16 of gemm_tile.h: the compiler does not count these loads, the waits for them are written by hand)
  struct Src { u32x4 r; uint32_t base, stride; int soff; };   // a step's activations: resource, this thread's offset, row pass stride, k offset
  auto dma = [&](const Src& s, int c, uint32_t buf) {
    uint32_t off = 0;
    if constexpr (GROUPED) off = xrow[c];
    else off = s.base + (uint32_t)c * s.stride;
    dma16(buf + dma_wave + (uint32_t)c * 4096u, s.r, off, s.soff);
  };
  // steps 0 and 1 are requested ahead of the adapter bookkeeping below, which touches no memory
#pragma unroll
  for (int st = 0; st < 2; ++st)
#pragma unroll
    for (int c = 0; c < PASSES; ++c) dma(Src{rx, xbase, xstride, st * 128}, c, (uint32_t)st * SB);
  __builtin_amdgcn_sched_barrier(0);
  const uint32_t evoff = (uint32_t)(wn * (CT * 4096) + (lq >> 1) * 1024 + (lq & 1) * 512 + lm * 16);
  const int wt0 = ntile * ktiles;

  // LoRA: the two steps behind the last are the row block of t = bf16(x . A), columns [toff_a, +64) and [toff_b, +64) (the
  // host sends only shapes whose work-groups span at most two adapter segments here)
  int toff[CT];
  int toff_a = 0, toff_b = 0;
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) toff[ct] = 0;
  if constexpr (LORA != 0) {
    if (a.lora_nseg < 0) {
      toff_b = a.lora_rank;
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) toff[ct] = (ct & 1) * a.lora_rank;
    } else {
      int e0 = (int)a.lora_seg_end[0], e1 = (int)a.lora_seg_end[1], e2 = (int)a.lora_seg_end[2];
      int t0 = a.lora_seg_toff[0], t1 = a.lora_seg_toff[1], t2 = a.lora_seg_toff[2], t3 = a.lora_seg_toff[3];
      asm volatile("" : "+s"(e0), "+s"(e1), "+s"(e2), "+s"(t0), "+s"(t1), "+s"(t2), "+s"(t3));
      auto seg_idx = [&](int nt16) {
        const int col = nt16 * 16;
        return (int)(a.lora_nseg > 1 && col >= e0) + (int)(a.lora_nseg > 2 && col >= e1) +
               (int)(a.lora_nseg > 3 && col >= e2);
      };
      auto idx_toff = [&](int i) {
        auto pick = [](int cur, int cand, bool c) { return cur ^ ((cur ^ cand) & (0 - (int)c)); };
        return pick(pick(pick(t0, t1, i == 1), t2, i == 2), t3, i == 3);
      };
      const int last = (int)ntiles - 1;
      toff_a = idx_toff(seg_idx(min(ntile * 16, last)));
      toff_b = idx_toff(seg_idx(min(ntile * 16 + 15, last)));
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) toff[ct] = idx_toff(seg_idx(min((int)ntile0 + ct, last)));
    }
  }
  uint32_t tbase = 0;
  if constexpr (LORA != 0)   // (chunks past the rank: beyond the buffer, which reads zeros)
    tbase = (int)chs * 8 < a.lora_rank ? (uint32_t)((tid >> 3) * a.t_ld + toff_a + (int)chs * 8) * 2u : 0x80000000u;
  const u32x4 rt_ = LORA != 0 ? raw_rsrc(a.t + m0 * a.t_ld, (uint64_t)rows_here * a.t_ld * 2) : rx;
  const uint32_t tstride = (uint32_t)(32 * a.t_ld * 2);
  // B^T of the adapter: this lane's column of every tile, ranks 32 j + 8 (lane / 16) ..+7
  u32x4 lbv[CT][2];
#pragma unroll
  for (int ct = 0; ct < CT; ++ct)
#pragma unroll
    for (int j = 0; j < 2; ++j) lbv[ct][j] = u32x4{0, 0, 0, 0};
  auto load_adapter_b = [&]() {
    const rsrc_t rb = make_rsrc(a.lora_b, (uint64_t)a.N * a.lora_rank * 2);
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int j = 0; j < 2; ++j)
        if (j * 32 < a.lora_rank)
          lbv[ct][j] = buf_load128(rb, (((uint32_t)(ntile0 + ct) * 16u + (uint32_t)lm) * (uint32_t)a.lora_rank +
                                        (uint32_t)(j * 32 + lq * 8)) * 2u);
  };
  constexpr bool EARLY_B = RT == 16;   // (two work-groups per unit: no registers to park them in, and the other one covers their round trip)
  if constexpr (EARLY_B && LORA != 0) load_adapter_b();

  f32x4 acc[RT][CT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) zero_acc(acc[rt][ct]);
  u32x4 xf[RT];         // activation fragments of the current slab; a tile's is replaced by the next slab's behind its four MFMAs
  u32x4 wr[S][CT];      // weight fragments, slab % S
  // slab p (0 | 1) of a step: this lane's row lane % 16 of a tile (a row tile is an immediate), k-chunk 4 p + lane / 16;
  // flips between buffers 0 | 1 and 2 | 3
  uint32_t xaddr[2];
#pragma unroll
  for (int p = 0; p < 2; ++p) xaddr[p] = (uint32_t)lm * 128u + (((uint32_t)(4 * p + lq) ^ pre_swizzle((uint32_t)lm)) * 16u);

  // where the activations of a step come from
  auto source = [&](int step) -> Src {
    Src s{rx, xbase, xstride, min(step, ksteps - 1) * 128};
    if constexpr (LORA != 0) {   // (bit selects: a branch here would cut the loop into blocks)
      const uint32_t um = 0u - (uint32_t)(step >= ksteps);
#pragma unroll
      for (int i = 0; i < 3; ++i) s.r[i] ^= (rx[i] ^ rt_[i]) & um;
      s.base ^= (xbase ^ tbase) & um;
      s.stride ^= (xstride ^ tstride) & um;
      const uint32_t seg = (uint32_t)((toff_b - toff_a) * 2) & (0u - (uint32_t)(step > ksteps));
      s.soff = (int)((uint32_t)s.soff ^ (((uint32_t)s.soff ^ seg) & um));
    }
    return s;
  };
  auto load_w = [&](auto Qc, int ct, int kt) {   // slab Q (0..3) of k-tile kt
    constexpr int Q = decltype(Qc)::value;
    wr[Q % S][ct] = __builtin_amdgcn_raw_buffer_load_b128(re, evoff + (uint32_t)(ct & 1) * 256u,
                                                         (wt0 + min(kt, ktiles - 1)) * 65536 + (ct >> 1) * 8192 + Q * 2048,
                                                         KIND == kPreHeadOnce ? kStreamOnce : 0);
  };
  // One slab (32 k) of k-tile kt: RT x 4 MFMAs, and with them the fragments of the next slab, the weights of the slab three
  // further on into the stage that the slab before has finished with, and half a step of activations for the buffer
  // whose last reader was the slab before the barrier.
  auto slab = [&](auto Uc, int kt, uint32_t dbuf) {
    constexpr int U = decltype(Uc)::value, UN = (U + 1) & 3, UL = (U + 3) & 3;
    const Src src = source(2 * kt + (U == 0 ? 3 : U < 3 ? 4 : 5));
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
#pragma unroll
      for (int j = 0; j < CT; ++j) {
        const int ct = (rt & 1) ? CT - 1 - j : j;
        // (three waves per unit leave the weights of some slabs in accumulator registers, from which the compiler copies them right in front of
        // their use; the stream of the weights, which bounds this form, hides the wait states)
        if constexpr (pre_waves(RT, KIND) == 3) mfma16_acc_wait(wr[U % S][ct], xf[rt], acc[rt][ct]);
        else mfma16_acc(wr[U % S][ct], xf[rt], acc[rt][ct]);
        if (j == 1 && rt % (RT / CT) == RT / CT - 1) load_w(ic<UL>{}, rt / (RT / CT), kt + ((U + 3) >> 2));
        if (j == CT / 2 && (rt & 3) == 1) dma(src, ((U & 1) ? 0 : HALF) + (rt >> 2), dbuf);
        if (j == CT - 1) xf[rt] = lds_ld128(xaddr[UN & 1] + (uint32_t)(rt * 2048) + ((UN >> 1) ? SB : 0u));
        __builtin_amdgcn_sched_barrier(0);   // in the order written
      }
    }
    if (U == 1) xaddr[0] ^= 2 * SB;
    if (U == 2) xaddr[1] ^= 2 * SB;
    __builtin_amdgcn_sched_barrier(0);
  };
  // step 2 and the first half of 3 (slab 0 of the loop brings the other), the weights of three slabs
#pragma unroll
  for (int st = 2; st < 4; ++st) {
    const Src src = source(st);
#pragma unroll
    for (int c = 0; c < (st < 3 ? PASSES : HALF); ++c) dma(src, c, (uint32_t)st * SB);
  }
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) load_w(ic<0>{}, ct, 0);
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) load_w(ic<1>{}, ct, 0);
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) load_w(ic<2>{}, ct, 0);
  // step 0 has landed: behind it 2 PASSES + HALF loads into LDS and twelve fragments
  tnx_wait_vm(2 * PASSES + HALF + 3 * CT);
  __syncthreads();
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) xf[rt] = lds_ld128(xaddr[0] + (uint32_t)(rt * 2048));
  // A barrier stands in front of the first read of a step.  The last load of that step was issued in the first slab of two steps
  // before; behind it a slab issues its last fragment load, and then come four slabs of HALF + 4 loads each.
  constexpr int kBehind = 4 * (HALF + CT);
  uint32_t b3 = 3 * SB, b4 = 0, b5 = SB;   // buffers of steps 2 kt + 3, + 4, + 5
  int kt = 0;
  do {   // (at least one k-tile: a loop that may not run would merge its accumulators with the zeros before it, copy by copy)
    __builtin_amdgcn_sched_barrier(0);
    slab(ic<0>{}, kt, b3);
    tnx_wait_vm(kBehind);
    __syncthreads();
    __builtin_amdgcn_sched_barrier(0);
    slab(ic<1>{}, kt, b4);
    slab(ic<2>{}, kt, b4);
    tnx_wait_vm(kBehind);
    __syncthreads();
    __builtin_amdgcn_sched_barrier(0);
    slab(ic<3>{}, kt, b5);
    b3 ^= 2 * SB;
    b4 ^= 2 * SB;
    b5 ^= 2 * SB;
  } while (++kt < ktiles);
  // the MFMAs are assembly: what reads their results next waits out the pipe by hand
  auto settle = [&]() {
    asm volatile("s_nop 15\n\ts_nop 15");
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) pin_acc(acc[rt][ct]);
  };
  if constexpr (LORA != kLoraInPlace) settle();
  tnx_wait_vm(0);   // no load into LDS is still on its way
  __syncthreads();

  if constexpr (LORA != 0) {
    if constexpr (!EARLY_B) load_adapter_b();
    uint32_t tl[CT];   // this lane's place in the segment of each column tile
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) tl[ct] = (uint32_t)((ksteps & 3) + (toff[ct] == toff_a ? 0 : 1)) * SB + (uint32_t)lm * 128u;
    uint32_t tc[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) tc[j] = ((uint32_t)(4 * j + lq) ^ pre_swizzle((uint32_t)lm)) * 16u;
    u32x4 tf[2][CT][2];   // fragments one row tile ahead
    auto load_t = [&](int rt) {
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int j = 0; j < 2; ++j) tf[rt & 1][ct][j] = lds_ld128(tl[ct] + tc[j] + (uint32_t)(rt * 2048));
    };
    load_t(0);
    if constexpr (LORA == kLoraInPlace) {
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int q = 0; q < 4; ++q) lbv[ct][j][q] = pack2bf(bflo(lbv[ct][j][q]) * a.lora_scale, bfhi(lbv[ct][j][q]) * a.lora_scale);
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        if (rt + 1 < RT) load_t(rt + 1);
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) mfma16_acc_wait(lbv[ct][0], tf[rt & 1][ct][0], acc[rt][ct]);
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) mfma16_acc_wait(lbv[ct][1], tf[rt & 1][ct][1], acc[rt][ct]);
        __builtin_amdgcn_sched_barrier(0);   // (all tiles' fragments at once do not fit the registers)
      }
      settle();
    } else {
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        if (rt + 1 < RT) load_t(rt + 1);
        f32x4 part[CT];
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) part[ct] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) part[ct] = mfma16(lbv[ct][0], tf[rt & 1][ct][0], part[ct]);
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) part[ct] = mfma16(lbv[ct][1], tf[rt & 1][ct][1], part[ct]);
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[rt][ct][i] += a.lora_scale * part[ct][i];
          pin_acc(acc[rt][ct]);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    __syncthreads();  // every wave is done with the buffers: they become the output stage
  }

  // A lane holds, for row rt * 16 + lane % 16 and column tile ct, the columns 4 (lane / 16) + e of the tile.
  constexpr bool mul = pre_mul(KIND);
  if constexpr (KIND == kPreF32) {   // fp32 results leave from the accumulators, 16 bytes per lane
    float* y = reinterpret_cast<float*>(a.y);
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      if (rt * 16 + lm >= rows_here) continue;
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) {
        const int64_t col = (int64_t)ntile * kWideCols + wn * (16 * CT) + ct * 16 + 4 * lq;
        float* o = y + (m0 + rt * 16 + lm) * a.ldy + col;
        if (col + 4 <= a.N && (a.ldy & 3) == 0) {
          *reinterpret_cast<f32x4*>(o) = acc[rt][ct];
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (col + e < a.N) o[e] = acc[rt][ct][e];
        }
      }
    }
    return;
  }
  constexpr int sld = (mul ? kWideCols / 2 : kWideCols) + 8;
  auto put = [&](int at, float v0, float v1, float v2, float v3) {
    *reinterpret_cast<__attribute__((address_space(3))) u32x2*>(static_cast<uintptr_t>(at * 2)) = u32x2{pack2bf(v0, v1), pack2bf(v2, v3)};
  };
  if constexpr (mul) {   // column tiles 2 c | 2 c + 1 are the gate and the up columns
    auto gated = [](float z, float u) {
      if constexpr (KIND == kPreSilu) return rbf(silu_bf16(rbf(z))) * rbf(u);
      else if constexpr (KIND == kPreGelu) return rbf(gelu_tanh_bf16(rbf(z))) * rbf(u);
      else if constexpr (KIND == kPreSiluF32) return z / (1.0f + expf(-z)) * u;
      else return gelu_tanh_fast(z) * u;
    };
#pragma unroll
    for (int c = 0; c < CT / 2; ++c)
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        const f32x4 g = acc[rt][2 * c], u = acc[rt][2 * c + 1];
        put((rt * 16 + lm) * sld + wn * (8 * CT) + c * 16 + 4 * lq, gated(g[0], u[0]), gated(g[1], u[1]), gated(g[2], u[2]), gated(g[3], u[3]));
      }
  } else {
    auto stage_tile = [&](auto f) {
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
          const f32x4 v = acc[rt][ct];
          put((rt * 16 + lm) * sld + wn * (16 * CT) + ct * 16 + 4 * lq, f(v[0]), f(v[1]), f(v[2]), f(v[3]));
        }
    };
    if constexpr (KIND == kPreRelu2) {
      stage_tile([](float v) { return fmaxf(v, 0.f) * fmaxf(v, 0.f); });
    } else if constexpr (pre_head(KIND) && LORA == 0) {   // (the soft cap comes with dense heads only)
      if (h.softcap > 0.f) stage_tile([&](float v) { return soft_cap_fast(v, h.softcap); });
      else stage_tile([](float v) { return v; });
    } else {
      stage_tile([](float v) { return v; });
    }
  }
  __syncthreads();
  wide_tile_out<ROWS, GROUPED, pre_head(KIND), mul>(a, h, ntile, m0, rows_here);
}


template <int RT, bool GROUPED, int KIND, int LORA, bool HALVES>
__global__ __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(pre_waves(RT, KIND), pre_waves(RT, KIND))))
void qgemm_pre_kernel(const QLArgs a, const WideHead h) {
  constexpr int ROWS = 16 * RT;
  extern __shared__ __align__(16) unsigned char smem[];   // (addressed absolutely: no static LDS in this kernel, checked by the host)
  const int lane = threadIdx.x & 63;
  const int tiles_m = (int)((a.M + ROWS - 1) / ROWS), tiles_n = (int)((a.N + kWideCols - 1) / kWideCols);
  int mtile, ntile, expert = 0, m_from = 0, m_end = 0;
  // tile number `tile` of row blocks x column tiles: in groups of `group` row blocks, inside a group column tile by column tile.  With groups of
  // 1024 rows an XCD works on about 1024 rows x 8 column tiles at a time (2048 or 4096 rows: the same at 16 row tiles, 3 to 20 % slower at 8).
  auto tile_in = [&](int tile, int row_blocks, int group) {
    const int per_group = group * tiles_n, g = tile / per_group, r = tile % per_group;
    const int gm = min(group, row_blocks - g * group);
    mtile = g * group + r % gm;
    ntile = r / gm;
  };
  constexpr int GR = 1024 / ROWS;
  if constexpr (GROUPED) {
    // Tiles expert by expert; every wave finds its own: 256 experts at a time, four to a lane, from one round trip for all their offsets and a running
    // sum by DPP: it stands in front of a work-group's first load, a tenth of its time at short contractions (clock stamps).  With the places of the stored rows asked for
    // at once (wide_out.h), us before (a round trip and a chain of exchanges through LDS per 64 experts, twice) | now: 57288 routes of 128 experts
    // 768 -> 2048 286 | 262, 2048 -> 1536 gated 428 | 424; 65536 of 64 768 -> 2048 302 | 283, 2048 -> 768 232 | 225.
    const int E = a.n_experts;
    int from[4], to[4], nb[4], end[4];   // an expert's routes and its blocks; the blocks up to its last one
    auto count = [&](int base, int before) -> int {   // returns `before` and the blocks of these experts
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        from[c] = a.offsets[min(base + 64 * c + lane, E)];
        to[c] = a.offsets[min(base + 64 * c + lane + 1, E)];
      }
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        nb[c] = (to[c] - from[c] + ROWS - 1) / ROWS;
        end[c] = wave_scan(nb[c]) + before;
        before = __builtin_amdgcn_readlane(end[c], 63);
      }
      return before;
    };
    int total = 0;
    for (int base = 0; base < E; base += 256) total = count(base, total);
    const int tile = xcd_tile((int)blockIdx.x, total * tiles_n);
    if (tile < 0) return;   // past the last block (the grid covers an upper bound)
    const int block = tile / tiles_n;
    int found_at = 0, found_nb = 1;
    for (int base = 0, before = 0; base < E; base += 256) {
      if (E > 256) before = count(base, before);
      bool found = false;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const uint64_t hit = __ballot(block < end[c] && block >= end[c] - nb[c]);   // (one lane: the blocks of an expert are its own)
        if (hit) {
          const int l = __builtin_ctzll(hit);
          expert = base + 64 * c + l;
          found_nb = __builtin_amdgcn_readlane(nb[c], l);
          found_at = tile - (__builtin_amdgcn_readlane(end[c], l) - found_nb) * tiles_n;
          m_from = __builtin_amdgcn_readlane(from[c], l);
          m_end = __builtin_amdgcn_readlane(to[c], l);
          found = true;
        }
      }
      if (found) break;
    }
    // an expert of many rows in groups of 1024 rows or near it, equal ones, or its few last blocks would draw all weights for themselves:
    // 8 experts of 8000 rows x 4096 -> 4096 took 2340 us with all row blocks per column tile against 1710 (256-row tiles), 2395 against
    // 1760 (128); 8 of 1300 rows, eleven blocks, 340 us in groups of eight and three against 318 in one of eleven.
    const int groups = max(1, (found_nb + GR / 2) / GR);
    tile_in(found_at, found_nb, (found_nb + groups - 1) / groups);
  } else if constexpr (HALVES) {
    // every XCD's share of the whole tiles, and behind it its share of the halves: the slots that the whole ones leave over take those,
    // two in turn
    const int id = (int)blockIdx.x, whole = tiles_m * (tiles_n - 1);
    const int mine = (whole >> 3) + (int)((id & 7) < (whole & 7)), s = id >> 3;
    if (s >= mine) {
      const int half = xcd_tile((s - mine) * 8 + (id & 7), tiles_m);
      if (half < 0) return;
      pre_tile<RT, false, KIND, LORA, 2>(a, h, half, tiles_n - 1, 0, 0, 0);
      return;
    }
    const int tile = xcd_tile(id, whole), per_group = GR * (tiles_n - 1), g = tile / per_group, r = tile % per_group;
    const int gm = min(GR, tiles_m - g * GR);
    mtile = g * GR + r % gm;
    ntile = r / gm;
  } else {
    tile_in(xcd_tile((int)blockIdx.x, tiles_m * tiles_n), tiles_m, GR);
  }
  pre_tile<RT, GROUPED, KIND, LORA, 4>(a, h, mtile, ntile, expert, m_from, m_end);
}

}  // namespace
