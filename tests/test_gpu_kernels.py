"""GPU parity of every kernel family against the CPU oracle, called through the C ABI.

Bars: bit-exact for integer / index outputs (codes, scales, arg-max ids, routes); for bf16
outputs the kernel and the oracle round the same fp32 value, so they may differ by one bf16 ulp
where the accumulation order moves a sum across a rounding boundary: the tests allow
|diff| <= 2^-7 * |ref| + atol (one ulp) and require the bulk of the elements to be bit-equal.
"""
import math

import numpy as np
import pytest
import torch

from oracle import model_ref as MR
from oracle import quant_ref as Q
from oracle import rl_ref, threefry as TF
from oracle import sampler_ref as SR

pytestmark = pytest.mark.gpu


def bf(x):
  return x.to(torch.bfloat16)


def rnd(shape, seed, scale=1.0):
  g = torch.Generator().manual_seed(seed)
  return (torch.randn(*shape, generator=g) * scale).to(torch.bfloat16).float()


def assert_bf16_close(got, ref, atol=1e-6, min_equal=0.97, what="", mag=None, ulps=1):
  """mag: magnitude the one-ulp allowance is taken from when it is not the result itself (a sum
  with a residual can cancel: the ulp that matters is the one of the larger operand).  ulps: for
  results computed from several rounded intermediates, each of which may be one ulp off."""
  got, ref = got.float().cpu(), ref.float().cpu()
  diff = (got - ref).abs()
  # one ulp of the larger of the two values (the spacing doubles at a power of two: two
  # neighbouring bf16 values on either side of it differ by the ulp of the upper one)
  big = torch.maximum(ref.abs(), got.abs())
  tol = (big if mag is None else torch.maximum(big, mag.float().cpu().abs())) * (ulps * 2.0 ** -7) + atol
  bad = (diff > tol).sum().item()
  eq = (got == ref).float().mean().item()
  assert bad == 0, f"{what}: {bad} elements beyond one bf16 ulp, max diff {diff.max().item()}"
  assert eq >= min_equal, f"{what}: only {eq:.4f} of the elements are bit-equal"


@pytest.mark.parametrize("qtype", [Q.INT4, Q.NF4])
@pytest.mark.parametrize("group", [32, 64, 128, 256])
@pytest.mark.parametrize("interleave", [False, True])
def test_quantize_pack_bit_exact(gpu, qtype, group, interleave):
  from tunix_amd import ops
  K, N = 512, 96 if not interleave else 128
  w = rnd((K, N), 11 + group, 0.02)
  w[0:group, 3] = 0.0  # an all-zero group
  codes, scale = Q.quantize(w.numpy(), group, qtype)
  ref_c, ref_s = Q.pack_qw(codes, scale, group, interleave)
  c, s = ops.quantize_pack(bf(w).to(gpu), group, qtype, interleave)
  np.testing.assert_array_equal(c.cpu().numpy().view(np.uint32), ref_c)
  got_s = s.cpu().view(torch.int16).numpy().view(np.uint16)
  assert got_s.size == ref_s.size + 8          # 16 bytes of tail padding for 8-byte scale reads
  np.testing.assert_array_equal(got_s[:ref_s.size], ref_s)
  deq = ops.qw_dequant(c, s, K, N, group, qtype, interleave).cpu().numpy()
  np.testing.assert_array_equal(deq, Q.dequantize(codes, scale, group, qtype))


@pytest.mark.parametrize("bound", [7.0, 7.5, 8.0])
def test_quantize_pack_int4_bound(gpu, bound):
  """scale = bf16(absmax / bound) for the bounds a symmetric int4 quantiser may use: codes and
  scales bit-exact against the oracle; a bound <= 0 selects 7."""
  from tunix_amd import ops
  K, N, g = 256, 64, 64
  w = rnd((K, N), 5, 0.02)
  codes, scale = Q.quantize(w.numpy(), g, Q.INT4, int4_bound=bound)
  ref_c, ref_s = Q.pack_qw(codes, scale, g, False)
  c, s = ops.quantize_pack(bf(w).to(gpu), g, Q.INT4, False, bound)
  np.testing.assert_array_equal(c.cpu().numpy().view(np.uint32), ref_c)
  np.testing.assert_array_equal(s.cpu().view(torch.int16).numpy().view(np.uint16)[:ref_s.size], ref_s)
  if bound == 7.0:
    c0, s0 = ops.quantize_pack(bf(w).to(gpu), g, Q.INT4, False, 0.0)
    assert torch.equal(c0, c) and torch.equal(s0[:ref_s.size], s[:ref_s.size])


@pytest.mark.parametrize("B,T,D,V,scale", [(128, 1, 4096, 1000, 1.0), (5, 7, 1152, 300, 1152 ** 0.5), (3, 2, 100, 50, 1.0)])
def test_embed_gathers_rows_and_scales_in_bf16(gpu, B, T, D, V, scale):
  """tnx_embed: out[b*T + t] = table[ids[b, col + t]] * bf16(scale), ids read at a device-resident
  column; Gemma-3's sqrt(D) is rounded to bf16 before the product (gemma3/model.py:353-358); ids
  outside the vocabulary (pad sentinels) read row 0.  Bit-exact (16-byte path and scalar path)."""
  from tunix_amd import ops
  table = rnd((V, D), 3, 0.02)
  rng = np.random.default_rng(B)
  L = T + 5
  ids = rng.integers(0, V, size=(B, L)).astype(np.int32)
  ids[0, 3] = V + 7      # beyond the vocabulary
  ids[B - 1, 3] = -1
  col = 3
  out = torch.full((B * T, D), 9.0, dtype=torch.bfloat16, device=gpu)
  ops.embed(bf(table).to(gpu), torch.from_numpy(ids).to(gpu), torch.tensor([col], dtype=torch.int32, device=gpu),
            B, T, scale, out)
  src = ids[:, col:col + T].reshape(-1).astype(np.int64)
  src = np.where((src < 0) | (src >= V), 0, src)
  want = Q.rb(table)[src]
  if scale != 1.0:
    want = Q.rb(want * Q.rb(torch.tensor(scale, dtype=torch.float32)))
  assert torch.equal(out.float().cpu(), want)


@pytest.mark.parametrize("E,k", [(1, 1), (63, 5), (64, 8), (65, 3), (128, 64), (200, 8), (257, 8), (300, 16), (512, 4), (513, 9), (1024, 64)])
def test_moe_route_picks_the_largest_lowest_first(gpu, E, k):
  """Every number of experts per lane: ids in the order of the scores, the lower one first among equals, weights that add up."""
  from tunix_amd import ops
  M = 37
  scores = bf(rnd((M, E), 121))
  scores[3] = 0.25
  scores[5, E // 2:] = 1.5
  tw, ti = torch.empty(M, k, dtype=torch.bfloat16, device=gpu), torch.empty(M, k, dtype=torch.int32, device=gpu)
  ops.moe_route_topk(scores.to(gpu), k, tw, ti)
  val, idx = torch.sort(scores.float(), dim=-1, descending=True, stable=True)
  assert torch.equal(ti.cpu().long(), idx[:, :k])
  want = torch.softmax(val[:, :k], -1)
  assert ((tw.float().cpu() - want).abs() <= 2.0 ** -8 * want + 1e-6).all()   # (rounded to bf16)


def test_moe_route_keeps_ids_in_range_for_nan_scores(gpu):
  """A row of router scores with a NaN (a hidden state gone bad): the k ids stay distinct and
  inside [0, E) -- the route sort and the grouped GEMM index memory with them -- and the row's
  weights are NaN, so the NaN reaches the output instead of a memory fault; other rows are
  untouched."""
  from tunix_amd import ops
  M, E, k = 6, 128, 8
  scores = rnd((M, E), 70)
  clean = scores.clone()
  scores[2, 17] = float("nan")
  scores[4, :] = float("nan")
  tw = torch.empty(M, k, dtype=torch.bfloat16, device=gpu)
  ti = torch.full((M, k), -5, dtype=torch.int32, device=gpu)
  ops.moe_route_topk(bf(scores).to(gpu), k, tw, ti)
  ids = ti.cpu().numpy()
  assert ((ids >= 0) & (ids < E)).all()
  for m in range(M):
    assert len(set(ids[m].tolist())) == k
  assert torch.isnan(tw[2].float()).all() and torch.isnan(tw[4].float()).all()
  tw2 = torch.empty_like(tw)
  ti2 = torch.empty_like(ti)
  ops.moe_route_topk(bf(clean).to(gpu), k, tw2, ti2)
  for m in (0, 1, 3, 5):
    assert torch.equal(ti[m], ti2[m]) and torch.equal(tw[m], tw2[m])
  counts = torch.empty(E, dtype=torch.int32, device=gpu)
  offs = torch.empty(E + 1, dtype=torch.int32, device=gpu)
  sr = torch.full((M * k,), -1, dtype=torch.int32, device=gpu)
  ops.moe_sort_routes(ti, E, counts, offs, sr)
  assert sorted(sr.cpu().tolist()) == list(range(M * k))      # every route placed exactly once


def _lora(K, N, r, seed):
  return rnd((K, r), seed, 0.02), rnd((r, N), seed + 1, 0.01)


def _pad_lora(a, b, rp):
  K, r = a.shape
  N = b.shape[1]
  a_t = torch.zeros(rp, K)
  a_t[:r] = a.t()
  b_t = torch.zeros(N, rp)
  b_t[:, :r] = b.t()
  return a_t, b_t


@pytest.mark.parametrize("M,K,N,group,qtype,r,split", [
    (8, 512, 512, 64, Q.INT4, 8, 1),
    (128, 4096, 1024, 64, Q.NF4, 64, 1),
    (128, 4096, 1024, 64, Q.NF4, 64, 4),
    (64, 1152, 1024, 128, Q.INT4, 16, 3),
    (33, 768, 208, 256, Q.NF4, 0, 1),
    (130, 256, 48, 32, Q.INT4, 32, 1),
    # the activation tiles' road into LDS at its corners: a single k-tile (the adapter block is the
    # second tile), one whole turn of the weight ring, every row-tile count, uneven k splits
    (128, 128, 256, 64, Q.NF4, 64, 1),
    (16, 384, 256, 64, Q.INT4, 32, 1),
    (32, 640, 384, 128, Q.NF4, 64, 2),
    (100, 896, 512, 64, Q.INT4, 64, 3),
    (17, 256, 128, 32, Q.NF4, 16, 1),
    (64, 1024, 256, 64, Q.NF4, 32, 8),
])
def test_qlinear_lora_matches_oracle(gpu, M, K, N, group, qtype, r, split):
  from tunix_amd import _lib as L
  from tunix_amd import ops
  x = rnd((M, K), 1)
  w = rnd((K, N), 2, 0.02)
  codes, scale = Q.quantize(w.numpy(), group, qtype)
  a = b = None
  if r:
    a, b = _lora(K, N, r, 3)
  ref = Q.rb(Q.qlinear_lora(x, codes, scale, group, qtype, a, b, lora_scale=2.0))
  c, s = ops.quantize_pack(bf(w).to(gpu), group, qtype)
  y = torch.empty(M, N, dtype=torch.bfloat16, device=gpu)
  kw = {}
  if r:
    rp = (r + 31) // 32 * 32
    a_t, b_t = _pad_lora(a, b, rp)
    t = torch.zeros(M, rp, dtype=torch.bfloat16, device=gpu)
    ops.lora_down(bf(x).to(gpu), bf(a_t).to(gpu), t)
    t_ref = Q.rb((x.double() @ a.double()).float())
    assert_bf16_close(t[:, :r], t_ref, what="lora_down")
    kw = dict(lora_rank=rp, lora_nseg=1, lora_seg_end=[N], lora_seg_toff=[0], t=t, t_ld=rp,
              lora_b=bf(b_t).to(gpu), lora_scale=2.0)
  ws = torch.full((split * M * N,), float('nan'), dtype=torch.float32, device=gpu) if split > 1 else None
  d = ops.make_qlinear_desc(M=M, K=K, N=N, group=group, qtype=qtype, x=bf(x).to(gpu), codes=c,
                            scales=s, y=y, split_k=split, ws=ws, **kw)
  ops.qlinear(d)
  torch.cuda.synchronize()
  assert_bf16_close(y, ref, what="qlinear")


@pytest.mark.parametrize("M,K,N,split,group,qtype,rank,nseg,epi", [
    (1, 512, 128, 1, 64, Q.INT4, 64, 1, "store"),         # one row of int4, a turn of the ring
    (3, 1280, 208, 1, 32, Q.NF4, 32, 1, "residual"),      # a last column block of five tiles, four scales per k-tile
    (8, 3584, 512, 3, 64, Q.INT4, 64, 3, "store"),        # 28 k-tiles in splits of 10, 10, 8; three adapter segments
    (4, 1792, 512, 2, 64, Q.NF4, 64, 1, "residual"),      # seven per split: two turns less one
    (5, 2176, 768, 1, 128, Q.NF4, 64, -1, "silu"),        # 17 k-tiles, gate | up with the next adapter's planes
    (7, 1024, 25600, 1, 64, Q.INT4, 64, -1, "gelu"),      # eight k-tiles, work-groups for most of the device
    (9, 2048, 12288, 1, 64, Q.NF4, 0, 1, "f32"),          # 16 k-tiles of sixteen rows
    (16, 3712, 384, 2, 64, Q.INT4, 96, 1, "store"),       # 15 and 14; an adapter of more than 64 ranks
    (12, 4096, 320, 2, 256, Q.NF4, 64, -1, "gelu"),       # sixteen per split
    (16, 2304, 8192, 1, 64, Q.NF4, 64, -1, "silu"),       # eighteen
    (20, 1280, 208, 1, 32, Q.INT4, 64, 1, "f32"),         # two row tiles
    (32, 2688, 512, 3, 64, Q.NF4, 64, 3, "residual"),     # seven per split
    (27, 1536, 768, 1, 128, Q.INT4, 64, -1, "gelu"),
])
def test_few_rows_equal_the_shared_form(gpu, M, K, N, split, group, qtype, rank, nseg, epi):
  """At most 32 rows (a column tile per wave, all activations in LDS) against the same rows in a call of 72, which runs on another kernel (tiles of
  128 x 128, the waves sharing a k-tile behind a barrier).  Same products; a column's fp32 sum of K terms in another order, so a
  rounded result may be the neighbouring bf16 value."""
  from tunix_amd import _lib as L
  from tunix_amd import ops
  mul = epi in ("silu", "gelu")
  x, t, res = bf(rnd((72, K), 111)).to(gpu), bf(rnd((72, 320), 112)).to(gpu), bf(rnd((72, N), 113)).to(gpu)
  c, s = ops.quantize_pack(bf(rnd((K, N), 114, 0.03)).to(gpu), group, qtype, mul)
  lb = bf(rnd((N, max(rank, 32)), 115, 0.1)).to(gpu)
  ends = [N] if nseg < 2 else [N // 2, N * 3 // 4 // 16 * 16, N][:nseg]
  nxt = bf(rnd((64, N // 2), 116, 0.05)).to(gpu)

  def run(n):
    y = torch.full((n, N // 2 if mul else N), 7.0, dtype=torch.float32 if epi == "f32" else torch.bfloat16, device=gpu)
    ws = torch.full((split * n * N,), float("nan"), device=gpu) if split > 1 else None
    kw = dict(lora_rank=rank, lora_nseg=nseg, lora_seg_end=ends, lora_seg_toff=[i * 64 for i in range(len(ends))], t=t,
              t_ld=320, lora_b=lb, lora_scale=1.5) if rank else {}
    planes = None
    if mul and split == 1:
      planes = torch.full(((N + 127) // 128 * 8192,), float("nan"), device=gpu)
      kw.update(next_a_t=nxt, next_rank=64, next_tpart=planes)
    d = ops.make_qlinear_desc(M=n, K=K, N=N, group=group, qtype=qtype, x=x, codes=c, scales=s, y=y, split_k=split, ws=ws,
                              epilogue={"store": L.TNX_EPI_STORE, "residual": L.TNX_EPI_RESIDUAL, "f32": L.TNX_EPI_F32,
                                        "silu": L.TNX_EPI_SILU_MUL, "gelu": L.TNX_EPI_GELU_MUL}[epi],
                              residual=res if epi == "residual" else None, **kw)
    ops.qlinear(d)
    tn = None
    if planes is not None:
      tn = torch.zeros(n, 64, dtype=torch.bfloat16, device=gpu)
      ops.lora_reduce(planes, n, (N + 127) // 128, 64, tn)
    torch.cuda.synchronize()
    return y, tn

  (few, tf), (many, tm) = run(M), run(72)
  # (magnitude of a result's terms: gated products and sums with a residual are rounded more than once)
  ulps = 3 if mul else 1
  if epi == "f32":
    # |sum error| <= 2 K eps * sum |terms|: K terms of about 0.03 in random signs
    assert (few - many[:M]).abs().max().item() <= 2 * K * 2.0 ** -24 * K * 0.03
  else:
    mag = None if epi != "residual" else torch.maximum(many[:M].float().abs(), res[:M].float().abs())
    assert_bf16_close(few, many[:M], min_equal=0.95, what=epi, mag=mag, ulps=ulps)
  if tf is not None:
    assert torch.isfinite(tf.float()).all()
    # t of the next adapter: products of activations that may differ by an ulp each
    assert (tf.float() - tm[:M].float()).abs().max().item() <= 2.0 ** -6 * tm.float().abs().max().item()


@pytest.mark.parametrize("M,K,N,split,group,qtype,rank,mul", [
    (1, 128, 16, 1, 64, Q.NF4, 0, False),        # one k-tile, one column tile
    (8, 640, 272, 2, 32, Q.INT4, 64, False),     # three and two k-tiles; a last block of one column tile
    (8, 6144, 128, 1, 64, Q.NF4, 64, False),     # 48 k-tiles: what LDS holds of eight rows
    (5, 7296, 256, 1, 64, Q.NF4, 32, True),      # 57: two chunks of slots filled again, the last with one
    (7, 10368, 128, 1, 128, Q.INT4, 96, False),  # 81: one more than without a table; a rank past 64
    (9, 3072, 128, 1, 64, Q.NF4, 64, True),      # 24, of sixteen rows
    (16, 4224, 144, 1, 32, Q.NF4, 64, False),    # 33
    (13, 5248, 256, 1, 64, Q.INT4, 0, True),     # 41 (40 are held)
    (17, 1536, 128, 1, 64, Q.NF4, 64, False),    # 12, of 32 rows
    (32, 2176, 384, 1, 64, Q.NF4, 64, True),     # 17
    (31, 2688, 160, 1, 128, Q.INT4, 64, True),   # 21 (20 are held)
    (24, 8192, 128, 4, 32, Q.NF4, 32, False),    # sixteen per split
    (33, 512, 144, 1, 64, Q.NF4, 64, False),     # four row tiles: unsplit, the form of 64 x 128 tiles
    (64, 2048, 272, 8, 32, Q.INT4, 96, False),   # two per split
    (5, 1152, 144, 8, 64, Q.NF4, 64, False),     # nine k-tiles in eight splits of two: three splits of none
    (16, 4480, 128, 8, 64, Q.INT4, 64, False),   # 35 in eight of five: one of none
    (40, 1152, 144, 8, 64, Q.NF4, 64, False),
    (48, 1024, 1024, 8, 64, Q.NF4, 64, False),   # one, 64 work-groups: the most that come here
    (48, 1024, 1040, 8, 64, Q.NF4, 64, False),   # 72
    (57, 1152, 384, 3, 128, Q.INT4, 0, False),   # three per split
])
def test_few_rows_at_the_edges_of_what_lds_holds(gpu, M, K, N, split, group, qtype, rank, mul):
  """Linears of few rows against 64 bits over the same weights, both rounded to bf16.  The fp32 sum of K products of about 0.03 is off by
  some eps of the sum of their magnitudes, 2^-23 * 0.03 K (`off`, what a result near zero may differ by), a hundredth of a bf16 ulp of the usual
  result of 0.03 sqrt(K): the rounded values are equal but for near ties.  Gated products are rounded at every step."""
  off = 2.0 ** -23 * 0.03 * K
  from tunix_amd import _lib as L
  from tunix_amd import ops
  x, t = bf(rnd((M, K), 311)).to(gpu), bf(rnd((M, 2 * max(rank, 32)), 312)).to(gpu)
  w = bf(rnd((K, N), 313, 0.03)).to(gpu)
  c, s = ops.quantize_pack(w, group, qtype, mul)
  lb = bf(rnd((N, max(rank, 32)), 314, 0.1)).to(gpu)
  # (interleaved: column tile 2 i is gate tile i, 2 i + 1 up tile i; the dequantised weights come back as they went in)
  deq = ops.qw_dequant(c, s, K, N, group, qtype, mul).double()
  cols = torch.arange(N, device=gpu)
  place = (cols % (N // 2)) // 16 * 32 + cols // (N // 2) * 16 + cols % 16 if mul else cols   # packed column of each
  y64 = x.double() @ deq
  if rank:
    seg = cols // (N // 2) if mul else torch.zeros_like(cols)
    td = t.double()
    for g in range(2 if mul else 1):
      at = torch.nonzero(seg == g)[:, 0]
      y64[:, at] += 1.5 * (td[:, g * rank:(g + 1) * rank] @ lb.double()[place[at], :rank].T)
  kw = dict(lora_rank=rank, lora_nseg=-1 if mul else 1, lora_seg_end=[N // 2, N] if mul else [N], lora_seg_toff=[0, rank] if mul else [0], t=t,
            t_ld=t.shape[1], lora_b=lb, lora_scale=1.5) if rank else {}
  y = torch.full((M, N // 2 if mul else N), 7.0, dtype=torch.bfloat16, device=gpu)
  ws = torch.full((split * M * N,), float("nan"), device=gpu) if split > 1 else None
  nxt = {}
  if mul:
    nxt = dict(next_a_t=bf(rnd((64, N // 2), 315, 0.05)).to(gpu), next_rank=64, next_tpart=torch.full(((N + 127) // 128 * 8192,), float("nan"), device=gpu))
  ops.qlinear(ops.make_qlinear_desc(M=M, K=K, N=N, group=group, qtype=qtype, x=x, codes=c, scales=s, y=y, split_k=split, ws=ws,
                                    epilogue=L.TNX_EPI_SILU_MUL if mul else L.TNX_EPI_STORE, **kw, **nxt))
  torch.cuda.synchronize()
  if mul:
    r = lambda v: v.float().bfloat16().double()
    g, u = r(y64[:, :N // 2]), r(y64[:, N // 2:])
    assert_bf16_close(y, r(r(g * r(torch.sigmoid(g))) * u), min_equal=0.95, what="gated", ulps=3, atol=2 * off * g.abs().max().item())
    tn = torch.zeros(M, 64, dtype=torch.bfloat16, device=gpu)
    ops.lora_reduce(nxt["next_tpart"], M, (N + 127) // 128, 64, tn)
    torch.cuda.synchronize()
    want = y.double() @ nxt["next_a_t"].double().T
    # (products of the same activations, summed in fp32 and rounded once)
    assert_bf16_close(tn, r(want), min_equal=0.95, what="next adapter", atol=1e-5 * want.abs().max().item())
  else:
    assert_bf16_close(y, y64.float().bfloat16(), what="linear", atol=off)


@pytest.mark.parametrize("M,K,N,split,group,qtype,rank,epi", [
    (1, 128, 16, 1, 64, Q.INT4, 32, "store"),        # one k-tile, one column tile, half of the ranks
    (8, 1024, 1152, 8, 128, Q.INT4, 64, "store"),    # one k-tile per split
    (5, 1152, 272, 5, 32, Q.NF4, 64, "store"),       # two per split, one in the last; a last block of one column tile
    (9, 512, 256, 1, 64, Q.NF4, 64, "residual"),     # four, unsplit
    (16, 1920, 384, 3, 64, Q.NF4, 32, "store"),      # five per split: past the form for few
    (13, 4224, 128, 1, 64, Q.NF4, 64, "f32"),        # 33: slots are filled again
    (17, 384, 128, 1, 128, Q.INT4, 64, "store"),     # two row tiles, three k-tiles
    (32, 2176, 256, 1, 32, Q.NF4, 64, "residual"),   # 17 of 32 rows: slots are filled again
    (33, 384, 144, 1, 64, Q.NF4, 64, "store"),       # four row tiles, three k-tiles
    (64, 1152, 384, 3, 128, Q.INT4, 32, "store"),    # three per split
    (57, 512, 272, 1, 32, Q.NF4, 64, "residual"),    # four
    (5, 1152, 144, 8, 64, Q.NF4, 64, "store"),       # nine k-tiles in eight splits of two: three splits of none
    (16, 4480, 128, 8, 64, Q.INT4, 32, "store"),     # 35 in eight of five: one of none
    (40, 1152, 144, 8, 64, Q.INT4, 64, "f32"),
])
def test_few_rows_form_the_adapters_down_projection(gpu, M, K, N, split, group, qtype, rank, epi):
  """y = x . W + 1.5 (x . A) . B with x . A formed inside, against 64 bits: x . A is a pair of bf16, 2^-17 of itself off, so the result is the
  rounded one but for near ties (`off`: the fp32 sums, as above, and those 2^-17 of the adapter's share)."""
  from tunix_amd import _lib as L
  from tunix_amd import ops
  x, w, res = bf(rnd((M, K), 411)).to(gpu), bf(rnd((K, N), 412, 0.03)).to(gpu), bf(rnd((M, N), 413)).to(gpu)
  a_t, lb = bf(rnd((rank, K), 414, 0.03)).to(gpu), bf(rnd((N, rank), 415, 0.1)).to(gpu)
  c, s = ops.quantize_pack(w, group, qtype)
  share = 1.5 * (x.double() @ a_t.double().T) @ lb.double().T
  ref = x.double() @ ops.qw_dequant(c, s, K, N, group, qtype).double() + share
  off = 2.0 ** -23 * 0.03 * K + 2.0 ** -17 * share.abs().max().item()
  y = torch.full((M, N), 7.0, dtype=torch.float32 if epi == "f32" else torch.bfloat16, device=gpu)
  ws = torch.full((split * M * N,), float("nan"), device=gpu) if split > 1 else None
  t = torch.full((M, rank), float("nan"), dtype=torch.bfloat16, device=gpu)   # (not read)
  d = ops.make_qlinear_desc(M=M, K=K, N=N, group=group, qtype=qtype, x=x, codes=c, scales=s, y=y, split_k=split, ws=ws, lora_rank=rank, lora_nseg=1,
                            lora_seg_end=[N], lora_seg_toff=[0], t=t, t_ld=rank, lora_b=lb, lora_scale=1.5, residual=res if epi == "residual" else None,
                            epilogue={"store": L.TNX_EPI_STORE, "residual": L.TNX_EPI_RESIDUAL, "f32": L.TNX_EPI_F32}[epi])
  assert ops.qlinear_inner_rows(K, N, rank, split) >= M
  ops.qlinear(d, a_frag=ops.lora_frag(a_t))
  torch.cuda.synchronize()
  if epi == "f32":
    assert (y.double() - ref).abs().max().item() <= off
  elif epi == "residual":
    ref = ref.float().bfloat16()
    assert_bf16_close(y, (ref.float() + res.float()).bfloat16(), what=epi, atol=off, mag=torch.maximum(ref.float().abs(), res.float().abs()))
  else:
    assert_bf16_close(y, ref.float().bfloat16(), what=epi, atol=off)


@pytest.mark.parametrize("off", [1, 2, 4])
@pytest.mark.parametrize("M,K,N,split,qtype,rank,inside", [
    (1, 512, 144, 1, Q.INT4, 0, False),       # four k-tiles
    (16, 4224, 128, 1, Q.NF4, 64, False),     # 33: slots are filled again
    (31, 2688, 160, 1, Q.INT4, 32, True),     # 21 of 32 rows: here too, with the adapter inside
    (5, 1152, 272, 5, Q.NF4, 64, True),       # two per split
    (57, 1024, 256, 8, Q.INT4, 0, False),     # four row tiles, one k-tile per split
])
def test_few_rows_of_any_alignment(gpu, M, K, N, split, qtype, rank, inside, off):
  """Rows that start `off` elements behind a 16-byte boundary, which loads straight into LDS ask for: the bits of the same rows on one."""
  from tunix_amd import ops
  x = bf(rnd((M, K), 431)).to(gpu)
  c, s = ops.quantize_pack(bf(rnd((K, N), 432, 0.03)).to(gpu), 64, qtype)
  a_t, lb, t = bf(rnd((max(rank, 32), K), 433, 0.03)).to(gpu), bf(rnd((N, max(rank, 32)), 434, 0.1)).to(gpu), bf(rnd((M, 64), 435)).to(gpu)

  def run(rows):
    y = torch.full((M, N), 7.0, dtype=torch.bfloat16, device=gpu)
    ws = torch.full((split * M * N,), float("nan"), device=gpu) if split > 1 else None
    kw = dict(lora_rank=rank, lora_nseg=1, lora_seg_end=[N], lora_seg_toff=[0], t=t, t_ld=64, lora_b=lb, lora_scale=1.5) if rank else {}
    d = ops.make_qlinear_desc(M=M, K=K, N=N, group=64, qtype=qtype, x=rows, codes=c, scales=s, y=y, split_k=split, ws=ws, **kw)
    ops.qlinear(d, a_frag=ops.lora_frag(a_t) if inside else None)
    torch.cuda.synchronize()
    return y

  shifted = torch.full((M * K + 16,), float("nan"), dtype=torch.bfloat16, device=gpu)
  assert shifted.data_ptr() % 16 == 0
  shifted[off:off + M * K] = x.view(-1)
  assert torch.equal(run(shifted[off:off + M * K].view(M, K)), run(x))


@pytest.mark.parametrize("M,K,N,split,qtype,rank", [
    (3, 1152, 272, 5, Q.NF4, 64),      # short splits
    (16, 2176, 128, 1, Q.INT4, 32),    # a ring of k-tiles, half of the ranks
    (32, 1024, 144, 2, Q.NF4, 32),
    (57, 512, 128, 1, Q.NF4, 64),
])
def test_adapter_inside_of_infinite_rows(gpu, M, K, N, split, qtype, rank):
  """x . A formed inside, of rows with an infinite element or with products of A near the largest number: where the rounded t of
  a launch ahead gives an infinite result or none, so does this form; every other row keeps its bits."""
  from tunix_amd import ops
  sign = torch.where(torch.arange(N) % 3 == 0, -1.0, 1.0)
  w, a, lb = rnd((K, N), 441, 0.03), rnd((rank, K), 442, 0.03), rnd((N, rank), 443, 0.1).abs() * sign[:, None]
  w[7], a[:, 7], a[:, 8] = 0.05 * sign, 1.9921875, 1.0   # (both products of element 7 have one sign in a column)
  c, s = ops.quantize_pack(bf(w).to(gpu), 64, qtype)
  a_t, lb, x = bf(a).to(gpu), bf(lb).to(gpu), bf(rnd((M, K), 444)).to(gpu)
  odd = x.clone()
  odd[0, 7], odd[1, 7], odd[1, 8] = float("inf"), 2.0 ** 127, 1.5 * 2.0 ** 119   # (row 1: t past the largest bf16, in 32 bits finite)
  odd[2, 7] = float("nan")

  def run(rows, inside):
    y = torch.full((M, N), 7.0, dtype=torch.bfloat16, device=gpu)
    ws = torch.full((split * M * N,), 7.0, device=gpu) if split > 1 else None
    t = torch.full((M, rank), 7.0, dtype=torch.bfloat16, device=gpu)
    if not inside:
      ops.lora_down(rows, a_t, t, M=M)
    ops.qlinear(ops.make_qlinear_desc(M=M, K=K, N=N, group=64, qtype=qtype, x=rows, codes=c, scales=s, y=y, split_k=split, ws=ws, lora_rank=rank,
                                      lora_nseg=1, lora_seg_end=[N], lora_seg_toff=[0], t=t, t_ld=rank, lora_b=lb, lora_scale=1.5),
                a_frag=ops.lora_frag(a_t) if inside else None)
    torch.cuda.synchronize()
    return y

  got, ahead, plain = run(odd, True), run(odd, False), run(x, True)
  assert torch.isposinf(ahead[0]).sum() == (sign > 0).sum() and torch.isneginf(ahead[0]).sum() == (sign < 0).sum()
  assert torch.isinf(ahead[1]).all() and torch.isnan(ahead[2]).all()
  assert torch.equal(got[:2], ahead[:2]) and torch.isnan(got[2]).all()
  assert torch.equal(got[3:], plain[3:])


def test_adapter_inside_needs_no_t(gpu):
  """A descriptor without t, which the form with the adapter inside does not read, split: the call and the pass that sums its planes."""
  from tunix_amd import ops
  M, K, N = 5, 1024, 256
  x, a_t, lb = bf(rnd((M, K), 451)).to(gpu), bf(rnd((64, K), 452, 0.03)).to(gpu), bf(rnd((N, 64), 453, 0.1)).to(gpu)
  c, s = ops.quantize_pack(bf(rnd((K, N), 454, 0.03)).to(gpu), 64, Q.NF4)
  out = []
  for t in (None, torch.zeros(M, 64, dtype=torch.bfloat16, device=gpu)):
    y, ws = torch.full((M, N), 7.0, dtype=torch.bfloat16, device=gpu), torch.full((4 * M * N,), float("nan"), device=gpu)
    ops.qlinear(ops.make_qlinear_desc(M=M, K=K, N=N, group=64, qtype=Q.NF4, x=x, codes=c, scales=s, y=y, split_k=4, ws=ws, lora_rank=64, lora_nseg=1,
                                      lora_seg_end=[N], lora_seg_toff=[0], t=t, t_ld=0 if t is None else 64, lora_b=lb, lora_scale=1.5),
                a_frag=ops.lora_frag(a_t))
    torch.cuda.synchronize()
    out.append(y)
  assert torch.equal(*out) and torch.isfinite(out[0].float()).all()


def test_adapter_inside_refuses_other_shapes(gpu):
  from tunix_amd import _lib as L
  from tunix_amd import ops
  assert ops.qlinear_inner_rows(512, 256, 96) == 0 and ops.qlinear_inner_rows(500, 256, 64) == 0
  assert ops.qlinear_inner_rows(512, 256, 64) == 64 and ops.qlinear_inner_rows(640, 256, 64) == 32 and ops.qlinear_inner_rows(640, 256, 64, 2) == 64
  w = bf(rnd((512, 256), 421, 0.03)).to(gpu)
  c, s = ops.quantize_pack(w, 64, Q.NF4)
  a_t, lb = bf(rnd((64, 512), 422)).to(gpu), bf(rnd((256, 64), 423)).to(gpu)

  def call(M=4, rank=64, nseg=1, epi=L.TNX_EPI_STORE):
    x, y = bf(rnd((M, 512), 424)).to(gpu), torch.empty(M, 256, dtype=torch.bfloat16, device=gpu)
    ops.qlinear(ops.make_qlinear_desc(M=M, K=512, N=256, group=64, qtype=Q.NF4, x=x, codes=c, scales=s, y=y, lora_rank=rank, lora_nseg=nseg,
                                      lora_seg_end=[128, 256][-abs(nseg):], lora_seg_toff=[0, 64][:abs(nseg)], lora_b=lb, lora_scale=1.0, epilogue=epi),
                a_frag=ops.lora_frag(a_t))

  call()
  for bad in (dict(M=65), dict(rank=96), dict(rank=0), dict(nseg=2), dict(nseg=-1, epi=L.TNX_EPI_SILU_MUL)):
    with pytest.raises(ValueError):
      call(**bad)


@pytest.mark.parametrize("rows,copy,split", [(65536, False, 1), (65536, True, 1), (100, False, 1), (100, False, 2), (16, False, 1)])
def test_silu_of_every_gate(gpu, rows, copy, split):
  """Gates of every finite bf16 value (weights that pick one element of x), among them those whose sigmoid is not a normal fp32
  number any more: x * sigmoid(x) with both factors' roundings, no result lost to zero before the exponential overflows."""
  from tunix_amd import _lib as L
  from tunix_amd import ops
  K, N = 512, 32
  w = torch.zeros(K, N)
  w[0, :N // 2] = 1.0
  w[1, N // 2:] = 1.0
  codes, scales = ops.quantize_pack(bf(w).to(gpu), 64, Q.NF4, True)
  gates = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)
  gates = gates[torch.isfinite(gates.float())]
  if rows < 65536:                       # (the whole range in one large call, its ends and the far tail in small ones)
    gates = torch.cat([gates[gates.float().abs() < 1e-30][:rows // 4], bf(torch.linspace(-92, -80, rows // 2)), gates[-(rows // 4):]])
  g = gates.double()
  x = torch.zeros(len(gates), K, dtype=torch.bfloat16)
  x[:, 0], x[:, 1] = gates, 1.0
  x = x.to(gpu)
  M = len(gates)
  y = torch.full((M, N // 2), float("nan"), dtype=torch.bfloat16, device=gpu)
  ops.qlinear(ops.make_qlinear_desc(M=M, K=K, N=N, group=64, qtype=Q.NF4, x=x, codes=codes, scales=scales, y=y, epilogue=L.TNX_EPI_SILU_MUL,
                                    split_k=split, ws=torch.empty(split * M * N, device=gpu) if split > 1 else None,
                                    w_expanded=ops.qw_expand(codes, scales, K, N, 64, Q.NF4) if copy else None))
  torch.cuda.synchronize()
  got = y.double().cpu()
  assert (got == got[:, :1]).all()
  want = g * torch.sigmoid(g)
  # one ulp (2^-8 and 2^-8 of the two roundings, the exponential's error may move the first by one), the spacing of bf16 sigmoids
  # below the normal range, and exp(-g) overflows from -88.72 on
  bound = 2.0 ** -7 * 1.01 * want.abs() + g.abs() * 2.0 ** -133 + 2.0 ** -133
  bound = torch.where(g < -88.7, want.abs() + 2.0 ** -133, bound)
  bad = (got[:, 0] - want).abs() > bound
  assert not bad.any(), [(float(a), float(b), float(c)) for a, b, c in zip(g[bad], got[bad, 0], want[bad])][:5]


@pytest.mark.parametrize("M,K,N,split", [
    (128, 4096, 1024, 1),       # 32 k-tiles: two behind the whole turns of the weight ring
    (128, 4096, 1024, 4),       # eight of each split: two
    (100, 1280, 512, 1),        # ten: one
    (600, 640, 24576, 1),       # many rows, from the codes: five, two behind the turn
])
def test_qlinear_lora_repeats_bit_for_bit(gpu, M, K, N, split):
  """The k-tiles behind the last whole turn of the weight ring request no weights, so nothing younger than
  the activations is in flight there: their wait covers all of it.  (One that left as many loads out as in
  the turns multiplied rows of the adapter's block that had not landed, now and then.)"""
  from tunix_amd import ops
  x, t = bf(rnd((M, K), 61)).to(gpu), bf(rnd((M, 64), 62)).to(gpu)
  c, s = ops.quantize_pack(bf(rnd((K, N), 63, 0.02)).to(gpu), 64, Q.NF4)
  lb = bf(rnd((N, 64), 64, 0.1)).to(gpu)
  outs = []
  for _ in range(40):
    y = torch.empty(M, N, dtype=torch.bfloat16, device=gpu)
    ws = torch.empty(split * M * N, dtype=torch.float32, device=gpu) if split > 1 else None
    ops.qlinear(ops.make_qlinear_desc(M=M, K=K, N=N, group=64, qtype=Q.NF4, x=x, codes=c, scales=s, y=y, split_k=split,
                                      ws=ws, lora_rank=64, lora_nseg=1, lora_seg_end=[N], lora_seg_toff=[0], t=t, t_ld=64,
                                      lora_b=lb, lora_scale=2.0))
    outs.append(y)
    torch.cuda.synchronize()
  assert all(torch.equal(outs[0], o) for o in outs[1:])


@pytest.mark.parametrize("M,K,N,group,qtype,r,seg_widths,epi", [
    (1100, 256, 7424, 64, Q.NF4, 64, None, "store"),             # ragged rows, one adapter
    (640, 384, 13312, 128, Q.INT4, 16, [8192, 2560, 2560], "store"),  # three adapter segments, 3 k-tiles
    (520, 128, 13440, 32, Q.NF4, 0, None, "residual"),           # ragged last column tile, group 32, one k-tile
    (1024, 512, 8448, 64, Q.INT4, 32, None, "silu"),             # gate|up pair with its two adapters
    (515, 640, 16896, 64, Q.NF4, 0, None, "gelu"),
    # integer codes are converted without the table: group 32 (four scales per k-tile) over one
    # and over five k-tiles, ragged rows with an adapter
    (520, 128, 13440, 32, Q.INT4, 0, None, "residual"),
    (515, 640, 16896, 32, Q.INT4, 0, None, "gelu"),
    (1100, 256, 7424, 64, Q.INT4, 64, None, "store"),
    # 71 / 66 row blocks: one full group of 64 of the work-group id -> tile map and a ragged one
    (9000, 128, 2048, 64, Q.INT4, 0, None, "store"),
    (8400, 128, 2304, 64, Q.NF4, 16, None, "store"),
])
def test_qlinear_many_rows_matches_oracle(gpu, M, K, N, group, qtype, r, seg_widths, epi):
  """Row counts that go to the 128 x 256-tile kernel (prefill, per-token logps): every epilogue,
  adapter segments, ragged row and column tiles, against the oracle."""
  from tunix_amd import _lib as L
  from tunix_amd import ops
  x = rnd((M, K), 21)
  w = rnd((K, N), 22, 0.02)
  codes, scale = Q.quantize(w.numpy(), group, qtype)
  mul = epi in ("silu", "gelu")
  widths = seg_widths or ([N // 2, N // 2] if mul else [N])
  rp = (r + 31) // 32 * 32 if r else 0
  gx = bf(x).to(gpu)
  a_t = torch.zeros(len(widths) * max(rp, 1), K)
  b_full = torch.zeros(N, max(rp, 1))
  lora = []
  off = 0
  for i, wd in enumerate(widths):
    if r:
      a, b = _lora(K, wd, r, 30 + 2 * i)
      a_t[i * rp: i * rp + r] = a.t()
      b_full[off: off + wd, :r] = b.t()
      lora.append(b)
    off += wd
  t = t_host = None
  if r:
    # t = bf16(x . A) by the kernel for these row counts (128-row MFMA tiles), checked on its own;
    # the linear's reference then uses the kernel's t, so that a t element rounded the other way
    # (one bf16 ulp, allowed) is not counted against the linear
    t = torch.zeros(M, len(widths) * rp, dtype=torch.bfloat16, device=gpu)
    ops.lora_down(gx, bf(a_t).to(gpu), t)
    assert_bf16_close(t, Q.rb((x.double() @ a_t.t().double()).float()), what="lora_down, many rows")
    t_host = t.float().cpu()
  ref = torch.empty(M, N)
  off = 0
  for i, wd in enumerate(widths):
    seg = Q.qlinear_lora(x, codes[:, off: off + wd], scale[:, off: off + wd], group, qtype).double()
    if r:
      seg = seg + 0.5 * (t_host[:, i * rp: i * rp + r].double() @ lora[i].double())
    ref[:, off: off + wd] = seg.float()
    off += wd
  ref = Q.rb(ref)
  res = mag = None
  if epi == "residual":
    res = rnd((M, N), 23)
    mag = ref
    ref = Q.rb(ref + res)
  elif mul:
    gte, up = ref[:, : N // 2], ref[:, N // 2:]
    act = Q.rb(gte * Q.rb(torch.sigmoid(gte))) if epi == "silu" else \
        Q.rb(torch.nn.functional.gelu(gte, approximate="tanh"))
    ref = Q.rb(act * up)
  c, s = ops.quantize_pack(bf(w).to(gpu), group, qtype, mul)
  y = torch.empty(M, N // 2 if mul else N, dtype=torch.bfloat16, device=gpu)
  kw = {}
  if r:
    b_t = b_full
    if mul:
      b_t = torch.zeros_like(b_full)
      b_t[torch.from_numpy(Q.packed_col(np.arange(N), N, True))] = b_full
    ends = list(np.cumsum(widths))
    kw = dict(lora_rank=rp, lora_nseg=-1 if mul else len(widths), lora_seg_end=[int(e) for e in ends],
              lora_seg_toff=[i * rp for i in range(len(widths))], t=t, t_ld=len(widths) * rp,
              lora_b=bf(b_t).to(gpu), lora_scale=0.5)
  e = {"store": L.TNX_EPI_STORE, "residual": L.TNX_EPI_RESIDUAL, "silu": L.TNX_EPI_SILU_MUL,
       "gelu": L.TNX_EPI_GELU_MUL}[epi]
  if res is not None:
    kw["residual"] = bf(res).to(gpu)
  ops.qlinear(ops.make_qlinear_desc(M=M, K=K, N=N, group=group, qtype=qtype, x=gx, codes=c, scales=s, y=y,
                                    epilogue=e, **kw))
  # the same call fed with the converted second copy of the weight (the fragments the kernel
  # would have formed from the codes): bit for bit the same output
  y2 = torch.full_like(y, float("nan"))
  ops.qlinear(ops.make_qlinear_desc(M=M, K=K, N=N, group=group, qtype=qtype, x=gx, codes=c, scales=s, y=y2,
                                    epilogue=e, w_expanded=ops.qw_expand(c, s, K, N, group, qtype), **kw))
  torch.cuda.synchronize()
  assert torch.equal(y.view(torch.int16), y2.view(torch.int16)), "expanded weights: output differs"
  # act(gate) * up: gate and up may each be one ulp off; linear + residual: a linear output one ulp
  # off can move the rounded sum by one more step of the sum's own (finer) spacing
  assert_bf16_close(y, ref, atol=1e-5 if mul else 1e-6, min_equal=0.9 if mul else 0.97, what=f"wide {epi}", mag=mag,
                    ulps=3 if mul else 2 if epi == "residual" else 1)


@pytest.mark.parametrize("M,K,N,group,qtype,r,epi,reads", [
    (128, 256, 33024, 64, Q.NF4, 0, "store", False),      # 258 tiles of 128 x 128, but one row block
    (129, 256, 16384, 64, Q.NF4, 32, "residual", False),  # 256 tiles: one turn of the device
    (129, 256, 16400, 64, Q.NF4, 32, "store", True),      # 258, a ragged last column tile and a row block of one row
    (300, 128, 11008, 32, Q.INT4, 64, "silu", True),      # 258
    (1300, 1152, 3072, 128, Q.INT4, 0, "residual", True),  # 264
    (1024, 384, 4096, 64, Q.INT4, 64, "gelu", False),     # 256
])
def test_linears_between_the_kernels_read_their_copy(gpu, M, K, N, group, qtype, r, epi, reads):
  """Fewer rows and tiles than the many-row kernel takes from the codes: a linear with a converted copy goes there as soon as
  128 x 128 tiles no longer fit the device in one turn (a copy of NaN shows which calls read it), with the sums of the codes."""
  from tunix_amd import _lib as L
  from tunix_amd import ops
  mul = epi in ("silu", "gelu")
  c, s = ops.quantize_pack(bf(rnd((K, N), 702, 0.02)).to(gpu), group, qtype, mul)
  kw = {}
  if epi == "residual":
    kw["residual"] = bf(rnd((M, N), 703)).to(gpu)
  if r:
    widths = [N // 2, N // 2] if mul else [N]
    kw.update(lora_rank=r, lora_nseg=-1 if mul else 1, lora_seg_end=[int(e) for e in np.cumsum(widths)], lora_seg_toff=[i * r for i in range(len(widths))],
              t=bf(rnd((M, len(widths) * r), 704)).to(gpu), t_ld=len(widths) * r, lora_b=bf(rnd((N, r), 705, 0.1)).to(gpu), lora_scale=0.5)
  e = {"store": L.TNX_EPI_STORE, "residual": L.TNX_EPI_RESIDUAL, "silu": L.TNX_EPI_SILU_MUL, "gelu": L.TNX_EPI_GELU_MUL}[epi]
  x = bf(rnd((M, K), 701)).to(gpu)
  copy = ops.qw_expand(c, s, K, N, group, qtype)
  outs = []
  for exp in (None, copy, torch.full_like(copy, float("nan"))):
    y = torch.full((M, N // 2 if mul else N), float("nan"), dtype=torch.bfloat16, device=gpu)
    ops.qlinear(ops.make_qlinear_desc(M=M, K=K, N=N, group=group, qtype=qtype, x=x, codes=c, scales=s, y=y, epilogue=e, w_expanded=exp, **kw))
    outs.append(y)
  torch.cuda.synchronize()
  assert bool(outs[2].isnan().any()) == reads
  assert not outs[0].isnan().any()
  # the same bf16 products in another order of the float32 sum: one step of bf16 where a sum lies between two, which the gate and
  # the residual's own rounding can make two and three
  assert_bf16_close(outs[1], outs[0].float().cpu(), atol=1e-5 if mul else 1e-6, min_equal=0.9, what=f"copy {epi}",
                    mag=(outs[0].float() - kw["residual"].float()).cpu() if epi == "residual" else None, ulps=3 if mul else 2 if epi == "residual" else 1)


@pytest.mark.parametrize("M,K,R", [(12300, 256, 192), (6200, 384, 128), (700, 128, 32)])
def test_lora_down_many_rows(gpu, M, K, R):
  """The MFMA flavours of the LoRA down-projection (128-, 64- and 32-row tiles, chosen by how many
  work-groups the shape yields) against the oracle; t is written only in its R columns."""
  from tunix_amd import ops
  x, a_t = rnd((M, K), 41), rnd((R, K), 42, 0.02)
  t = torch.full((M, R + 32), 7.0, dtype=torch.bfloat16, device=gpu)
  ops.lora_down(bf(x).to(gpu), bf(a_t).to(gpu), t)
  assert_bf16_close(t[:, :R], Q.rb((x.double() @ a_t.t().double()).float()), what="lora_down rows")
  assert (t[:, R:].float() == 7.0).all()


@pytest.mark.parametrize("M,K,R", [(128, 4096, 64), (128, 4096, 192), (128, 14336, 64), (128, 6912, 128),
                                   (8, 512, 32), (64, 1152, 16), (33, 2048, 128), (100, 96, 48), (5, 20480, 16)])
def test_lora_down_decode_sizes(gpu, M, K, R):
  """The down-projection at decode sizes: operand rows through LDS whole (K * rows fits), in pieces
  (long rows), and the direct kernel (K not a multiple of 64); columns past R stay untouched."""
  from tunix_amd import ops
  x, a_t = rnd((M, K), 43), rnd((R, K), 44, 0.02)
  t = torch.full((M, R + 32), 7.0, dtype=torch.bfloat16, device=gpu)
  ops.lora_down(bf(x).to(gpu), bf(a_t).to(gpu), t)
  assert_bf16_close(t[:, :R], Q.rb((bf(x).double() @ bf(a_t).t().double()).float()), what="lora_down decode")
  assert (t[:, R:].float() == 7.0).all()


def test_qlinear_invariants(gpu):
  """Zero codes give zero; B = 0 leaves the base result; scale linearity (exact powers of 2)."""
  from tunix_amd import ops
  M, K, N, g = 16, 256, 64, 64
  x = rnd((M, K), 5)
  w = rnd((K, N), 6, 0.02)

  def run(wt, lora=None):
    c, s = ops.quantize_pack(bf(wt).to(gpu), g, Q.NF4)
    y = torch.empty(M, N, dtype=torch.bfloat16, device=gpu)
    kw = {}
    if lora is not None:
      a_t, b_t = lora
      t = torch.zeros(M, 32, dtype=torch.bfloat16, device=gpu)
      ops.lora_down(bf(x).to(gpu), bf(a_t).to(gpu), t)
      kw = dict(lora_rank=32, lora_nseg=1, lora_seg_end=[N], lora_seg_toff=[0], t=t, t_ld=32,
                lora_b=bf(b_t).to(gpu), lora_scale=1.0)
    ops.qlinear(ops.make_qlinear_desc(M=M, K=K, N=N, group=g, qtype=Q.NF4, x=bf(x).to(gpu),
                                      codes=c, scales=s, y=y, **kw))
    return y.float().cpu()

  assert run(torch.zeros(K, N)).abs().max().item() == 0.0
  base = run(w)
  a_t = rnd((32, K), 7, 0.02)
  assert torch.equal(run(w, (a_t, torch.zeros(N, 32))), base)
  assert torch.equal(run(w * 4.0), base * 4.0)


@pytest.mark.parametrize("M", [1, 8, 16, 32, 40])
@pytest.mark.parametrize("epi", ["silu", "gelu", "residual"])
def test_qlinear_epilogues(gpu, epi, M):
  from tunix_amd import _lib as L
  from tunix_amd import ops
  K, F, g = 512, 256, 64
  x = rnd((M, K), 8)
  if epi == "residual":
    w = rnd((K, F), 9, 0.02)
    res = rnd((M, F), 10)
    codes, scale = Q.quantize(w.numpy(), g, Q.INT4)
    ref = Q.rb(Q.rb(Q.qlinear_lora(x, codes, scale, g, Q.INT4)) + res)
    c, s = ops.quantize_pack(bf(w).to(gpu), g, Q.INT4)
    y = torch.empty(M, F, dtype=torch.bfloat16, device=gpu)
    ops.qlinear(ops.make_qlinear_desc(M=M, K=K, N=F, group=g, qtype=Q.INT4, x=bf(x).to(gpu), codes=c,
                                      scales=s, y=y, epilogue=L.TNX_EPI_RESIDUAL,
                                      residual=bf(res).to(gpu)))
    assert_bf16_close(y, ref, what="residual epilogue")
    return
  wg, wu = rnd((K, F), 9, 0.05), rnd((K, F), 10, 0.05)
  cg, sg = Q.quantize(wg.numpy(), g, Q.INT4)
  cu, su = Q.quantize(wu.numpy(), g, Q.INT4)
  gte = Q.rb(Q.qlinear_lora(x, cg, sg, g, Q.INT4))
  up = Q.rb(Q.qlinear_lora(x, cu, su, g, Q.INT4))
  if epi == "silu":
    act = Q.rb(gte * Q.rb(torch.sigmoid(gte)))
  else:
    act = Q.rb(torch.nn.functional.gelu(gte, approximate="tanh"))
  ref = Q.rb(act * up)
  c, s = ops.quantize_pack(bf(torch.cat([wg, wu], 1)).to(gpu), g, Q.INT4, True)
  y = torch.empty(M, F, dtype=torch.bfloat16, device=gpu)
  ops.qlinear(ops.make_qlinear_desc(
      M=M, K=K, N=2 * F, group=g, qtype=Q.INT4, x=bf(x).to(gpu), codes=c, scales=s, y=y,
      epilogue=L.TNX_EPI_SILU_MUL if epi == "silu" else L.TNX_EPI_GELU_MUL))
  assert_bf16_close(y, ref, atol=1e-5, min_equal=0.9, what=f"{epi} epilogue")


class _Cfg:
  def __init__(self, family, eps=1e-6):
    self.family, self.norm_eps = family, eps


@pytest.mark.parametrize("family", ["llama3", "qwen3", "gemma3"])
def test_rmsnorm_flavours(gpu, family):
  from tunix_amd import ops
  from tunix_amd.model import _NORM
  M, D = 37, 1152
  x, res = rnd((M, D), 20, 2.0), rnd((M, D), 21)
  w = rnd((D,), 22, 0.5) + (0.0 if family == "gemma3" else 1.0)
  w = Q.rb(w)
  ref_m = MR.RefModel.__new__(MR.RefModel)
  ref_m.cfg, ref_m.bf16 = _Cfg(family, 1e-5), True
  ref = ref_m.rmsnorm(x, w)
  y = torch.empty(M, D, dtype=torch.bfloat16, device=gpu)
  ops.rmsnorm(bf(x).to(gpu), bf(w).to(gpu), y, 1e-5 if family != "gemma3" else 1e-6, _NORM[family])
  assert_bf16_close(y, ref, min_equal=0.95, what=f"rmsnorm {family}")
  # residual variants
  h = Q.rb(x + res)
  ref2 = Q.rb(ref_m.rmsnorm(h, w) + res)
  y2 = torch.empty_like(y)
  hout = torch.empty_like(y)
  ops.rmsnorm(bf(x).to(gpu), bf(w).to(gpu), y2, 1e-5 if family != "gemma3" else 1e-6, _NORM[family],
              res_pre=bf(res).to(gpu), h_out=hout, res_post=bf(res).to(gpu))
  assert torch.equal(hout.float().cpu(), h)
  assert_bf16_close(y2, ref2, min_equal=0.95, what=f"rmsnorm+residual {family}")


@pytest.mark.parametrize("family,D,split", [("llama3", 5120, 3), ("qwen3", 9216, 2), ("gemma3", 16384, 1),
                                            ("llama3", 4096, 11), ("gemma3", 1152, 9)])
def test_rmsnorm_wide_rows_and_many_planes(gpu, family, D, split):
  """The instances of the vector norm for 4 and 8 chunks per thread (rows wider than 4096) and
  the path for more than eight partial planes: a bf16 row against the oracle, and the same row
  handed over as `split` fp32 planes (summed in split order, rounded to bf16) bit-equal to it."""
  from tunix_amd import ops
  from tunix_amd.model import _NORM
  M = 5
  eps = 1e-6 if family == "gemma3" else 1e-5
  g = torch.Generator().manual_seed(300 + D + split)
  planes = torch.randn(split, M, D, generator=g) * (1.5 / split ** 0.5)
  acc = torch.zeros(M, D)
  for z in range(split):
    acc = acc + planes[z]
  x = Q.rb(acc)
  res = rnd((M, D), 301)
  w = Q.rb(rnd((D,), 302, 0.5) + (0.0 if family == "gemma3" else 1.0))
  ref_m = MR.RefModel.__new__(MR.RefModel)
  ref_m.cfg, ref_m.bf16 = _Cfg(family, eps), True
  h = Q.rb(x + res)
  ref = ref_m.rmsnorm(h, w)
  y1, h1 = (torch.empty(M, D, dtype=torch.bfloat16, device=gpu) for _ in range(2))
  ops.rmsnorm(bf(x).to(gpu), bf(w).to(gpu), y1, eps, _NORM[family], res_pre=bf(res).to(gpu), h_out=h1)
  assert torch.equal(h1.float().cpu(), h)
  assert_bf16_close(y1, ref, min_equal=0.95, what=f"rmsnorm {family} D={D}")
  y2, h2 = torch.empty_like(y1), bf(res).to(gpu)
  ops.rmsnorm_splitk(planes.to(gpu).contiguous().view(-1), split, bf(w).to(gpu), y2, eps, _NORM[family], M, D,
                     res_pre=h2, h_out=h2)
  torch.cuda.synchronize()
  assert torch.equal(h1, h2) and torch.equal(y1, y2)


@pytest.mark.parametrize("family,dh,Hq,Hkv", [("llama3", 128, 8, 2), ("qwen3", 64, 8, 2),
                                               ("gemma3", 256, 4, 1),
                                               # half a head is not whole waves
                                               ("qwen3", 160, 3, 1), ("qwen3", 192, 4, 2), ("gemma3", 320, 2, 1), ("qwen3", 34, 2, 1)])
def test_rope_kvwrite(gpu, family, dh, Hq, Hkv):
  from tunix_amd import _lib as L
  from tunix_amd import ops
  from tunix_amd.model import _NORM, _ROPE, rope_timescale
  B, T, S = 3, 5, 16
  col = 4
  theta = 1e6 if family != "gemma3" else 1e4
  qkv = rnd((B * T, (Hq + 2 * Hkv) * dh), 30)
  pos = torch.randint(0, 900, (B, S), generator=torch.Generator().manual_seed(31), dtype=torch.int32)
  qn, kn = Q.rb(rnd((dh,), 32, 0.3) + 1), Q.rb(rnd((dh,), 33, 0.3) + 1)
  rm = MR.RefModel.__new__(MR.RefModel)
  rm.cfg, rm.bf16 = _Cfg(family), True
  x = qkv.view(B, T, Hq + 2 * Hkv, dh)
  q, k, v = x[:, :, :Hq], x[:, :, Hq:Hq + Hkv], x[:, :, Hq + Hkv:]
  if family != "llama3":
    q, k = rm.rmsnorm(q, qn), rm.rmsnorm(k, kn)
  p = pos[:, col:col + T].long()
  sf = 8.0 if family == "gemma3" else 1.0
  q, k = rm.rope(q, p, theta, scale_factor=sf), rm.rope(k, p, theta, scale_factor=sf)
  if family == "gemma3":
    q = Q.rb(q * Q.rb(torch.tensor(dh ** -0.5)))
  d = L.RopeDesc()
  d.B, d.T, d.S, d.Hq, d.Hkv, d.dh = B, T, S, Hq, Hkv, dh
  d.rope_flavor, d.rope_scale = _ROPE[family], sf
  ts = torch.from_numpy(rope_timescale(dh, theta)).to(gpu)
  d.timescale = ts.data_ptr()
  wq, wk = bf(qn).to(gpu), bf(kn).to(gpu)
  if family != "llama3":
    d.qk_norm, d.norm_eps, d.q_norm_w, d.k_norm_w = _NORM[family], 1e-6, wq.data_ptr(), wk.data_ptr()
  else:
    d.qk_norm = -1
  d.q_prescale = dh ** -0.5 if family == "gemma3" else 0.0
  g_qkv, g_pos = bf(qkv).to(gpu), pos.to(gpu)
  colp = torch.tensor([col], dtype=torch.int32, device=gpu)
  qo = torch.empty(B * T, Hq * dh, dtype=torch.bfloat16, device=gpu)
  kc = torch.zeros(B, Hkv, S, dh, dtype=torch.bfloat16, device=gpu)
  vc = torch.zeros_like(kc)
  d.qkv, d.positions, d.pos_ld, d.col_ptr = g_qkv.data_ptr(), g_pos.data_ptr(), S, colp.data_ptr()
  d.q_out, d.kcache, d.vcache = qo.data_ptr(), kc.data_ptr(), vc.data_ptr()
  ops.rope_kvwrite(d)
  torch.cuda.synchronize()
  assert_bf16_close(qo.view(B, T, Hq, dh), q, min_equal=0.9, what="rope q")
  assert_bf16_close(kc[:, :, col:col + T].permute(0, 2, 1, 3), k, min_equal=0.9, what="rope k")
  assert torch.equal(vc[:, :, col:col + T].permute(0, 2, 1, 3).float().cpu(), v)
  assert kc[:, :, :col].abs().max().item() == 0 and kc[:, :, col + T:].abs().max().item() == 0


def _attn_ref(q, kc, vc, tokens, pad_id, col, T, scale, window):
  """Oracle attention with the dense masks of the reference."""
  from oracle import utils_ref as U
  B, S = kc.shape[0], kc.shape[2]
  rm = MR.RefModel.__new__(MR.RefModel)
  rm.bf16, rm.acc = True, torch.float64
  k_all, v_all = kc.permute(0, 2, 1, 3), vc.permute(0, 2, 1, 3)
  tok = tokens.numpy()
  if T == 1:
    mask = U.compute_attention_masks(col, S, tok == pad_id)
    if window:
      mask = U.create_sliding_window_mask(mask, window) & mask
  else:
    assert col == 0
    mask = U.make_causal_attn_mask(tok[:, :T] != pad_id, S)
    if window:
      ones = torch.ones(T, S, dtype=torch.bool)
      sm = (torch.triu(ones, -window + 1) & torch.tril(ones, window - 1)).numpy()
      mask = mask & sm[None]
  return rm.attention(q, k_all, v_all, torch.from_numpy(mask), scale)


@pytest.mark.parametrize("B,T,S,Hq,Hkv,dh,col,chunk,window", [
    (4, 1, 64, 8, 2, 64, 37, 0, 0),
    (4, 1, 320, 8, 2, 128, 300, 64, 0),
    (3, 1, 128, 4, 1, 256, 100, 32, 48),
    (2, 1, 96, 32, 4, 128, 95, 32, 0),
    (2, 1, 64, 6, 2, 128, 20, 0, 0),
    (3, 24, 32, 8, 2, 64, 0, 0, 0),
    (2, 40, 64, 4, 1, 256, 0, 0, 16),
    (3, 1, 70, 8, 2, 128, 50, 0, 0),      # rows of 70 slots: the token ids are read one by one
    (2, 1, 106, 8, 2, 64, 101, 0, 0),     # four whole key blocks, none left over; 106 % 4 != 0
    (2, 1, 256, 8, 2, 128, 160, 0, 0),    # five key blocks: two turns of the ring and one left over
])
def test_gqa_attention_matches_oracle(gpu, B, T, S, Hq, Hkv, dh, col, chunk, window):
  from tunix_amd import _lib as L
  from tunix_amd import ops
  pad = 0
  g = torch.Generator().manual_seed(40 + S)
  tokens = torch.randint(1, 100, (B, S), generator=g, dtype=torch.int32)
  tokens[0, :5] = pad            # left padding
  tokens[1, 7] = pad             # a pad id inside the sequence is masked as well
  q = rnd((B, T, Hq, dh), 41)
  kc, vc = rnd((B, Hkv, S, dh), 42), rnd((B, Hkv, S, dh), 43)
  scale = dh ** -0.5
  ref = _attn_ref(q, kc, vc, tokens, pad, col, T, scale, window)
  # slots above the current column hold garbage that must not matter
  kc_g, vc_g = kc.clone(), vc.clone()
  kc_g[:, :, col + T:] = 1e4
  vc_g[:, :, col + T:] = 1e4
  d = L.AttnDesc()
  d.B, d.T, d.S, d.Hq, d.Hkv, d.dh = B, T, S, Hq, Hkv, dh
  d.scale, d.window, d.pad_id = scale, window, pad
  gq, gk, gv = bf(q).reshape(B * T, Hq * dh).to(gpu), bf(kc_g).to(gpu), bf(vc_g).to(gpu)
  gt = tokens.to(gpu)
  colp = torch.tensor([col], dtype=torch.int32, device=gpu)
  out = torch.zeros(B * T, Hq * dh, dtype=torch.bfloat16, device=gpu)
  nb = ops.attn_ws_bytes(B, T, S, Hq, dh, chunk)
  ws = torch.empty(max(nb // 4, 1), dtype=torch.float32, device=gpu)
  d.q, d.kcache, d.vcache, d.tokens, d.tok_ld = gq.data_ptr(), gk.data_ptr(), gv.data_ptr(), gt.data_ptr(), S
  d.col_ptr, d.kv_chunk, d.ws, d.out = colp.data_ptr(), chunk, ws.data_ptr(), out.data_ptr()
  ops.gqa_attn(d)
  torch.cuda.synchronize()
  got = out.view(B, T, Hq, dh).float().cpu()
  # rows whose query token is itself pad attend nothing in the reference's mask: skip them
  valid = torch.ones(B, T, dtype=torch.bool)
  for b in range(B):
    for t in range(T):
      c = col + t
      if not ((tokens[b, :c + 1] != pad).any()):
        valid[b, t] = False
  diff = (got - ref).abs()[valid]
  # probabilities are rounded to bf16 before (oracle) or after (kernel, online softmax) the
  # normalisation, so outputs agree to bf16 resolution of O(1) values, not bit for bit
  assert diff.max().item() <= 2.0 ** -6 * max(1.0, ref.abs().max().item()), diff.max().item()
  assert diff.mean().item() <= 2e-3


@pytest.mark.parametrize("B,T,S,Hq,Hkv,col,window,seg", [
    (2, 256, 256, 8, 2, 0, 0, False),       # 64 query tiles per row: eight work-groups of eight tiles
    (3, 200, 320, 32, 8, 40, 0, False),     # a ragged last group, queries that start at column 40
    (2, 192, 192, 8, 1, 0, 48, False),      # sliding window: blocks before a tile's window are skipped
    (2, 272, 272, 4, 4, 0, 0, True),        # one query head per kv head, a packed batch (segment ids)
    (1, 100, 128, 16, 2, 0, 0, False),      # eight query heads per kv head: two positions per tile
])
def test_gqa_attention_through_lds_takes_rows_of_ids_off_alignment(gpu, B, T, S, Hq, Hkv, col, window, seg):
  """Many query positions at head_dim 128, keys and values staged through LDS: rows of ids that start off a 16-byte boundary
  give the bits that aligned ones give, pads inside the rows included; and the result against the oracle, or, for columns and segments that
  its masks do not cover, against plain attention in 64 bits.  (Against the kernel in which every wave loads its own keys:
  test_gqa_attention_many_positions_equals_few.)"""
  from tunix_amd import _lib as L
  from tunix_amd import ops
  dh, pad = 128, 0
  g = torch.Generator().manual_seed(70 + T)
  if seg:
    ids = torch.sort(torch.randint(1, 4, (B, S), generator=g, dtype=torch.int32), dim=1).values
  else:
    ids = torch.randint(1, 100, (B, S), generator=g, dtype=torch.int32)
    ids[0, :5] = pad
    ids[B - 1, 9] = pad
  q = bf(rnd((B, T, Hq, dh), 71)).reshape(B * T, Hq * dh).to(gpu)
  kc, vc = bf(rnd((B, Hkv, S, dh), 72)).to(gpu), bf(rnd((B, Hkv, S, dh), 73)).to(gpu)
  colp = torch.tensor([col], dtype=torch.int32, device=gpu)
  aligned = ids.to(gpu).contiguous()
  shifted_buf = torch.zeros(B * (S + 4) + 4, dtype=torch.int32, device=gpu)
  shifted = shifted_buf[1: 1 + B * (S + 4)].view(B, S + 4)       # rows start 4 bytes off a 16-byte boundary
  shifted[:, :S] = aligned
  outs = []
  for tk, ld in ((aligned, S), (shifted, S + 4)):
    d = L.AttnDesc()
    d.B, d.T, d.S, d.Hq, d.Hkv, d.dh = B, T, S, Hq, Hkv, dh
    d.scale, d.window, d.pad_id = dh ** -0.5, window, pad
    out = torch.full((B * T, Hq * dh), 7.0, dtype=torch.bfloat16, device=gpu)
    d.q, d.kcache, d.vcache = q.data_ptr(), kc.data_ptr(), vc.data_ptr()
    if seg:
      d.segment_ids = tk.data_ptr()
    else:
      d.tokens = tk.data_ptr()
    d.tok_ld, d.col_ptr, d.kv_chunk, d.out = ld, colp.data_ptr(), 0, out.data_ptr()
    ops.gqa_attn(d)
    outs.append(out)
  torch.cuda.synchronize()
  assert shifted.data_ptr() % 16 != 0 and aligned.data_ptr() % 16 == 0
  assert torch.equal(outs[0].view(torch.int16), outs[1].view(torch.int16))
  got = outs[0].view(B, T, Hq, dh).float().cpu()
  qr, kr, vr = q.float().cpu().view(B, T, Hq, dh), kc.float().cpu(), vc.float().cpu()
  at, key = torch.arange(T)[:, None] + col, torch.arange(S)[None]
  mask = ((key <= at) & (at - key < window) if window else key <= at)[None] & \
      (ids[:, None, :] == ids[:, col:col + T, None] if seg else ids[:, None, :] != pad)
  valid = mask.any(-1) & (ids[:, col:col + T] != pad)
  if not seg and col == 0:
    ref = _attn_ref(qr, kr, vr, ids, pad, col, T, dh ** -0.5, window)
  else:
    heads = lambda x: x.repeat_interleave(Hq // Hkv, 1).double()
    score = (qr.permute(0, 2, 1, 3).double() @ heads(kr).transpose(2, 3) * dh ** -0.5).masked_fill(~mask[:, None], -1e30)
    ref = (torch.softmax(score, -1) @ heads(vr)).permute(0, 2, 1, 3).float()
  diff = (got - ref).abs()[valid]
  assert valid.float().mean() > 0.9 and diff.max().item() <= 2.0 ** -6 * max(1.0, ref[valid].abs().max().item()), diff.max().item()


@pytest.mark.parametrize("B,T,S,Hq,Hkv,col,window,seg,scale", [
    (2, 61, 61, 8, 2, 0, 0, False, None),        # fewest tiles of the work-group form, odd rows of ids and slots
    (3, 131, 333, 6, 2, 77, 0, False, 1.0),      # three query heads in lanes of four, queries from column 77, no scaling
    (1, 1023, 1023, 4, 4, 0, 0, True, None),     # a packed batch of several segments, one head per kv head
    (2, 259, 263, 8, 1, 3, 40, False, None),     # a window inside two key blocks
    (1, 65, 70, 32, 2, 5, 0, True, 0.125),       # sixteen heads per kv head: one position per tile
])
def test_gqa_attention_many_positions_equals_few(gpu, B, T, S, Hq, Hkv, col, window, seg, scale):
  """head_dim 128: all positions in one call (keys and values through LDS) against calls of a few
  positions each (every wave loads its own), bit for bit: the same blocks in the same order with the
  same arithmetic."""
  from tunix_amd import _lib as L
  from tunix_amd import ops
  dh, pad = 128, 0
  g = torch.Generator().manual_seed(90 + T)
  if seg:
    ids = torch.sort(torch.randint(1, 5, (B, S), generator=g, dtype=torch.int32), dim=1).values
  else:
    ids = torch.randint(1, 100, (B, S), generator=g, dtype=torch.int32)
    ids[0, :5] = pad
    ids[B - 1, 9] = pad
  q = bf(rnd((B, T, Hq * dh), 91)).to(gpu)
  kc, vc = bf(rnd((B, Hkv, S, dh), 92)).to(gpu), bf(rnd((B, Hkv, S, dh), 93)).to(gpu)
  ids = ids.to(gpu).contiguous()

  def attn(t0, n):
    qs = q[:, t0:t0 + n].contiguous()
    out = torch.full((B, n, Hq * dh), 7.0, dtype=torch.bfloat16, device=gpu)
    colp = torch.tensor([col + t0], dtype=torch.int32, device=gpu)
    d = L.AttnDesc()
    d.B, d.T, d.S, d.Hq, d.Hkv, d.dh = B, n, S, Hq, Hkv, dh
    d.scale, d.window, d.pad_id = dh ** -0.5 if scale is None else scale, window, pad
    d.q, d.kcache, d.vcache, d.out = qs.data_ptr(), kc.data_ptr(), vc.data_ptr(), out.data_ptr()
    if seg:
      d.segment_ids = ids.data_ptr()
    else:
      d.tokens = ids.data_ptr()
    d.tok_ld, d.col_ptr, d.kv_chunk = S, colp.data_ptr(), 0
    ops.gqa_attn(d)
    torch.cuda.synchronize()
    return out

  whole = attn(0, T)
  G = Hq // Hkv
  few = 3 * max(1, 16 // (1 << (G - 1).bit_length()))       # three tiles of queries
  parts = torch.cat([attn(t0, min(few, T - t0)) for t0 in range(0, T, few)], dim=1)
  assert torch.isfinite(whole.float()).all()
  assert torch.equal(whole.view(torch.int16), parts.view(torch.int16))


@pytest.mark.parametrize("T,col,window", [(62, 0, 0), (62, 2, 0), (62, 3, 0), (62, 35, 0), (62, 66, 0), (62, 67, 0),   # 2, 2, 3, 4, 4, 5 key blocks
                                          (93, 31, 30), (93, 33, 33), (64, 64, 1)])    # windows that start on either block of a pair
def test_attention_key_blocks_in_pairs(gpu, T, col, window):
  """Numbers of key blocks around the pair that a work-group takes behind one barrier, its waves starting and ending at either of the two.  (No
  number of positions that leaves a single one for the last of the calls compared with: one position's keys are divided among waves.)"""
  test_gqa_attention_many_positions_equals_few(gpu, 2, T, col + T + 1, 8, 2, col, window, False, None)


@pytest.mark.parametrize("M,D,V,temperature", [(1, 128, 65536, 1.0), (17, 384, 65552, 0.7), (64, 256, 66000, 1.0),
                                               (65, 256, 65536, 1.0), (128, 128, 65600, 1.0)])
def test_dense_head_over_few_rows_equals_many(gpu, M, D, V, temperature):
  """A dense head's copy over at most 64 rows takes a tile of 64 rows (up to 128: one of 128): every statistic is bit for bit that
  of the same rows inside a call of 200 (the sums run over the same k in the same order)."""
  from tunix_amd import _lib as L
  from tunix_amd import ops
  w = bf(rnd((V, D), 101, 0.05)).to(gpu)
  we = ops.dense_expand(w)
  x = bf(rnd((200, D), 102)).to(gpu)
  targets = torch.randint(0, V, (200,), generator=torch.Generator().manual_seed(103), dtype=torch.int32).to(gpu)

  def run(n):
    d = L.LmHeadDesc()
    nvb = (V + 127) // 128
    part = torch.full((n, nvb, 4), float("nan"), device=gpu)
    out = [torch.empty(n, dtype=t, device=gpu) for t in (torch.int32, torch.float32, torch.float32, torch.float32)]
    d.M, d.D, d.V, d.x, d.w_bf16, d.w_expanded = n, D, V, x.data_ptr(), w.data_ptr(), we.data_ptr()
    d.targets, d.part, d.temperature = targets.data_ptr(), part.data_ptr(), temperature
    d.best_id, d.best_logp, d.target_logp, d.lse = (o.data_ptr() for o in out)
    ops.lmhead(d)
    torch.cuda.synchronize()
    return out, part

  (few, fp), (many, mp) = run(M), run(200)
  assert torch.isfinite(few[3]).all()
  for a, b in zip(few, many):
    assert torch.equal(a, b[:M])
  assert torch.equal(fp.view(torch.int32), mp[:M].view(torch.int32))
  ref = torch.log_softmax((x[:M].float().cpu() @ w.float().cpu().T).bfloat16().float() / temperature, -1)
  got = few[2].cpu()
  want = ref.gather(1, targets[:M].long().cpu()[:, None])[:, 0]
  # (a logit may round to the neighbouring bf16 value: one ulp of the largest, scaled by the temperature)
  assert (got - want).abs().max() <= 2.0 ** -7 * ref.abs().max() / temperature


@pytest.mark.parametrize("M,D,V,dense", [(8, 512, 32000, True), (128, 512, 4096, True),
                                         (130, 256, 1040, True),   # two row blocks, partial last column block
                                         (50, 256, 1040, False), (130, 256, 4096, False)])
def test_lmhead_greedy_and_logp(gpu, M, D, V, dense):
  from tunix_amd import _lib as L
  from tunix_amd import ops
  x = rnd((M, D), 50)
  w = rnd((D, V), 51, 0.05)
  g = torch.Generator().manual_seed(52)
  targets = torch.randint(0, V, (M,), generator=g, dtype=torch.int32)
  d = L.LmHeadDesc()
  d.M, d.D, d.V = M, D, V
  gx = bf(x).to(gpu)
  d.x = gx.data_ptr()
  keep = []
  if dense:
    logits = Q.rb((x.double() @ w.double()).float())
    gw = bf(w).t().contiguous().to(gpu)
    d.w_bf16 = gw.data_ptr()
  else:
    codes, scale = Q.quantize(w.numpy(), 128, Q.INT4)
    a, b = _lora(D, V, 32, 53)
    logits = Q.rb(Q.qlinear_lora(x, codes, scale, 128, Q.INT4, a, b, lora_scale=1.0))
    c, s = ops.quantize_pack(bf(w).to(gpu), 128, Q.INT4)
    a_t, b_t = _pad_lora(a, b, 32)
    t = torch.zeros(M, 32, dtype=torch.bfloat16, device=gpu)
    ops.lora_down(gx, bf(a_t).to(gpu), t)
    gb = bf(b_t).to(gpu)
    d.codes, d.scales, d.group, d.qtype = c.data_ptr(), s.data_ptr(), 128, Q.INT4
    d.lora_rank, d.t, d.t_ld, d.lora_b, d.lora_scale = 32, t.data_ptr(), 32, gb.data_ptr(), 1.0
    keep += [c, s, t, gb]
  temperature = 0.7
  d.temperature = temperature
  nvb = ops.lmhead_nblocks(V)
  part = torch.empty(M * nvb * 4, dtype=torch.float32, device=gpu)
  best = torch.empty(M, dtype=torch.int32, device=gpu)
  blp = torch.empty(M, dtype=torch.float32, device=gpu)
  tlp = torch.empty(M, dtype=torch.float32, device=gpu)
  lse = torch.empty(M, dtype=torch.float32, device=gpu)
  lg_out = torch.empty(M, V, dtype=torch.float32, device=gpu)
  gt = targets.to(gpu)
  d.targets, d.part, d.best_id, d.best_logp = gt.data_ptr(), part.data_ptr(), best.data_ptr(), blp.data_ptr()
  d.target_logp, d.lse, d.logits_out = tlp.data_ptr(), lse.data_ptr(), lg_out.data_ptr()
  ops.lmhead(d)
  torch.cuda.synchronize()
  raw_logits = lg_out.cpu()
  scaled = logits / np.float32(temperature)
  # the materialised logits are the raw bf16 values; the statistics use logits / T
  assert_bf16_close(raw_logits, logits, atol=1e-6, min_equal=0.97, what="logits")
  got_logits = raw_logits / np.float32(temperature)
  # the fused statistics must agree with the logits the kernel itself produced
  ref_best = torch.from_numpy(np.argmax(got_logits.numpy(), axis=-1))
  assert torch.equal(best.cpu().long(), ref_best), "arg-max (first maximal index)"
  ref_lse = torch.logsumexp(got_logits, dim=-1)
  np.testing.assert_allclose(lse.cpu().numpy(), ref_lse.numpy(), rtol=0, atol=2e-5)
  ref_t = rl_ref.selective_log_softmax(got_logits, targets)
  np.testing.assert_allclose(tlp.cpu().numpy(), ref_t.numpy(), rtol=0, atol=2e-5)
  np.testing.assert_allclose(blp.cpu().numpy(), (got_logits.max(-1).values - ref_lse).numpy(), atol=2e-5)
  # and with the oracle's logits within the bf16 tolerance of the path
  ref_t2 = rl_ref.selective_log_softmax(scaled, targets)
  assert (tlp.cpu() - ref_t2).abs().max().item() < 2e-2


@pytest.mark.parametrize("M,D,V,group,qtype,r,entropy", [(1030, 256, 8208, 128, Q.INT4, 64, True),
                                                         (2048, 384, 4096, 64, Q.NF4, 0, False),
                                                         (640, 256, 16384, 64, Q.NF4, 32, True)])
def test_lmhead_many_rows_quantized_head(gpu, M, D, V, group, qtype, r, entropy):
  """The quantised head from 512 rows on (per-token log-probabilities at training scale) runs on
  the many-rows GEMM kernel with a statistics epilogue.  Tight check: the plain linear of the
  same kernel materialises the very logits the epilogue sees, and arg-max, logsumexp, target
  log-probability and entropy must follow from them (ids exact, 2e-5).  Against the oracle's
  logits: the tolerance of the bf16 path (2e-2).  Cases: a partial last row tile and a last
  column tile of 16 columns; no adapter; an odd temperature."""
  from tunix_amd import _lib as L
  from tunix_amd import ops
  x = rnd((M, D), 60)
  w = rnd((D, V), 61, 0.05)
  g = torch.Generator().manual_seed(62)
  targets = torch.randint(0, V, (M,), generator=g, dtype=torch.int32)
  gx = bf(x).to(gpu)
  c, s = ops.quantize_pack(bf(w).to(gpu), group, qtype)
  codes, scale = Q.quantize(w.numpy(), group, qtype)
  kw, a, b = {}, None, None
  d = L.LmHeadDesc()
  if r:
    a, b = _lora(D, V, r, 63)
    a_t, b_t = _pad_lora(a, b, r)
    t = torch.zeros(M, r, dtype=torch.bfloat16, device=gpu)
    ops.lora_down(gx, bf(a_t).to(gpu), t)
    gb = bf(b_t).to(gpu)
    kw = dict(lora_rank=r, lora_nseg=1, lora_seg_end=[V], lora_seg_toff=[0], t=t, t_ld=r, lora_b=gb, lora_scale=1.0)
    d.lora_rank, d.t, d.t_ld, d.lora_b, d.lora_scale = r, t.data_ptr(), r, gb.data_ptr(), 1.0
  y = torch.empty(M, V, dtype=torch.bfloat16, device=gpu)
  ops.qlinear(ops.make_qlinear_desc(M=M, K=D, N=V, group=group, qtype=qtype, x=gx, codes=c, scales=s, y=y,
                                    epilogue=L.TNX_EPI_STORE, **kw))
  temperature = 0.7
  d.M, d.D, d.V, d.x = M, D, V, gx.data_ptr()
  d.codes, d.scales, d.group, d.qtype = c.data_ptr(), s.data_ptr(), group, qtype
  d.temperature = temperature
  nvb = ops.lmhead_nblocks(V)
  part = torch.full((M * nvb * 4,), float("nan"), dtype=torch.float32, device=gpu)
  pent = torch.full((M * nvb,), float("nan"), dtype=torch.float32, device=gpu)
  best = torch.empty(M, dtype=torch.int32, device=gpu)
  blp, tlp, lse, ent = (torch.empty(M, dtype=torch.float32, device=gpu) for _ in range(4))
  gt = targets.to(gpu)
  d.targets, d.part, d.best_id, d.best_logp = gt.data_ptr(), part.data_ptr(), best.data_ptr(), blp.data_ptr()
  d.target_logp, d.lse = tlp.data_ptr(), lse.data_ptr()
  if entropy:
    d.part_entropy, d.entropy = pent.data_ptr(), ent.data_ptr()
  ops.lmhead(d)
  torch.cuda.synchronize()
  assert not torch.isnan(part).any(), "every (row, block) statistic is written"
  got = (y.float() / np.float32(temperature)).cpu()
  assert torch.equal(best.cpu().long(), torch.argmax(got, dim=-1)), "arg-max (first maximal index)"
  ref_lse = torch.logsumexp(got, dim=-1)
  np.testing.assert_allclose(lse.cpu().numpy(), ref_lse.numpy(), rtol=0, atol=2e-5)
  np.testing.assert_allclose(tlp.cpu().numpy(), rl_ref.selective_log_softmax(got, targets).numpy(), rtol=0, atol=2e-5)
  np.testing.assert_allclose(blp.cpu().numpy(), (got.max(-1).values - ref_lse).numpy(), atol=2e-5)
  if entropy:
    np.testing.assert_allclose(ent.cpu().numpy(), rl_ref.compute_entropy_from_logits(got).numpy(), rtol=0, atol=5e-5)
  # the same head read from its converted copy (two work-groups per compute unit): same bits
  first = [v.clone() for v in (best, blp, tlp, lse, ent if entropy else lse)]
  for v in (blp, tlp, lse, ent, part, pent):
    v.fill_(float("nan"))
  w_exp = ops.qw_expand(c, s, D, V, group, qtype)
  d.w_expanded = w_exp.data_ptr()
  ops.lmhead(d)
  torch.cuda.synchronize()
  for u, v in zip(first, (best, blp, tlp, lse, ent if entropy else lse)):
    assert torch.equal(u, v), "expanded head: statistics differ"
  logits = Q.rb(Q.qlinear_lora(x, codes, scale, group, qtype, a, b, lora_scale=1.0) if r else
                Q.qlinear_lora(x, codes, scale, group, qtype, None, None, lora_scale=0.0))
  ref_t = rl_ref.selective_log_softmax(logits / np.float32(temperature), targets)
  assert (tlp.cpu() - ref_t).abs().max().item() < 2e-2


@pytest.mark.parametrize("M,D,V,dense,r", [(300, 512, 8208, False, 64), (128, 512, 4096, True, 0), (1030, 256, 8192, False, 32)])
def test_lmhead_fp32_accumulate_reference_mode(gpu, M, D, V, dense, r):
  """logits_fp32: the fp32 accumulators are the logits (no rounding to bf16).  Against an fp64
  evaluation of the same operands -- bf16 hidden states, weights dequantised to bf16, bf16
  adapter intermediate t -- the per-token log-probabilities, logsumexp and entropy agree to 1e-4
  (the tolerance the fp32-accumulate reference mode is held to), where the normal mode, whose
  logits are bf16 values, is only good to bf16 resolution; the arg-max is that of the fp64 logits
  except at margins below 1e-4.  The many-row shape, which the bf16 mode sends through the
  128 x 256 kernel, takes the 128 x 128 head kernel here (that one stages its tile in bf16)."""
  from tunix_amd import _lib as L
  from tunix_amd import ops
  x = rnd((M, D), 160)
  w = rnd((D, V), 161, 0.05)
  g = torch.Generator().manual_seed(162)
  targets = torch.randint(0, V, (M,), generator=g, dtype=torch.int32)
  gx = bf(x).to(gpu)
  d = L.LmHeadDesc()
  d.M, d.D, d.V, d.x = M, D, V, gx.data_ptr()
  if dense:
    gw = bf(w).t().contiguous().to(gpu)
    d.w_bf16 = gw.data_ptr()
    ref_lg = x.double() @ Q.rb(w).double()
  else:
    c, s = ops.quantize_pack(bf(w).to(gpu), 128, Q.INT4)
    d.codes, d.scales, d.group, d.qtype = c.data_ptr(), s.data_ptr(), 128, Q.INT4
    codes, scale = Q.quantize(w.numpy(), 128, Q.INT4)
    wd = torch.from_numpy(Q.dequantize(codes, scale, 128, Q.INT4)).double()
    ref_lg = x.double() @ wd
  if r:
    a, b = _lora(D, V, r, 163)
    a_t, b_t = _pad_lora(a, b, r)
    t = torch.zeros(M, r, dtype=torch.bfloat16, device=gpu)
    ops.lora_down(gx, bf(a_t).to(gpu), t)
    gb = bf(b_t).to(gpu)
    d.lora_rank, d.t, d.t_ld, d.lora_b, d.lora_scale = r, t.data_ptr(), r, gb.data_ptr(), 2.0
    ref_lg = ref_lg + 2.0 * (t.cpu().double() @ b.double())       # the kernel's own bf16 t
    assert_bf16_close(t, Q.rb((x.double() @ a.double()).float()), what="t")
  temperature = 0.9
  d.temperature = temperature
  nvb = ops.lmhead_nblocks(V)
  part = torch.empty(M * nvb * 4, dtype=torch.float32, device=gpu)
  pent = torch.empty(M * nvb, dtype=torch.float32, device=gpu)
  best = torch.empty(M, dtype=torch.int32, device=gpu)
  gt = targets.to(gpu)
  d.targets, d.part, d.best_id = gt.data_ptr(), part.data_ptr(), best.data_ptr()
  d.part_entropy = pent.data_ptr()
  ref = ref_lg / temperature
  ref_lp = torch.log_softmax(ref, -1)
  want_t = torch.gather(ref_lp, -1, targets.long()[:, None])[:, 0]
  want_ent = -(ref_lp.exp() * ref_lp).sum(-1)
  errs = {}
  for mode in (1, 0):
    tlp, lse, ent, blp = (torch.empty(M, dtype=torch.float32, device=gpu) for _ in range(4))
    d.target_logp, d.lse, d.entropy, d.best_logp = tlp.data_ptr(), lse.data_ptr(), ent.data_ptr(), blp.data_ptr()
    d.logits_fp32 = mode
    ops.lmhead(d)
    torch.cuda.synchronize()
    errs[mode] = (tlp.cpu().double() - want_t).abs().max().item()
    if mode == 1:
      assert errs[1] <= 1e-4, errs[1]
      assert (lse.cpu().double() - torch.logsumexp(ref, -1)).abs().max().item() <= 1e-4
      assert (ent.cpu().double() - want_ent).abs().max().item() <= 1e-4
      top = ref.max(-1)
      differs = best.cpu().long() != top.indices
      gap = top.values - torch.gather(ref, -1, best.cpu().long()[:, None])[:, 0]
      assert (gap[differs] <= 1e-4).all()
      assert (blp.cpu().double() - (top.values - torch.logsumexp(ref, -1))).abs().max().item() <= 1e-4
  assert errs[0] > 10 * errs[1]        # the bf16 logits of the normal mode are visibly coarser
  assert errs[0] <= 2e-2


def test_lmhead_forbidden_and_ties(gpu):
  """Equal maxima resolve to the lowest index; forbidden ids are never chosen."""
  from tunix_amd import _lib as L
  from tunix_amd import ops
  M, D, V = 4, 128, 512
  x = torch.zeros(M, D)
  x[:, 0] = 1.0
  w = torch.zeros(D, V)
  w[0, [5, 300, 511]] = 2.0      # three-way tie
  d = L.LmHeadDesc()
  d.M, d.D, d.V = M, D, V
  gx, gw = bf(x).to(gpu), bf(w).t().contiguous().to(gpu)
  d.x, d.w_bf16, d.temperature = gx.data_ptr(), gw.data_ptr(), 1.0
  part = torch.empty(M * ops.lmhead_nblocks(V) * 4, dtype=torch.float32, device=gpu)
  best = torch.empty(M, dtype=torch.int32, device=gpu)
  d.part, d.best_id = part.data_ptr(), best.data_ptr()
  ops.lmhead(d)
  assert best.cpu().tolist() == [5] * M
  fb = torch.tensor([5, 300], dtype=torch.int32, device=gpu)
  d.forbidden, d.n_forbidden = fb.data_ptr(), 2
  ops.lmhead(d)
  assert best.cpu().tolist() == [511] * M


@pytest.mark.parametrize("M,V,variant", [(128, 4096, 0), (40, 1040, 1), (7, 512, 0)])
def test_lmhead_categorical_draw_matches_oracle(gpu, M, V, variant):
  """The whole-vocabulary draw inside the head: ids equal jax.random.categorical (restated by the
  oracle) over the logits the kernel itself produced, divided by the temperature, with a
  forbidden id; the log-probabilities agree to 2e-5; tnx_sample_topk on the materialised logits
  draws the same ids."""
  from tunix_amd import _lib as L
  from tunix_amd import ops
  D, temp, step = 256, 0.9, 41
  x, w = rnd((M, D), 54), rnd((D, V), 55, 0.3)
  gx, gw = bf(x).to(gpu), bf(w).t().contiguous().to(gpu)
  key = TF.prng_key(777)
  nvb = ops.lmhead_nblocks(V)
  d = L.LmHeadDesc()
  d.M, d.D, d.V, d.x, d.w_bf16, d.temperature = M, D, V, gx.data_ptr(), gw.data_ptr(), temp
  part = torch.empty(M * nvb * 4, dtype=torch.float32, device=gpu)
  pdraw = torch.empty(M * nvb * 3, dtype=torch.float32, device=gpu)
  lg_out = torch.empty(M, V, dtype=torch.float32, device=gpu)
  ids = torch.empty(M, dtype=torch.int32, device=gpu)
  lp = torch.empty(M, dtype=torch.float32, device=gpu)
  stp = torch.tensor([step], dtype=torch.int32, device=gpu)
  fb = torch.tensor([3], dtype=torch.int32, device=gpu)
  d.part, d.logits_out, d.forbidden, d.n_forbidden = part.data_ptr(), lg_out.data_ptr(), fb.data_ptr(), 1
  d.part_draw, d.draw_key0, d.draw_key1, d.draw_rng_variant = pdraw.data_ptr(), int(key[0]), int(key[1]), variant
  d.draw_step_ptr, d.draw_id, d.draw_logp = stp.data_ptr(), ids.data_ptr(), lp.data_ptr()
  ops.lmhead(d)
  torch.cuda.synchronize()
  raw = lg_out.cpu()
  masked = raw.clone()
  masked[:, 3] = -np.inf
  tok_ref, lp_ref = SR.sample_top_p(masked, TF.fold_in(key, step), temp, 1.0, None, partitionable=bool(variant))
  assert ids.cpu().long().tolist() == tok_ref.tolist()
  np.testing.assert_allclose(lp.cpu().numpy(), lp_ref.numpy(), atol=2e-5)
  assert len(set(ids.cpu().tolist())) > 1 or M < 4
  ids2 = torch.empty_like(ids)
  lp2 = torch.empty_like(lp)
  ws = torch.empty(ops.sample_topk_ws_bytes(M, V, 0) // 4, dtype=torch.float32, device=gpu)
  ops.sample_topk(lg_out, 0, 1.0, temp, (int(key[0]), int(key[1])), variant, stp, ws, ids2, lp2, forbidden=fb)
  torch.cuda.synchronize()
  assert torch.equal(ids, ids2)
  np.testing.assert_allclose(lp.cpu().numpy(), lp2.cpu().numpy(), atol=2e-5)


@pytest.mark.parametrize("M,V,D,variant,temp", [
    (128, 4096, 256, 0, 0.9), (128, 8208, 256, 1, 1.0), (40, 1040, 256, 0, 0.7), (7, 4096, 256, 1, 1.3),   # (the head kernel either way)
    (1, 65536, 256, 0, 0.8), (17, 65552, 256, 1, 1.0), (33, 66000, 128, 0, 1.3), (64, 66000, 256, 1, 0.9),  # 64-row tiles, ragged last blocks
    (65, 65536, 256, 0, 1.0), (120, 65552, 256, 1, 0.7), (128, 65536, 128, 0, 0.9),                         # 128-row tiles
    (150, 65536, 2048, 1, 0.8),                                                                             # 256-row tiles
    (200, 65552, 128, 0, 1.0)])                                                                             # two blocks of rows
def test_lmhead_categorical_draw_on_the_many_row_kernel(gpu, M, V, D, variant, temp):
  """The same draw with the dense head's expanded copy, i.e. (from 256 column tiles on) in the statistics epilogue of the
  many-row kernel: ids equal the oracle's jax.random.categorical over the logits the kernel
  wrote; log-probabilities to 2e-5; the same of the head kernel that reads the plain weights, whose logits are within an ulp."""
  from tunix_amd import _lib as L
  from tunix_amd import ops
  step = 17
  x, w = rnd((M, D), 254), rnd((D, V), 255, 0.3 * (256 / D) ** 0.5)
  gx, gw = bf(x).to(gpu), bf(w).t().contiguous().to(gpu)
  w_exp = ops.dense_expand(gw)
  key = TF.prng_key(4242)
  nvb = ops.lmhead_nblocks(V)
  stp = torch.tensor([step], dtype=torch.int32, device=gpu)
  res = []
  for expanded in (True, False):
    d = L.LmHeadDesc()
    d.M, d.D, d.V, d.x, d.w_bf16, d.temperature = M, D, V, gx.data_ptr(), gw.data_ptr(), temp
    if expanded:
      d.w_expanded = w_exp.data_ptr()
    part = torch.full((M * nvb * 4,), float("nan"), dtype=torch.float32, device=gpu)
    pdraw = torch.full((M * nvb * 3,), float("nan"), dtype=torch.float32, device=gpu)
    lg_out = torch.empty(M, V, dtype=torch.float32, device=gpu)
    ids = torch.full((M,), -1, dtype=torch.int32, device=gpu)
    lp = torch.empty(M, dtype=torch.float32, device=gpu)
    d.part, d.logits_out = part.data_ptr(), lg_out.data_ptr()
    d.part_draw, d.draw_key0, d.draw_key1, d.draw_rng_variant = pdraw.data_ptr(), int(key[0]), int(key[1]), variant
    d.draw_step_ptr, d.draw_id, d.draw_logp = stp.data_ptr(), ids.data_ptr(), lp.data_ptr()
    ops.lmhead(d)
    torch.cuda.synchronize()
    assert not torch.isnan(pdraw).any()
    res.append((ids.cpu(), lp.cpu(), lg_out.cpu()))
  (_, _, lg_w), (_, _, lg_h) = res
  many_rows = (M + 127) // 128 * ((V + 255) // 256) >= 256
  assert torch.equal(lg_w, lg_h) or many_rows
  assert ((lg_w - lg_h).abs() <= 2.0 ** -7 * torch.maximum(lg_w.abs(), lg_h.abs()) + D * 2.0 ** -24 * 16).all()
  for ids, lp, lg in res if many_rows else res[:1]:
    tok_ref, lp_ref = SR.sample_top_p(lg, TF.fold_in(key, step), temp, 1.0, None, partitionable=bool(variant))
    assert ids.long().tolist() == tok_ref.tolist()
    np.testing.assert_allclose(lp.numpy(), lp_ref.numpy(), atol=2e-5)
  if not many_rows:
    assert torch.equal(res[0][0], res[1][0])
    np.testing.assert_allclose(res[0][1].numpy(), res[1][1].numpy(), atol=2e-5)
  assert len(set(res[0][0].tolist())) > 1 or M < 4


@pytest.mark.parametrize("V", [3000, 40001])
@pytest.mark.parametrize("segmented", [False, True])
@pytest.mark.parametrize("k,top_p,variant", [(50, 1.0, 0), (50, 0.7, 0), (8, 0.9, 1), (0, 1.0, 0)])
def test_sample_topk_matches_oracle(gpu, k, top_p, variant, segmented, V):
  """Both flavours of the kernel (one work-group per row; row segments + merge, chosen by passing
  a workspace) against the oracle's sample_top_p: ids exactly, log-probabilities to 2e-5.
  V = 40001 spans three segments, with ties that straddle them."""
  from tunix_amd import ops
  M = 16
  g = torch.Generator().manual_seed(60)
  logits = (torch.randn(M, V, generator=g) * 2).float()
  logits[:, 17] = logits[:, 29]                      # ties inside the top-k
  top = torch.topk(logits, 3, dim=1).values
  logits[:, V - 7] = top[:, 1]                       # ... and across segments, at the far end
  logits[:, V // 2] = top[:, 2]
  key = TF.prng_key(1234)
  step = 77
  temp = 0.7
  forbidden = [int(torch.argmax(logits[0])), 5]
  tok_ref, lp_ref = SR.sample_top_p(logits, TF.fold_in(key, step), temp, top_p, k if k else None,
                                    partitionable=bool(variant))
  ids = torch.empty(M, dtype=torch.int32, device=gpu)
  lp = torch.empty(M, dtype=torch.float32, device=gpu)
  stp = torch.tensor([step], dtype=torch.int32, device=gpu)
  ws = None
  if segmented:
    nb = ops.sample_topk_ws_bytes(M, V, k)
    assert nb > 0
    ws = torch.empty(max(nb // 4, 1), dtype=torch.float32, device=gpu)
  ops.sample_topk(logits.to(gpu), k, top_p, temp, (int(key[0]), int(key[1])), variant, stp, ws, ids, lp)
  torch.cuda.synchronize()
  assert ids.cpu().long().tolist() == tok_ref.tolist()
  np.testing.assert_allclose(lp.cpu().numpy(), lp_ref.numpy(), atol=2e-5)
  # forbidden ids behave like -inf logits (tunix/generate/sampler.py:490-491)
  masked = logits.clone()
  masked[:, forbidden] = -np.inf
  tok_ref2, lp_ref2 = SR.sample_top_p(masked, TF.fold_in(key, step), temp, top_p, k if k else None,
                                      partitionable=bool(variant))
  fb = torch.tensor(forbidden, dtype=torch.int32, device=gpu)
  ops.sample_topk(logits.to(gpu), k, top_p, temp, (int(key[0]), int(key[1])), variant, stp, ws, ids, lp,
                  forbidden=fb)
  assert ids.cpu().long().tolist() == tok_ref2.tolist()
  np.testing.assert_allclose(lp.cpu().numpy(), lp_ref2.numpy(), atol=2e-5)


def _block_stats(logits, temp, forbidden=None):
  """What a head call at temperature `temp` leaves for tnx_sample_topk_head: per 128-column block
  the largest scaled (and masked) logit in slot 0 of its four statistics, and the row's lse."""
  M, V = logits.shape
  q = logits / np.float32(temp)
  if forbidden:
    q[:, forbidden] = -np.inf
  nvb = (V + 127) // 128
  pad = torch.full((M, nvb * 128), -np.inf)
  pad[:, :V] = q
  part = torch.zeros(M, nvb, 4)
  part[:, :, 0] = pad.view(M, nvb, 128).max(-1).values
  return part, torch.logsumexp(q.double(), -1).float()


@pytest.mark.parametrize("V", [3000, 40001, 262144])
@pytest.mark.parametrize("k,top_p,variant", [(50, 1.0, 0), (64, 0.7, 0), (8, 0.9, 1), (1, 1.0, 0)])
def test_sample_topk_head_matches_oracle(gpu, k, top_p, variant, V):
  """The one-launch top-k draw that starts from the head's block maxima, against the oracle's
  sample_top_p and against tnx_sample_topk on the same logits: ids exactly, log-probabilities to
  2e-5; ties inside the top-k, across blocks and at the far end of the row; forbidden ids."""
  from tunix_amd import ops
  M = 16
  assert ops.sample_topk_head_ok(V, k)
  g = torch.Generator().manual_seed(60)
  logits = (torch.randn(M, V, generator=g) * 2).float()
  logits[:, 17] = logits[:, 29]
  top = torch.topk(logits, 3, dim=1).values
  logits[:, V - 7] = top[:, 1]
  logits[:, V // 2] = top[:, 2]
  key = TF.prng_key(1234)
  step, temp = 77, 0.7
  stp = torch.tensor([step], dtype=torch.int32, device=gpu)
  gl = logits.to(gpu)
  for forbidden in (None, [int(torch.argmax(logits[0])), 5]):
    masked = logits.clone()
    if forbidden:
      masked[:, forbidden] = -np.inf
    tok_ref, lp_ref = SR.sample_top_p(masked, TF.fold_in(key, step), temp, top_p, k, partitionable=bool(variant))
    part, lse = _block_stats(logits.clone(), temp, forbidden)
    fb = torch.tensor(forbidden, dtype=torch.int32, device=gpu) if forbidden else None
    ids = torch.full((M,), -1, dtype=torch.int32, device=gpu)
    lp = torch.empty(M, dtype=torch.float32, device=gpu)
    ops.sample_topk_head(gl, part.to(gpu), lse.to(gpu), k, top_p, temp, (int(key[0]), int(key[1])), variant, stp,
                         ids, lp, forbidden=fb)
    ids2, lp2 = torch.empty_like(ids), torch.empty_like(lp)
    ws = torch.empty(max(ops.sample_topk_ws_bytes(M, V, k) // 4, 1), dtype=torch.float32, device=gpu)
    ops.sample_topk(gl, k, top_p, temp, (int(key[0]), int(key[1])), variant, stp, ws, ids2, lp2, forbidden=fb)
    torch.cuda.synchronize()
    assert ids.cpu().long().tolist() == tok_ref.tolist()
    assert torch.equal(ids, ids2)
    np.testing.assert_allclose(lp.cpu().numpy(), lp_ref.numpy(), atol=2e-5)
    np.testing.assert_allclose(lp.cpu().numpy(), lp2.cpu().numpy(), atol=2e-5)


@pytest.mark.parametrize("V,k", [(50000, 50), (300000, 64), (300000, 3), (130, 64)])
def test_sample_topk_head_with_massive_ties(gpu, V, k):
  """Only a handful of distinct values: every block has the same maximum (more than 2048 equal
  block maxima at V = 300000: the exact radix select of the block stage) and thousands of
  elements tie at the k-th value (the same path of the element stage); the k lowest indices among
  them are taken.  V = 130: two blocks, the second with two columns."""
  from tunix_amd import ops
  M, top_p, temp, step = 6, 0.95, 1.0, 3
  g = torch.Generator().manual_seed(61)
  logits = torch.round(torch.randn(M, V, generator=g)).float()
  logits[0] = 1.0
  logits[1, : V // 2] = 5.0
  key = TF.prng_key(99)
  tok_ref, lp_ref = SR.sample_top_p(logits, TF.fold_in(key, step), temp, top_p, k)
  part, lse = _block_stats(logits.clone(), temp)
  ids = torch.full((M,), -1, dtype=torch.int32, device=gpu)
  lp = torch.empty(M, dtype=torch.float32, device=gpu)
  stp = torch.tensor([step], dtype=torch.int32, device=gpu)
  ops.sample_topk_head(logits.to(gpu), part.to(gpu), lse.to(gpu), k, top_p, temp, (int(key[0]), int(key[1])), 0, stp,
                       ids, lp)
  torch.cuda.synchronize()
  assert ids.cpu().long().tolist() == tok_ref.tolist()
  # (log-softmax in fp64: an fp32 sum over 300000 exponentials of this size is itself 2e-4 off)
  lp64 = torch.log_softmax(logits.double() / temp, -1).gather(1, tok_ref[:, None])[:, 0]
  np.testing.assert_allclose(lp.cpu().numpy(), lp64.float().numpy(), atol=2e-5)


def test_sample_topk_head_after_a_head_call(gpu):
  """The pairing the sampler uses: a dense head at the sampling temperature writes logits, block
  statistics and lse; the draw from them equals tnx_sample_topk's on the logits and the oracle's."""
  from tunix_amd import _lib as L
  from tunix_amd import ops
  M, D, V, k, top_p, temp, step = 70, 256, 8208, 50, 0.9, 0.8, 5
  x, w = rnd((M, D), 154), rnd((D, V), 155, 0.3)
  gx, gw = bf(x).to(gpu), bf(w).t().contiguous().to(gpu)
  key = TF.prng_key(31)
  nvb = ops.lmhead_nblocks(V)
  stp = torch.tensor([step], dtype=torch.int32, device=gpu)
  for expanded in (False, True):
    d = L.LmHeadDesc()
    d.M, d.D, d.V, d.x, d.w_bf16, d.temperature = M, D, V, gx.data_ptr(), gw.data_ptr(), temp
    w_exp = ops.dense_expand(gw) if expanded else None
    if expanded:
      d.w_expanded = w_exp.data_ptr()
    part = torch.empty(M * nvb * 4, dtype=torch.float32, device=gpu)
    lg_out = torch.empty(M, V, dtype=torch.float32, device=gpu)
    lse = torch.empty(M, dtype=torch.float32, device=gpu)
    d.part, d.logits_out, d.lse = part.data_ptr(), lg_out.data_ptr(), lse.data_ptr()
    ops.lmhead(d)
    ids = torch.full((M,), -1, dtype=torch.int32, device=gpu)
    lp = torch.empty(M, dtype=torch.float32, device=gpu)
    ops.sample_topk_head(lg_out, part, lse, k, top_p, temp, (int(key[0]), int(key[1])), 0, stp, ids, lp)
    ids2, lp2 = torch.empty_like(ids), torch.empty_like(lp)
    ws = torch.empty(ops.sample_topk_ws_bytes(M, V, k) // 4, dtype=torch.float32, device=gpu)
    ops.sample_topk(lg_out, k, top_p, temp, (int(key[0]), int(key[1])), 0, stp, ws, ids2, lp2)
    torch.cuda.synchronize()
    tok_ref, lp_ref = SR.sample_top_p(lg_out.cpu(), TF.fold_in(key, step), temp, top_p, k)
    assert ids.cpu().long().tolist() == tok_ref.tolist()
    assert torch.equal(ids, ids2)
    np.testing.assert_allclose(lp.cpu().numpy(), lp_ref.numpy(), atol=2e-5)
    # the block maxima are bit for bit the maxima of the scaled logits the draw recomputes
    q = (lg_out / np.float32(temp)).cpu()
    pad = torch.full((M, nvb * 128), -np.inf)
    pad[:, :V] = q
    assert torch.equal(part.view(M, nvb, 4)[:, :, 0].cpu(), pad.view(M, nvb, 128).max(-1).values)


@pytest.mark.parametrize("segmented", [False, True])
def test_sample_topk_with_massive_ties(gpu, segmented):
  """Logits with only a handful of distinct values: thousands of elements tie at the k-th value,
  the k lowest indices among them must be taken (jax.lax.top_k order); in the segmented kernel
  this is the exact radix-select path behind the pivot shortcut."""
  from tunix_amd import ops
  M, V, k, top_p, temp, step = 8, 50000, 50, 0.95, 1.0, 3
  g = torch.Generator().manual_seed(61)
  logits = torch.round(torch.randn(M, V, generator=g)).float()     # values in {-4 .. 4}
  logits[0] = 1.0                                                   # a constant row
  key = TF.prng_key(99)
  tok_ref, lp_ref = SR.sample_top_p(logits, TF.fold_in(key, step), temp, top_p, k)
  ids = torch.empty(M, dtype=torch.int32, device=gpu)
  lp = torch.empty(M, dtype=torch.float32, device=gpu)
  stp = torch.tensor([step], dtype=torch.int32, device=gpu)
  ws = torch.empty(ops.sample_topk_ws_bytes(M, V, k) // 4, dtype=torch.float32, device=gpu) if segmented else None
  ops.sample_topk(logits.to(gpu), k, top_p, temp, (int(key[0]), int(key[1])), 0, stp, ws, ids, lp)
  torch.cuda.synchronize()
  assert ids.cpu().long().tolist() == tok_ref.tolist()
  np.testing.assert_allclose(lp.cpu().numpy(), lp_ref.numpy(), atol=2e-5)


@pytest.mark.parametrize("V,top_p,variant", [(3000, 0.7, 0), (40001, 0.9, 0), (40001, 0.3, 1)])
def test_sample_top_p_over_the_whole_vocabulary(gpu, V, top_p, variant):
  """top_p < 1 with top_k absent: the reference sorts the whole row (sampler.py:126-127); ids
  against the oracle exactly, log-probabilities to 2e-5; without a workspace the call is refused."""
  from tunix_amd import ops
  from tunix_amd._lib import TnxError
  M, temp, step = 16, 0.8, 11
  g = torch.Generator().manual_seed(62)
  logits = (torch.randn(M, V, generator=g) * 3).float()
  logits[:, 17] = logits[:, 29]
  key = TF.prng_key(4321)
  tok_ref, lp_ref = SR.sample_top_p(logits, TF.fold_in(key, step), temp, top_p, None, partitionable=bool(variant))
  ids = torch.empty(M, dtype=torch.int32, device=gpu)
  lp = torch.empty(M, dtype=torch.float32, device=gpu)
  stp = torch.tensor([step], dtype=torch.int32, device=gpu)
  nb = ops.sample_fullsort_ws_bytes(M, V)
  assert nb >= 4 * M * V * 4
  ws = torch.empty(nb // 4, dtype=torch.float32, device=gpu)
  ops.sample_topk(logits.to(gpu), 0, top_p, temp, (int(key[0]), int(key[1])), variant, stp, ws, ids, lp)
  torch.cuda.synchronize()
  assert ids.cpu().long().tolist() == tok_ref.tolist()
  np.testing.assert_allclose(lp.cpu().numpy(), lp_ref.numpy(), atol=2e-5)
  with pytest.raises((TnxError, ValueError), match="workspace"):
    ops.sample_topk(logits.to(gpu), 0, top_p, temp, (int(key[0]), int(key[1])), variant, stp, None, ids, lp)


@pytest.mark.parametrize("M,V", [(3, 100), (5, 4097), (4, 262144), (130, 2000)])
def test_full_row_sort_is_stable_and_descending(gpu, M, V):
  """The library's own radix sort behind the whole-row path (jax.lax.top_k(k = V): descending,
  the lower index first among equal values): the sorted keys and ids it leaves in the workspace
  against numpy's stable sort, bit for bit -- rows full of ties, negative values, zeros of both
  signs, forbidden ids (-inf, sorted last), fewer elements than the sort has threads."""
  from tunix_amd import ops
  rng = np.random.default_rng(7 + V)
  lg = rng.standard_normal((M, V)).astype(np.float32) * 4
  lg[0] = np.round(lg[0])                               # a row of heavy ties
  lg[1, ::3] = 0.0
  lg[1, 1::7] = -0.0
  lg[2, : V // 2] = lg[2, V // 2: 2 * (V // 2)]         # every value twice
  temp = 0.7
  forbidden = torch.tensor([1, V - 1, 17 % V], dtype=torch.int32, device=gpu)
  ids = torch.empty(M, dtype=torch.int32, device=gpu)
  lp = torch.empty(M, dtype=torch.float32, device=gpu)
  stp = torch.tensor([3], dtype=torch.int32, device=gpu)
  nb = ops.sample_fullsort_ws_bytes(M, V)
  ws = torch.zeros(nb // 4, dtype=torch.float32, device=gpu)
  ops.sample_topk(torch.from_numpy(lg).to(gpu), 0, 0.9, temp, (1, 2), 0, stp, ws, ids, lp, forbidden=forbidden)
  torch.cuda.synchronize()
  up = (M * V * 4 + 255) // 256 * 256 // 4
  keys = ws[: M * V].view(M, V).cpu().numpy()
  sids = ws[2 * up: 2 * up + M * V].view(torch.int32).view(M, V).cpu().numpy()
  y = (torch.from_numpy(lg) / np.float32(temp)).numpy()
  y[:, [1, V - 1, 17 % V]] = -np.inf
  # descending with the lower index first among equals; -0.0 sorts below +0.0 (bit patterns)
  for m in range(M):
    order = np.lexsort((np.arange(V), np.signbit(y[m]) & (y[m] == 0), -y[m].astype(np.float64)))
    assert np.array_equal(sids[m], order.astype(np.int32)), m
    assert np.array_equal(keys[m].view(np.uint32), y[m][order].view(np.uint32)), m
  assert 0 <= int(ids.min()) and int(ids.max()) < V


def test_sample_commit_and_fill(gpu):
  from tunix_amd import ops
  B, Ld = 5, 12
  tokens = torch.full((B, Ld), 9, dtype=torch.int32, device=gpu)
  lps = torch.zeros(B, Ld, dtype=torch.float32, device=gpu)
  done = torch.zeros(B, dtype=torch.int32, device=gpu)
  step = torch.tensor([6], dtype=torch.int32, device=gpu)
  ids = torch.tensor([3, 4, 2, 7, 2], dtype=torch.int32, device=gpu)
  lp = torch.arange(B, dtype=torch.float32, device=gpu) * -0.5
  eos = torch.tensor([2, 11], dtype=torch.int32, device=gpu)
  ops.sample_commit(ids, lp, tokens, lps, done, eos, step)
  assert step.item() == 7
  assert tokens[:, 7].cpu().tolist() == [3, 4, 2, 7, 2] and tokens[:, 6].cpu().tolist() == [9] * B
  assert lps[:, 7].cpu().tolist() == [0.0, -0.5, -1.0, -1.5, -2.0]
  assert done.cpu().tolist() == [0, 0, 1, 0, 1]
  buf = torch.ones(1000, dtype=torch.int32, device=gpu)
  ops.fill_u32(buf, 0)
  assert buf.sum().item() == 0


@pytest.mark.parametrize("M", [1, 2, 3, 4, 5])
def test_head_of_the_fewest_rows(gpu, M):
  """A row's statistics, log-probabilities and raw logits do not depend on how many rows of its tile there are."""
  from tunix_amd import _lib as L
  from tunix_amd import ops
  D, V = 256, 1040
  x, w = bf(rnd((16, D), 701)).to(gpu), bf(rnd((V, D), 702)).to(gpu)
  targets = torch.arange(5, 5 + 16, dtype=torch.int32, device=gpu) * 40
  outs = []
  for rows in (16, M):
    ids, best, tgt, lse = (torch.full((16,), -7, dtype=t, device=gpu) for t in (torch.int32, torch.float32, torch.float32, torch.float32))
    ent, part, part_ent = torch.zeros(16, device=gpu), torch.empty(16 * 9 * 4, device=gpu), torch.empty(16 * 9, device=gpu)
    logits = torch.zeros(16, V, device=gpu)
    d = L.LmHeadDesc()
    d.M, d.D, d.V, d.x, d.w_bf16, d.part, d.temperature, d.targets = rows, D, V, x.data_ptr(), w.data_ptr(), part.data_ptr(), 0.9, targets.data_ptr()
    d.best_id, d.best_logp, d.target_logp, d.lse = ids.data_ptr(), best.data_ptr(), tgt.data_ptr(), lse.data_ptr()
    d.entropy, d.part_entropy, d.logits_out = ent.data_ptr(), part_ent.data_ptr(), logits.data_ptr()
    ops.lmhead(d)
    outs.append([t.cpu() for t in (ids, best, tgt, lse, ent, logits)])
  for a, b in zip(*outs):
    assert torch.equal(a[:M], b[:M]) and (b[M:] == b[M:].flatten()[0]).all()


@pytest.mark.parametrize("B,T,D,R,scale,dh,flavor", [
    (1, 1, 256, 32, 1.0, 0, 1), (1, 1, 4096, 192, 1.0, 128, 0), (16, 1, 4096, 192, 1.0, 128, 0),   # one launch, the table's rows behind the last
    (17, 1, 4096, 192, 1.0, 128, 0), (130, 1, 4096, 0, 1.0, 128, 0), (300, 1, 2048, 64, 1.0, 64, 1),   # the norm's launch has the table
    (64, 1, 1152, 64, 34.0, 0, 2), (3, 37, 1152, 64, 34.0, 0, 2), (2, 5, 96, 16, 1.0, 2, 1), (1, 3, 16384, 0, 1.0, 0, 0)])
def test_embedding_in_the_first_norm(gpu, B, T, D, R, scale, dh, flavor):
  """tnx_embed_norm against tnx_embed, tnx_norm_lora (or tnx_rmsnorm) and tnx_rope_table, bit for bit; ids outside the vocabulary included."""
  from tunix_amd import ops
  V, L, col, M = 77, T + 3, 2, B * T
  table, w = bf(rnd((V, D), 601)).to(gpu), bf(rnd((D,), 602)).to(gpu)
  a_t = bf(rnd((R, D), 603)).to(gpu) if R else None
  ids = torch.randint(-2, V + 2, (B, L), generator=torch.Generator().manual_seed(604), dtype=torch.int32).to(gpu)
  positions = torch.randint(0, 5000, (B, L), generator=torch.Generator().manual_seed(605), dtype=torch.int32).to(gpu)
  timescale = (10000.0 ** (torch.arange(max(dh // 2, 1)) / max(dh // 2, 1))).to(gpu)
  colp = torch.tensor([col], dtype=torch.int32, device=gpu)
  outs = []
  for fused in (False, True):
    h, y = (torch.full((M, D), 7.0, dtype=torch.bfloat16, device=gpu) for _ in range(2))
    t = torch.full((M, R + 16), 7.0, dtype=torch.bfloat16, device=gpu)
    sn, cs = (torch.full((B, max(dh // 2, 1)), 7.0, device=gpu) for _ in range(2))
    if fused:
      ops.embed_norm(table, ids, colp, B, T, scale, h, w, y, 1e-6, flavor, a_t, t, (positions, timescale, dh, sn, cs) if dh else None)
    else:
      ops.embed(table, ids, colp, B, T, scale, h)
      if R:
        ops.norm_lora(a_t, t, w, y, 1e-6, flavor, M, D, x=h)
      else:
        ops.rmsnorm(h, w, y, 1e-6, flavor)
      if dh:
        ops.rope_table(positions, colp, B, timescale, dh, sn, cs)
    outs.append([v.cpu() for v in (h, y, t, sn, cs)])
  for a, b in zip(*outs):
    assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))
  assert (outs[1][1] != 7.0).any() and (not dh or (outs[1][3] != 7.0).all())


@pytest.mark.parametrize("M,V,draw,lists", [(1, 640, False, True), (1, 640, True, False), (5, 9008, False, False), (17, 8256, True, True),
                                            (64, 640, False, True), (130, 9008, True, True), (1000, 640, False, True)])
def test_head_enters_its_own_choice(gpu, M, V, draw, lists):
  """tnx_lmhead_commit against tnx_lmhead_logp and tnx_sample_commit behind it, over several steps from one state each (the tickets are as they
  were after every call); all whole numbers and the same bits."""
  from tunix_amd import _lib as L
  from tunix_amd import ops
  D, steps, dev = 128, 3, gpu
  w = bf(rnd((V, D), 501)).to(dev)
  eos = torch.arange(0, V, 3, dtype=torch.int32, device=dev)
  states = []
  for fused in (False, True):
    tokens = torch.zeros(M, 4 + steps, dtype=torch.int32, device=dev)
    lps = torch.zeros(M, 4 + steps, dtype=torch.float32, device=dev) if lists else None
    done = torch.zeros(M, dtype=torch.int32, device=dev) if lists else None
    step, tickets = torch.tensor([2], dtype=torch.int32, device=dev), torch.zeros(1, dtype=torch.int32, device=dev)
    ids, lp = torch.empty(M, dtype=torch.int32, device=dev), torch.empty(M, dtype=torch.float32, device=dev)
    nvb = ops.lmhead_nblocks(V)
    part, part_draw = torch.empty(M * nvb * 4, device=dev), torch.empty(M * nvb * 3, device=dev)
    for i in range(steps):
      x = bf(rnd((M, D), 510 + i)).to(dev)
      d = L.LmHeadDesc()
      d.M, d.D, d.V, d.x, d.w_bf16, d.part, d.temperature = M, D, V, x.data_ptr(), w.data_ptr(), part.data_ptr(), 0.8 if draw else 1.0
      if draw:
        d.part_draw, d.draw_key0, d.draw_key1, d.draw_step_ptr = part_draw.data_ptr(), 5, 6, step.data_ptr()
        d.draw_id, d.draw_logp = ids.data_ptr(), lp.data_ptr()
      else:
        d.best_id, d.best_logp = ids.data_ptr(), lp.data_ptr()
      if fused:
        ops.lmhead_commit(d, ops.make_commit_desc(tokens, lps, done, eos if lists else None, step, tickets))
      else:
        ops.lmhead(d)
        ops.sample_commit(ids, lp if lists else None, tokens, lps, done, eos if lists else None, step)
    assert step.item() == 2 + steps and tickets.item() == 0
    states.append([t.cpu() for t in (tokens, lps, done, ids, lp) if t is not None])
  for a, b in zip(*states):
    assert torch.equal(a, b)
  if lists and M > 16:
    assert 0 < states[1][2].sum() < M
  c = ops.make_commit_desc(tokens, lps, done, None, step, tickets)
  d.draw_id, d.best_id = None, None
  with pytest.raises(ValueError, match="chooses nothing"):
    ops.lmhead_commit(d, c)


def test_grpo_ratio_matches_oracle(gpu):
  from tunix_amd import ops
  N, T = 4096, 64
  g = torch.Generator().manual_seed(70)
  logp = -torch.rand(N, generator=g) * 5
  old = logp + torch.randn(N, generator=g) * 0.05
  old[:8] = logp[:8] - 30.0          # exercises the +-20 clamp
  adv = torch.randn(N // T, generator=g)
  r_ref, l_ref, c_ref = rl_ref.grpo_ratio(logp.view(-1, T).numpy(), old.view(-1, T).numpy(),
                                          adv.numpy(), 0.2, 0.2)
  ratio = torch.empty(N, dtype=torch.float32, device=gpu)
  loss = torch.empty(N, dtype=torch.float32, device=gpu)
  clipped = torch.empty(N, dtype=torch.int32, device=gpu)
  ops.grpo_ratio(logp.to(gpu), old.to(gpu), adv.to(gpu), T, 0.2, 0.2, ratio, loss, clipped)
  np.testing.assert_allclose(ratio.cpu().numpy(), r_ref.reshape(-1), rtol=2e-6)
  np.testing.assert_allclose(loss.cpu().numpy(), l_ref.reshape(-1), rtol=2e-6, atol=1e-7)
  assert (clipped.cpu().numpy().astype(bool) == c_ref.reshape(-1)).mean() > 0.999
  # old = None: ratio is exactly one (tests/rl/algo_core_test.py:51-143 relies on it)
  ops.grpo_ratio(logp.to(gpu), None, adv.to(gpu), T, 0.2, 0.2, ratio, loss, None)
  assert torch.all(ratio == 1.0)


@pytest.mark.parametrize("n_tok,k,E", [(64, 8, 128), (1, 1, 1), (700, 8, 128), (3000, 2, 7), (33, 4, 640)])
def test_moe_sort_routes_is_a_stable_counting_sort(gpu, n_tok, k, E):
  """Routes sorted by expert, ties in route order, counts and offsets: against numpy's stable
  argsort -- one batch of 1024 routes and several, few and many experts (more than 512 experts
  take the general kernel), experts that receive nothing."""
  from tunix_amd import ops
  rng = np.random.Generator(np.random.PCG64(1000 + n_tok))
  ids = rng.integers(0, max(1, E - 1 if E > 2 else E), size=(n_tok, k)).astype(np.int32)   # the last expert stays empty
  ti = torch.from_numpy(ids).to(gpu)
  counts = torch.full((E,), -1, dtype=torch.int32, device=gpu)
  offs = torch.full((E + 1,), -1, dtype=torch.int32, device=gpu)
  sr = torch.full((n_tok * k,), -1, dtype=torch.int32, device=gpu)
  for _ in range(2):   # the second call sees the first call's leftovers in nothing it reads
    ops.moe_sort_routes(ti, E, counts, offs, sr)
  flat = ids.reshape(-1)
  np.testing.assert_array_equal(sr.cpu().numpy(), np.argsort(flat, kind="stable"))
  cnt = np.bincount(flat, minlength=E)
  np.testing.assert_array_equal(counts.cpu().numpy(), cnt)
  np.testing.assert_array_equal(offs.cpu().numpy(), np.concatenate([[0], np.cumsum(cnt)]))


@pytest.mark.parametrize("M,E,k,D,F", [(12, 16, 4, 256, 128), (64, 128, 8, 2048, 768)])
def test_moe_route_sort_gmm_combine(gpu, M, E, k, D, F):
  """Router top-k, route sort, grouped gate|up GEMM with SiLU-mul, grouped down GEMM and the
  weighted combine against the oracle's per-token form; the second case is the
  Qwen3-30B-A3B layer at its real width (128 experts, top-8, D 2048, expert MLP 768, batch 64:
  512 routes, about 4 rows per expert)."""
  from tunix_amd import _lib as L
  from tunix_amd import ops
  g = 128
  scores = rnd((M, E), 80)
  scores[3, 5] = scores[3, 9]                          # tie between experts
  probs = torch.softmax(scores, -1)
  order = torch.sort(probs, dim=-1, descending=True, stable=True).indices[:, :k]
  wts = torch.gather(probs, -1, order)
  wts = Q.rb(wts / wts.sum(-1, keepdim=True))
  tw = torch.empty(M, k, dtype=torch.bfloat16, device=gpu)
  ti = torch.empty(M, k, dtype=torch.int32, device=gpu)
  ops.moe_route_topk(bf(scores).to(gpu), k, tw, ti)
  assert torch.equal(ti.cpu().long(), order)
  assert_bf16_close(tw, wts, what="routing weights")
  counts = torch.empty(E, dtype=torch.int32, device=gpu)
  offs = torch.empty(E + 1, dtype=torch.int32, device=gpu)
  sr = torch.empty(M * k, dtype=torch.int32, device=gpu)
  ops.moe_sort_routes(ti, E, counts, offs, sr)
  flat = order.reshape(-1).numpy()
  ref_sorted = np.argsort(flat, kind="stable")
  np.testing.assert_array_equal(sr.cpu().numpy(), ref_sorted)
  np.testing.assert_array_equal(counts.cpu().numpy(), np.bincount(flat, minlength=E))
  # grouped gate|up with SiLU-mul, then down, then the weighted combine
  x = rnd((M, D), 81)
  wg, wu, wd = rnd((E, D, F), 82, 0.05), rnd((E, D, F), 83, 0.05), rnd((E, F, D), 84, 0.05)
  cb, sb = ops.qw_sizes(D, 2 * F, g)
  gc = torch.empty(E * cb // 4, dtype=torch.int32, device=gpu)
  gs = torch.empty(E * sb // 2, dtype=torch.bfloat16, device=gpu)
  cb2, sb2 = ops.qw_sizes(F, D, g)
  dc = torch.empty(E * cb2 // 4, dtype=torch.int32, device=gpu)
  ds = torch.empty(E * sb2 // 2, dtype=torch.bfloat16, device=gpu)
  used = set(order.reshape(-1).tolist())
  ref = torch.zeros(M, D, dtype=torch.float64)
  ref_mag = torch.zeros(M, D, dtype=torch.float64)    # sum of |w_j y_j|: the operands' magnitude
  for e in range(E):
    c, s = ops.quantize_pack(bf(torch.cat([wg[e], wu[e]], 1)).to(gpu), g, Q.INT4, True)
    gc[e * cb // 4:(e + 1) * cb // 4] = c
    gs[e * sb // 2:(e + 1) * sb // 2] = s
    c, s = ops.quantize_pack(bf(wd[e]).to(gpu), g, Q.INT4)
    dc[e * cb2 // 4:(e + 1) * cb2 // 4] = c
    ds[e * sb2 // 2:(e + 1) * sb2 // 2] = s
    if e not in used:
      continue
    dg, du, dd = (torch.from_numpy(Q.dequantize(*Q.quantize(m.numpy(), g, Q.INT4), g, Q.INT4)).double()
                  for m in (wg[e], wu[e], wd[e]))
    # all tokens routed to this expert at once (per token: the same arithmetic)
    rows, slots = torch.nonzero(order == e, as_tuple=True)
    gg = Q.rb((x[rows].double() @ dg).float())
    uu = Q.rb((x[rows].double() @ du).float())
    a = Q.rb(Q.rb(gg * Q.rb(torch.sigmoid(gg))) * uu)
    y = Q.rb((a.double() @ dd).float())
    ref.index_add_(0, rows, (wts[rows, slots][:, None] * y).double())
    ref_mag.index_add_(0, rows, (wts[rows, slots][:, None] * y).double().abs())
  # the combine adds the k expert outputs of a token in slot order j = 0..k-1; index_add_ above
  # adds them in expert order: both are sums of k bf16-exact products in double, equal to fp32
  # rounding, and the final rounding to bf16 absorbs the rest
  ref = Q.rb(ref.float())
  gx = bf(x).to(gpu)
  act = torch.empty(M * k, F, dtype=torch.bfloat16, device=gpu)
  yr = torch.empty(M * k, D, dtype=torch.bfloat16, device=gpu)
  d = L.MoeGmmDesc()
  d.n_routes, d.E, d.k, d.K, d.N, d.group, d.qtype = M * k, E, k, D, 2 * F, g, Q.INT4
  d.x, d.x_div, d.codes, d.scales = gx.data_ptr(), k, gc.data_ptr(), gs.data_ptr()
  d.offsets, d.sorted_route, d.epilogue, d.y = offs.data_ptr(), sr.data_ptr(), L.TNX_EPI_SILU_MUL, act.data_ptr()
  ops.moe_gmm(d)
  d2 = L.MoeGmmDesc()
  d2.n_routes, d2.E, d2.k, d2.K, d2.N, d2.group, d2.qtype = M * k, E, k, F, D, g, Q.INT4
  d2.x, d2.x_div, d2.codes, d2.scales = act.data_ptr(), 1, dc.data_ptr(), ds.data_ptr()
  d2.offsets, d2.sorted_route, d2.epilogue, d2.y = offs.data_ptr(), sr.data_ptr(), L.TNX_EPI_STORE, yr.data_ptr()
  ops.moe_gmm(d2)
  out = torch.empty(M, D, dtype=torch.bfloat16, device=gpu)
  ops.moe_combine(yr, tw, M, k, D, None, out)
  torch.cuda.synchronize()
  # the output is the rounded sum of k weighted expert rows, each a bf16 value that may sit one
  # ulp from the oracle's (it is computed from three rounded intermediates: gate, up,
  # activation); where the k terms cancel, the ulp that matters is that of the terms
  assert_bf16_close(out, ref, atol=1e-5, min_equal=0.85, what="moe", mag=ref_mag.float())


@pytest.mark.parametrize("E,n_tok,k,K,N,group,qtype,mul", [
    (16, 48, 2, 512, 256, 128, Q.INT4, True),     # experts of 40 and 17 rows: several 16-row blocks
    (16, 48, 2, 512, 256, 64, Q.NF4, False),
    (16, 48, 2, 256, 96, 32, Q.INT4, False),      # four scale slots per k-tile
    (256, 256, 4, 256, 288, 128, Q.INT4, False),  # 9 tile pairs per block, 2 per wave: runs span two blocks
    (256, 256, 4, 256, 576, 128, Q.NF4, True),
    (16, 48, 2, 384, 80, 128, Q.INT4, False),     # 5 column tiles: no pairs, the general kernel
    (8, 512, 2, 512, 256, 128, Q.INT4, False),    # ~128 rows per expert: the 128 x 256 tiles of the many-row kernel
    (8, 512, 2, 384, 512, 64, Q.NF4, True),
    (8, 512, 2, 256, 768, 32, Q.INT4, False),
    (8, 64, 2, 384, 96, 64, Q.NF4, False),        # 16 rows per expert on average: the 32-row tile kernel, whose
    (8, 128, 2, 256, 96, 128, Q.INT4, False),     # activation rows are gathered straight into LDS; 32: its 64-row form
])
def test_moe_gmm_skewed_routes(gpu, E, n_tok, k, K, N, group, qtype, mul, off=0):
  """The grouped GEMM alone, on routes built by hand: experts with no rows, with one row, with
  exactly one row block and with more (several row blocks of one expert), gathered through a
  shuffled route order; k-tile counts below the streaming kernel's ring depth; both code books,
  two and four scale slots, the plain and the SiLU-mul epilogue; decode-sized batches (the
  streaming kernel), a shape the general tile kernel takes, the 32- and 64-row tile kernels (whose
  loads straight into LDS take their row offsets from the gathered route list), and many rows per
  expert (the 128 x 256 tiles of the many-row kernel)."""
  from tunix_amd import _lib as L
  from tunix_amd import ops
  rng = np.random.Generator(np.random.PCG64(2000 + E + N))
  n_routes = n_tok * k
  if E == 16:
    cnt = np.zeros(E, dtype=np.int64)
    cnt[[0, 2, 3, 5, 6, 7]] = [40, 3, 17, 1, 16, n_routes - 77]
  elif E == 8 and n_routes >= 1024:   # empty experts, one row, exactly one 128-row block, one row more, several blocks
    cnt = np.array([300, 0, 129, 128, 1, 200, n_routes - 758, 0], dtype=np.int64)
  else:
    ids = rng.integers(0, E - 3, size=n_routes)
    ids[:40] = 7                                    # one expert far above the average
    cnt = np.bincount(ids, minlength=E)
  assert cnt.sum() == n_routes and cnt.min() == 0 and cnt.max() > 16
  expert_of = np.repeat(np.arange(E), cnt)          # expert of each sorted position
  sorted_route = rng.permutation(n_routes).astype(np.int32)   # position -> route (= output row)
  offs = np.concatenate([[0], np.cumsum(cnt)]).astype(np.int32)
  x_div = k if mul else 1
  x = rnd((n_routes // x_div, K), 90)
  w = rnd((E, K, N), 91, 0.05)
  cb, sb = ops.qw_sizes(K, N, group)
  gc = torch.empty(E * cb // 4, dtype=torch.int32, device=gpu)
  gs = torch.empty(E * sb // 2, dtype=torch.bfloat16, device=gpu)
  ncol = N // 2 if mul else N
  ref = torch.full((n_routes, ncol), 7.0)
  for e in range(E):
    c, s = ops.quantize_pack(bf(w[e]).to(gpu), group, qtype, mul)
    gc[e * cb // 4:(e + 1) * cb // 4] = c
    gs[e * sb // 2:(e + 1) * sb // 2] = s
    if cnt[e] == 0:
      continue
    dq = torch.from_numpy(Q.dequantize(*Q.quantize(w[e].numpy(), group, qtype), group, qtype)).double()
    routes = torch.from_numpy(sorted_route[offs[e]:offs[e + 1]].astype(np.int64))
    yy = Q.rb((x[routes // x_div].double() @ dq).float())
    if mul:
      gg, uu = yy[:, :N // 2], yy[:, N // 2:]
      yy = Q.rb(Q.rb(gg * Q.rb(torch.sigmoid(gg))) * uu)
    ref[routes] = yy
  y = torch.full((n_routes, ncol), 7.0, dtype=torch.bfloat16, device=gpu)
  d = L.MoeGmmDesc()
  d.n_routes, d.E, d.k, d.K, d.N, d.group, d.qtype = n_routes, E, k, K, N, group, qtype
  buf = torch.zeros(x.numel() + 8, dtype=torch.bfloat16, device=gpu)   # (on a boundary; x starts `off` elements behind it)
  gx = buf[off:off + x.numel()].view(x.shape).copy_(x)
  d.x, d.x_div, d.codes, d.scales = gx.data_ptr(), x_div, gc.data_ptr(), gs.data_ptr()
  go, gr = torch.from_numpy(offs).to(gpu), torch.from_numpy(sorted_route).to(gpu)
  d.offsets, d.sorted_route = go.data_ptr(), gr.data_ptr()
  d.epilogue, d.y = (L.TNX_EPI_SILU_MUL if mul else L.TNX_EPI_STORE), y.data_ptr()
  for _ in range(2):
    ops.moe_gmm(d)
  torch.cuda.synchronize()
  # (the activation is computed from two rounded tiles and rounded three more times: one ulp on
  # the gate and one on the up value can add up to three on the product)
  assert_bf16_close(y, ref, atol=1e-5, min_equal=0.9 if mul else 0.97, what="moe gmm", ulps=3 if mul else 1)


@pytest.mark.parametrize("E,n_tok,k,K,N,group,qtype,mul,off", [
    (16, 48, 2, 128, 128, 64, Q.NF4, True, 0),        # four rows to a kilobyte of LDS, fewer k-tiles than the ring has
    (256, 256, 4, 128, 576, 32, Q.INT4, False, 0),    # runs that span two blocks, work-groups of three
    (16, 48, 2, 4992, 96, 128, Q.INT4, False, 0),     # (256 compute units) the most that LDS holds of sixteen rows, and beyond it the form without
    (16, 48, 2, 5120, 96, 128, Q.INT4, False, 0),
    (16, 48, 2, 2944, 64, 64, Q.NF4, True, 0),        # the same next to a table of levels
    (16, 48, 2, 3072, 64, 64, Q.NF4, True, 0),
    (256, 256, 4, 2304, 32, 128, Q.INT4, False, 0),   # of two blocks
    (256, 256, 4, 2432, 32, 128, Q.INT4, False, 0),
    (16, 48, 2, 512, 256, 128, Q.INT4, True, 1),      # rows off a 16-byte boundary: the form without
    (16, 48, 2, 512, 256, 64, Q.NF4, False, 4),
])
def test_moe_gmm_rows_in_lds(gpu, E, n_tok, k, K, N, group, qtype, mul, off):
  """The decode-sized grouped GEMM at the edges of its form that stages the rows."""
  test_moe_gmm_skewed_routes(gpu, E, n_tok, k, K, N, group, qtype, mul, off)


@pytest.mark.parametrize("E,M,k,K,N,group,qtype,mul", [
    (128, 64, 8, 256, 128, 128, Q.INT4, True),
    (128, 1, 8, 256, 128, 64, Q.NF4, False),
    (65, 63, 3, 128, 96, 64, Q.NF4, True),
    (16, 65, 2, 256, 64, 32, Q.INT4, False),      # rows in both words of an expert's bits; experts of several blocks
    (300, 128, 8, 128, 64, 128, Q.INT4, True),    # 1024 routes, several turns of 64 experts
    (200, 128, 16, 128, 32, 64, Q.NF4, False),    # 2048: more than the work-group has threads
    (3, 2, 3, 128, 32, 64, Q.INT4, False),        # every expert for every row
    (64, 16, 4, 128, 64, 64, Q.INT4, True),
])
def test_moe_linears_that_sort_the_routes(gpu, E, M, k, K, N, group, qtype, mul):
  """The experts' linear from the ids alone against the sorted routes: the same bits, also where most rows choose the same experts."""
  from tunix_amd import _lib as L
  from tunix_amd import ops
  g = torch.Generator(device=gpu).manual_seed(E + M)
  w = [ops.quantize_pack((torch.randn(K, N, generator=g, device=gpu) * 0.05).bfloat16(), group, qtype, mul) for _ in range(min(E, 8))]
  codes, scales = (torch.cat([w[e % len(w)][i].reshape(-1) for e in range(E)]) for i in (0, 1))
  x = torch.randn(M if mul else M * k, K, generator=g, device=gpu).bfloat16()
  for skew in (0.0, 4.0):
    scores = torch.randn(M, E, generator=g, device=gpu) - skew * torch.arange(E, device=gpu) / E
    ids = scores.topk(k, dim=1).indices.int().contiguous()
    cnt, offs, sr = (torch.empty(n, dtype=torch.int32, device=gpu) for n in (E, E + 1, M * k))
    ops.moe_sort_routes(ids, E, cnt, offs, sr)
    outs = []
    for unsorted in (False, True):
      y = torch.full((M * k, N // 2 if mul else N), float("nan"), dtype=torch.bfloat16, device=gpu)
      d = L.MoeGmmDesc()
      d.n_routes, d.E, d.k, d.K, d.N, d.group, d.qtype = M * k, E, k, K, N, group, qtype
      d.x, d.x_div, d.codes, d.scales = x.data_ptr(), k if mul else 1, codes.data_ptr(), scales.data_ptr()
      d.epilogue, d.y = (L.TNX_EPI_SILU_MUL if mul else L.TNX_EPI_STORE), y.data_ptr()
      assert ops.moe_gmm_unsorted_ok(d)
      if unsorted:
        ops.moe_gmm_unsorted(d, ids)
      else:
        d.offsets, d.sorted_route = offs.data_ptr(), sr.data_ptr()
        ops.moe_gmm(d)
      outs.append(y)
    torch.cuda.synchronize()
    assert not outs[0].isnan().any() and torch.equal(outs[0].view(torch.int16), outs[1].view(torch.int16)), skew


def test_moe_linears_that_sort_refuse(gpu):
  """More than 128 rows, a part of a row, more rows per expert than the streaming kernel takes, and ids of another number."""
  from tunix_amd import _lib as L
  from tunix_amd import ops
  z = torch.zeros(1 << 16, dtype=torch.int32, device=gpu)
  for E, n_routes, k in ((64, 129 * 2, 2), (64, 127, 2), (4, 128, 2)):
    d = L.MoeGmmDesc()
    d.n_routes, d.E, d.k, d.K, d.N, d.group, d.qtype, d.x_div = n_routes, E, k, 128, 64, 64, Q.INT4, 1
    d.x = d.codes = d.scales = d.y = z.data_ptr()
    assert not ops.moe_gmm_unsorted_ok(d)
    with pytest.raises(ValueError, match="not a shape it takes"):
      ops.moe_gmm_unsorted(d, z[:n_routes])
  with pytest.raises(ValueError, match="all routes"):
    ops.moe_gmm_unsorted(d, z[:n_routes + 1])


def test_argument_errors_raise(gpu):
  from tunix_amd import ops
  with pytest.raises(ValueError, match="K % 128"):
    ops.qw_sizes(100, 64, 64)
  x = torch.zeros(4, 128, dtype=torch.bfloat16, device=gpu)
  with pytest.raises(ValueError):
    ops.quantize_pack(x.t().contiguous(), 48, 0)


@pytest.mark.parametrize("family,M,k,D", [("qwen3", 64, 8, 2048), ("llama3", 5, 11, 512), ("gemma3", 3, 1, 4104)])
def test_rmsnorm_moe_combine_equals_combine_then_norm(gpu, family, M, k, D):
  """The folded pass (weighted combine of a token's k routed rows + residual + norm) against the
  two separate kernels it replaces: the new residual stream and the normed row bit for bit; more
  routes per token than one group of loads takes, a width that is not a multiple of 2048."""
  from tunix_amd import ops
  from tunix_amd.model import _NORM
  yr = bf(rnd((M * k, D), 310)).to(gpu)
  tw = bf(torch.softmax(rnd((M, k), 311), -1)).to(gpu)
  res = bf(rnd((M, D), 312)).to(gpu)
  nw = bf(rnd((D,), 313, 0.3) + 1.0).to(gpu)
  h1 = res.clone()
  ops.moe_combine(yr, tw, M, k, D, h1, h1)
  y1 = torch.empty_like(h1)
  ops.rmsnorm(h1, nw, y1, 1e-6, _NORM[family])
  h2 = res.clone()
  y2 = torch.empty_like(h1)
  ops.rmsnorm_moe_combine(yr, tw, k, nw, y2, 1e-6, _NORM[family], M, D, res_pre=h2, h_out=h2)
  torch.cuda.synchronize()
  assert torch.equal(h1, h2) and torch.equal(y1, y2)
  assert not torch.equal(h1, res)


@pytest.mark.parametrize("family", ["llama3", "qwen3"])
def test_rmsnorm_splitk_equals_finish_then_norm(gpu, family):
  """The folded pass (sum of split-k planes + residual + norm) against the two separate
  kernels it replaces: bit for bit."""
  from tunix_amd import _lib as L
  from tunix_amd import ops
  from tunix_amd.model import _NORM
  M, K, D, g, split = 128, 1024, 512, 64, 4
  x, res = rnd((M, K), 80), rnd((M, D), 81)
  w = rnd((K, D), 82, 0.02)
  nw = bf(rnd((D,), 83, 0.3) + 1.0).to(gpu)
  c, s = ops.quantize_pack(bf(w).to(gpu), g, Q.NF4)
  gx, gres = bf(x).to(gpu), bf(res).to(gpu)
  ws = torch.empty(split * M * D, dtype=torch.float32, device=gpu)
  h1 = torch.empty(M, D, dtype=torch.bfloat16, device=gpu)
  d = ops.make_qlinear_desc(M=M, K=K, N=D, group=g, qtype=Q.NF4, x=gx, codes=c, scales=s, y=h1,
                            epilogue=L.TNX_EPI_RESIDUAL, residual=gres, split_k=split, ws=ws)
  ops.qlinear(d)                                   # partial planes + finishing pass
  y1 = torch.empty_like(h1)
  ops.rmsnorm(h1, nw, y1, 1e-5, _NORM[family])
  ops.qlinear(d, finish=False)                     # planes only
  h2 = gres.clone()
  y2 = torch.empty_like(h1)
  ops.rmsnorm_splitk(ws, split, nw, y2, 1e-5, _NORM[family], M, D, res_pre=h2, h_out=h2)
  torch.cuda.synchronize()
  assert torch.equal(h1, h2)
  assert torch.equal(y1, y2)


@pytest.mark.parametrize("family", ["llama3", "qwen3", "gemma3"])
@pytest.mark.parametrize("planes", [False, True])
def test_rmsnorm_pair_equals_two_norms(gpu, family, planes):
  """Post-norm + residual + next pre-norm in one launch (Gemma-3's block structure) against the
  launches it replaces -- split-k finishing pass, norm with residual, norm -- bit for bit, and
  the first norm against the oracle."""
  from tunix_amd import _lib as L
  from tunix_amd import ops
  from tunix_amd.model import _NORM
  M, K, D, g, split = 70, 1024, 1152, 128, 4
  x, res = rnd((M, K), 90), rnd((M, D), 91)
  w = rnd((K, D), 92, 0.02)
  w1 = bf(rnd((D,), 93, 0.3) + 1.0).to(gpu)
  w2 = bf(rnd((D,), 94, 0.3) + 1.0).to(gpu)
  c, s = ops.quantize_pack(bf(w).to(gpu), g, Q.INT4)
  gx = bf(x).to(gpu)
  ws = torch.empty(split * M * D, dtype=torch.float32, device=gpu)
  tmp = torch.empty(M, D, dtype=torch.bfloat16, device=gpu)
  d = ops.make_qlinear_desc(M=M, K=K, N=D, group=g, qtype=Q.INT4, x=gx, codes=c, scales=s, y=tmp,
                            split_k=split, ws=ws)
  ops.qlinear(d)                                   # planes + finishing pass -> tmp
  h1 = bf(res).to(gpu)
  xn1 = torch.empty_like(tmp)
  ops.rmsnorm(tmp, w1, h1, 1e-6, _NORM[family], res_post=h1)
  ops.rmsnorm(h1, w2, xn1, 1e-6, _NORM[family])
  h2 = bf(res).to(gpu)
  xn2 = torch.empty_like(tmp)
  if planes:
    ops.qlinear(d, finish=False)
    ops.rmsnorm_pair(w1, h2, w2, xn2, 1e-6, _NORM[family], M, D, ws=ws, split_k=split, res_post=h2)
  else:
    ops.rmsnorm_pair(w1, h2, w2, xn2, 1e-6, _NORM[family], M, D, x=tmp, res_post=h2)
  torch.cuda.synchronize()
  assert torch.equal(h1, h2)
  assert torch.equal(xn1, xn2)
  ref_m = MR.RefModel.__new__(MR.RefModel)
  ref_m.cfg, ref_m.bf16 = _Cfg(family, 1e-6), True
  ref_h = Q.rb(ref_m.rmsnorm(tmp.float().cpu(), w1.float().cpu()) + Q.rb(res))
  assert_bf16_close(h2, ref_h, min_equal=0.95, what="pair: first norm + residual")
  assert_bf16_close(xn2, ref_m.rmsnorm(h2.float().cpu(), w2.float().cpu()), min_equal=0.95, what="pair: second norm")
  with pytest.raises(ValueError):
    ops.rmsnorm_pair(w1, h2, w2, xn2, 1e-6, _NORM[family], M, D, res_post=h2)   # neither x nor ws


def assert_down_projection(t, x, a, what=""):
  """t against the exact product of bf16 rows and adapter columns.  32-bit sums: at most 16 products behind each other per thread, then
  two binary trees over 256 of them, i.e. 32 roundings of 2^-24 of the sum of magnitudes; and the rounding to bf16."""
  ref, mag = x.double() @ a.double().T, x.double().abs() @ a.double().abs().T
  bad = (t.double() - ref).abs() > 2.0 ** -8 * ref.abs() + 32 * 2.0 ** -24 * mag
  assert not bool(bad.any()), f"{what}: {int(bad.sum())} of {bad.numel()}"


@pytest.mark.parametrize("family", ["llama3", "qwen3", "gemma3"])
@pytest.mark.parametrize("src,M,D,R,parts", [
    ("rows", 1, 32, 16, 0), ("rows", 5, 4096, 48, 0),
    ("planes", 3, 2048, 192, 8), ("planes", 16, 4096, 192, 5), ("planes", 17, 4096, 64, 2),   # 17 rows of 4096: two launches
    ("planes", 8, 2080, 16, 11), ("planes", 64, 1152, 96, 8), ("planes", 256, 512, 32, 4), ("planes", 257, 512, 32, 4),
    ("planes", 2, 4128, 64, 3),                                                               # past 4096: two launches
    ("routes", 9, 2048, 128, 8), ("routes", 4, 3072, 48, 10),
    ("pair", 7, 1152, 96, 0), ("pair", 128, 1152, 64, 8), ("pair", 1, 4096, 208, 8),
])
def test_norm_and_down_projection_in_one_launch(gpu, family, src, M, D, R, parts):
  """tnx_norm_lora against the norm of its own (rows bit for bit) and the exact down-projection of what it wrote; with an output in
  place of an input it takes two launches, with the same rows."""
  from tunix_amd import ops
  from tunix_amd.model import _NORM
  fl, eps = _NORM[family], 1e-6
  w, w2 = bf(rnd((D,), 95, 0.3) + 1.0).to(gpu), bf(rnd((D,), 96, 0.3) + 1.0).to(gpu)
  a, res = bf(rnd((R, D), 97)).to(gpu), bf(rnd((M, D), 98)).to(gpu)
  x = bf(rnd((M, D), 99)).to(gpu)
  ws = rnd((max(parts, 1), M, D), 100).to(gpu)
  routes, tw = bf(rnd((M * max(parts, 1), D), 101)).to(gpu), bf(rnd((M, max(parts, 1)), 102, 0.2)).to(gpu)
  new = lambda: torch.full((M, D), float("nan"), dtype=torch.bfloat16, device=gpu)
  h1, y1, h2, y2 = new(), new(), new(), new()
  t = torch.full((M, R + 8), 7.0, dtype=torch.bfloat16, device=gpu)
  kw = dict(ws=ws, split_k=parts) if src != "pair" or parts else dict(x=x)
  if src == "rows":
    ops.rmsnorm(x, w, y1, eps, fl)
    one = lambda h_in, h_out, y: ops.norm_lora(a, t, w, y, eps, fl, M, D, x=x)
  elif src == "planes":
    ops.rmsnorm_splitk(ws, parts, w, y1, eps, fl, M, D, res_pre=res, h_out=h1)
    one = lambda h_in, h_out, y: ops.norm_lora(a, t, w, y, eps, fl, M, D, res_pre=h_in, h_out=h_out, **kw)
  elif src == "routes":
    ops.rmsnorm_moe_combine(routes, tw, parts, w, y1, eps, fl, M, D, res_pre=res, h_out=h1)
    one = lambda h_in, h_out, y: ops.norm_lora(a, t, w, y, eps, fl, M, D, y_route=routes, topk_w=tw, k=parts, res_pre=h_in, h_out=h_out)
  else:
    ops.rmsnorm_pair(w, h1, w2, y1, eps, fl, M, D, res_post=res, **kw)
    one = lambda h_in, h_out, y: ops.norm_lora(a, t, w, h_out, eps, fl, M, D, res_post=h_in, w2=w2, y2=y, **kw)
  one(res, h2, y2)
  torch.cuda.synchronize()
  assert torch.equal(y1, y2) and (src == "rows" or torch.equal(h1, h2))
  assert_down_projection(t[:, :R], y2, a, "apart")
  assert bool((t[:, R:] == 7.0).all())
  t.fill_(7.0)
  h3, y3 = res.clone(), new()
  one(h3, h3, y3)
  torch.cuda.synchronize()
  assert torch.equal(y1, y3) and (src == "rows" or torch.equal(h1, h3))
  assert_down_projection(t[:, :R], y3, a, "in place")
  with pytest.raises(ValueError):
    ops.norm_lora(a, t, w, y2, eps, fl, M, D)           # no input


@pytest.mark.parametrize("place", ["x", "ws", "y_route", "res_pre", "w", "h_out"])
def test_norm_and_down_projection_over_an_input(gpu, place):
  """tnx_norm_lora with t in the memory of an input, or of its other output, that row's other work-groups still read: two launches, whose bits it has."""
  from tunix_amd import ops
  M, D, R, parts = 16, 512, 32, 2
  got = []
  for one in (False, True):
    x, res, h, y = bf(rnd((M, D), 99)).to(gpu), bf(rnd((M, D), 98)).to(gpu), *(torch.zeros(M, D, dtype=torch.bfloat16, device=gpu) for _ in range(2))
    w = bf(torch.cat([rnd((D,), 95, 0.3) + 1.0, torch.zeros(M * R)])).to(gpu)
    ws, routes = rnd((parts, M, D), 100).to(gpu), bf(rnd((M * parts, D), 101)).to(gpu)
    tw, a = bf(rnd((M, parts), 102, 0.2)).to(gpu), bf(rnd((R, D), 97)).to(gpu)
    t = {"x": x, "ws": ws.view(torch.bfloat16), "y_route": routes, "res_pre": res, "w": w, "h_out": h}[place].reshape(-1)[:M * R].view(M, R)
    if place in ("x", "w"):
      ops.norm_lora(a, t, w, y, 1e-6, 0, M, D, x=x) if one else ops.rmsnorm(x, w, y, 1e-6, 0)
    elif place == "y_route":
      kw = dict(res_pre=res, h_out=h)
      ops.norm_lora(a, t, w, y, 1e-6, 0, M, D, y_route=routes, topk_w=tw, k=parts, **kw) if one else ops.rmsnorm_moe_combine(
          routes, tw, parts, w, y, 1e-6, 0, M, D, **kw)
    else:
      kw = dict(res_pre=res, h_out=h)
      ops.norm_lora(a, t, w, y, 1e-6, 0, M, D, ws=ws, split_k=parts, **kw) if one else ops.rmsnorm_splitk(ws, parts, w, y, 1e-6, 0, M, D, **kw)
    if not one:
      ops.lora_down(y, a, t)
    torch.cuda.synchronize()
    got.append((y.clone(), t.clone(), h.clone()))
  assert all(torch.equal(p, q) for p, q in zip(*got))


@pytest.mark.parametrize("B,Hq,Hkv,dh,S,kv_chunk,R,window,at", [
    (1, 8, 2, 64, 128, 32, 32, 0, 127), (3, 32, 8, 128, 128, 32, 64, 0, 40),     # chunks without a key
    (70, 4, 1, 256, 288, 32, 32, 0, 280), (5, 4, 1, 256, 500, 32, 48, 100, 470),   # nine and sixteen chunks, a window
    (2, 32, 8, 128, 160, 32, 64, 0, 150),                                           # five chunks of 4096: two launches
    (128, 4, 1, 64, 96, 32, 32, 0, 90), (129, 4, 1, 64, 96, 32, 32, 0, 90),         # 256 work-groups of rows and columns, and more: two launches
    (4, 8, 8, 64, 96, 96, 16, 0, 90), (9, 40, 8, 128, 64, 32, 16, 0, 63),           # one chunk; 5120 outputs
])
def test_attention_and_down_projection(gpu, B, Hq, Hkv, dh, S, kv_chunk, R, window, at):
  """tnx_gqa_attn_lora against tnx_gqa_attn (bit for bit) and the exact down-projection of its output."""
  from tunix_amd import _lib as L
  from tunix_amd import ops
  k, v = bf(rnd((B, Hkv, S, dh), 103)).to(gpu), bf(rnd((B, Hkv, S, dh), 104)).to(gpu)
  q, a = bf(rnd((B, Hq * dh), 105)).to(gpu), bf(rnd((R, Hq * dh), 106)).to(gpu)
  tokens = torch.ones(B, S, dtype=torch.int32, device=gpu)
  tokens[:, :5] = 0
  col = torch.full((1,), at, dtype=torch.int32, device=gpu)
  outs = [torch.full((B, Hq * dh), float("nan"), dtype=torch.bfloat16, device=gpu) for _ in range(2)]
  t = torch.full((B, R + 16), 7.0, dtype=torch.bfloat16, device=gpu)
  for i, out in enumerate(outs):
    ws = torch.full((max(ops.attn_ws_bytes(B, 1, S, Hq, dh, kv_chunk) // 4, 1),), float("nan"), device=gpu)
    d = L.AttnDesc()
    d.B, d.T, d.S, d.Hq, d.Hkv, d.dh = B, 1, S, Hq, Hkv, dh
    d.scale, d.window, d.pad_id = dh ** -0.5, window, 0
    d.q, d.kcache, d.vcache = q.data_ptr(), k.data_ptr(), v.data_ptr()
    d.tokens, d.tok_ld, d.col_ptr = tokens.data_ptr(), S, col.data_ptr()
    d.kv_chunk, d.ws, d.out = kv_chunk, ws.data_ptr(), out.data_ptr()
    if i:
      ops.gqa_attn_lora(d, a, t)
    else:
      ops.gqa_attn(d)
    torch.cuda.synchronize()
  assert torch.equal(*outs)
  assert bool(torch.isfinite(outs[0].float()).all())
  assert_down_projection(t[:, :R], outs[1], a)
  assert bool((t[:, R:] == 7.0).all())


@pytest.mark.parametrize("chunk,place", [(32, "t in ws"), (0, "out in planes"), (64, "ws in planes")])
def test_attention_outputs_over_what_it_reads(gpu, chunk, place):
  """The adapter's output in the memory of the chunks' partials, or the attention's in that of the qkv linear's planes, which other work-groups of
  the same row still read: separate launches, whose bits it has."""
  from tunix_amd import _lib as L
  from tunix_amd import ops
  from tunix_amd.model import rope_timescale
  B, S, Hq, Hkv, dh, R, parts = 4, 128, 8, 2, 64, 32, 4
  ts = torch.from_numpy(rope_timescale(dh, 1e4)).to(gpu)
  pos = torch.arange(S, dtype=torch.int32, device=gpu).repeat(B, 1).contiguous()
  tokens, col = torch.ones(B, S, dtype=torch.int32, device=gpu), torch.full((1,), 120, dtype=torch.int32, device=gpu)
  a = bf(rnd((R, Hq * dh), 106)).to(gpu)
  got = []
  for one in (False, True):
    k, v = bf(rnd((B, Hkv, S, dh), 103)).to(gpu), bf(rnd((B, Hkv, S, dh), 104)).to(gpu)
    planes, q = rnd((parts, B, (Hq + 2 * Hkv) * dh), 107).to(gpu), bf(rnd((B, Hq * dh), 105)).to(gpu)
    n_ws = max(ops.attn_ws_bytes(B, 1, S, Hq, dh, chunk) // 4, 1)
    ws, out = torch.zeros(n_ws, device=gpu), torch.zeros(B, Hq * dh, dtype=torch.bfloat16, device=gpu)
    t = torch.zeros(B, R, dtype=torch.bfloat16, device=gpu)
    if place == "t in ws":
      t = ws.view(torch.bfloat16)[:B * R].view(B, R)
    elif place == "out in planes":
      out = planes.view(torch.bfloat16).reshape(-1)[:B * Hq * dh].view(B, Hq * dh)
    else:
      assert n_ws <= planes.numel()
      ws = planes.view(-1)[:n_ws]
    rd, d = L.RopeDesc(), L.AttnDesc()
    for x in (rd, d):
      x.B, x.T, x.S, x.Hq, x.Hkv, x.dh = B, 1, S, Hq, Hkv, dh
      x.kcache, x.vcache, x.col_ptr = k.data_ptr(), v.data_ptr(), col.data_ptr()
    rd.rope_flavor, rd.rope_scale, rd.timescale, rd.qk_norm = L.TNX_ROPE_QWEN3, 1.0, ts.data_ptr(), -1
    rd.qkv_ws, rd.split_k, rd.positions, rd.pos_ld, rd.q_out = planes.data_ptr(), parts, pos.data_ptr(), S, q.data_ptr()
    d.scale, d.q, d.out, d.ws, d.kv_chunk = dh ** -0.5, q.data_ptr(), out.data_ptr(), ws.data_ptr(), chunk
    d.tokens, d.tok_ld = tokens.data_ptr(), S
    if place == "t in ws":
      ops.gqa_attn_lora(d, a, t) if one else ops.gqa_attn(d)
    elif one:
      ops.rope_gqa_attn_lora(rd, d, a, t)
    else:
      ops.rope_kvwrite(rd)
      ops.gqa_attn(d)
    if not one:
      ops.lora_down(out, a, t)
    torch.cuda.synchronize()
    got.append((out.clone(), t.clone(), k, v))
  assert all(torch.equal(x, y) for x, y in zip(*got))


@pytest.mark.parametrize("lora", [False, True])
@pytest.mark.parametrize("B,Hq,Hkv,dh,S,kv_chunk,where", [
    (2, 8, 2, 128, 200, 0, "q"), (2, 8, 2, 64, 60, 0, "q"), (3, 4, 1, 256, 300, 0, "k"), (2, 8, 2, 128, 384, 96, "q"),
    (2, 8, 2, 128, 384, 96, "k"), (2, 4, 2, 64, 128, 32, "k"), (2, 8, 2, 128, 256, 128, "v"), (600, 8, 1, 64, 128, 0, "k")])
def test_decode_attention_keeps_a_nan(gpu, B, Hq, Hkv, dh, S, kv_chunk, where, lora):
  """A NaN in a head's query, or in one key or value of its kv head, is in the output of those heads and of no other, however the keys are divided
  among waves and chunks: a share whose sum is NaN is none without a key."""
  from tunix_amd import _lib as L
  from tunix_amd import ops
  k, v, q = bf(rnd((B, Hkv, S, dh), 113)), bf(rnd((B, Hkv, S, dh), 114)), bf(rnd((B, Hq, dh), 115))
  want = torch.zeros(B, Hq, dh, dtype=torch.bool)
  if where == "q":
    q[1, 2, 5] = float("nan")
    want[1, 2] = True
  elif where == "k":
    k[1, 0, 40, 3] = float("nan")
    want[1, :Hq // Hkv] = True
  else:
    v[1, 0, 40, 3] = float("nan")
    want[1, :Hq // Hkv, 3] = True
  k, v, q = k.to(gpu), v.to(gpu), q.to(gpu)
  tokens, col = torch.ones(B, S, dtype=torch.int32, device=gpu), torch.full((1,), S - 1, dtype=torch.int32, device=gpu)
  ws = torch.full((max(ops.attn_ws_bytes(B, 1, S, Hq, dh, kv_chunk) // 4, 1),), float("nan"), device=gpu)
  out = torch.zeros(B, Hq * dh, dtype=torch.bfloat16, device=gpu)
  d = L.AttnDesc()
  d.B, d.T, d.S, d.Hq, d.Hkv, d.dh = B, 1, S, Hq, Hkv, dh
  d.scale, d.window, d.pad_id = dh ** -0.5, 0, 0
  d.q, d.kcache, d.vcache = q.data_ptr(), k.data_ptr(), v.data_ptr()
  d.tokens, d.tok_ld, d.col_ptr = tokens.data_ptr(), S, col.data_ptr()
  d.kv_chunk, d.ws, d.out = kv_chunk, ws.data_ptr(), out.data_ptr()
  if lora:
    a, t = bf(rnd((16, Hq * dh), 116)).to(gpu), torch.zeros(B, 16, dtype=torch.bfloat16, device=gpu)
    ops.gqa_attn_lora(d, a, t)
    torch.cuda.synchronize()
    assert torch.equal(torch.isnan(t).any(1).cpu(), want.flatten(1).any(1))
  else:
    ops.gqa_attn(d)
    torch.cuda.synchronize()
  assert torch.equal(torch.isnan(out).cpu().view(B, Hq, dh), want)


@pytest.mark.parametrize("kv_chunk,window,planes,Hq,split", [
    (0, 0, False, 8, 3), (32, 0, True, 8, 3), (0, 40, True, 8, 3), (64, 0, False, 8, 3),
    (0, 0, True, 16, 3),     # eight query heads per kv head: more than one set of plane loads
    (0, 0, True, 8, 11),     # more than eight partial planes
    (0, 0, True, 4, 8),      # two query heads per kv head, eight planes
])
def test_attention_with_fused_rope_equals_rope_then_attention(gpu, kv_chunk, window, planes, Hq, split):
  """Decode attention that rotates q / k and writes the step's key / value itself (from the qkv
  linear's bf16 output or its split-k planes) against the two launches it replaces: the cache
  ends up bit-identical, the output agrees to a bf16 ulp (the step's own key enters the online
  softmax as a block of its own instead of inside the last 32-key block)."""
  from tunix_amd import _lib as L
  from tunix_amd import ops
  from tunix_amd.model import rope_timescale
  B, S, Hkv, dh, col = 6, 96, 2, 128, 70
  ld = (Hq + 2 * Hkv) * dh
  g = torch.Generator().manual_seed(95)
  pl = torch.randn(split, B, ld, generator=g).float()
  qkv = pl.sum(0).to(torch.bfloat16)
  ws = pl.to(gpu).contiguous() if planes else None
  if planes:   # the reference path sees bf16(sum of planes in split order)
    acc = torch.zeros(B, ld)
    for z in range(split):
      acc = acc + pl[z]
    qkv = acc.to(torch.bfloat16)
  gq = qkv.to(gpu)
  pos = torch.randint(0, 900, (B, S), generator=g, dtype=torch.int32).to(gpu)
  ts = torch.from_numpy(rope_timescale(dh, 5e5)).to(gpu)
  tokens = torch.randint(1, 50, (B, S), generator=g, dtype=torch.int32)
  tokens[1, :9] = 0                                                # a left-padded row
  tokens = tokens.to(gpu)
  colp = torch.tensor([col], dtype=torch.int32, device=gpu)
  kc0 = torch.randn(B, Hkv, S, dh, generator=g).to(torch.bfloat16).to(gpu)
  vc0 = torch.randn(B, Hkv, S, dh, generator=g).to(torch.bfloat16).to(gpu)

  def attn(q, kc, vc, fused):
    d = L.AttnDesc()
    d.B, d.T, d.S, d.Hq, d.Hkv, d.dh = B, 1, S, Hq, Hkv, dh
    d.scale, d.window, d.pad_id = dh ** -0.5, window, 0
    d.kcache, d.vcache = kc.data_ptr(), vc.data_ptr()
    d.tokens, d.tok_ld, d.col_ptr = tokens.data_ptr(), S, colp.data_ptr()
    d.kv_chunk = kv_chunk
    wsa = torch.empty(max(ops.attn_ws_bytes(B, 1, S, Hq, dh, kv_chunk) // 4, 1), dtype=torch.float32, device=gpu)
    out = torch.empty(B, Hq * dh, dtype=torch.bfloat16, device=gpu)
    d.ws, d.out = wsa.data_ptr(), out.data_ptr()
    if fused:
      if planes:
        d.qkv_ws, d.qkv_split = ws.data_ptr(), split
      else:
        d.qkv = gq.data_ptr()
      sn = torch.empty(B, dh // 2, dtype=torch.float32, device=gpu)
      cs = torch.empty_like(sn)
      ops.rope_table(pos, colp, B, ts, dh, sn, cs)
      d.rope_sin, d.rope_cos = sn.data_ptr(), cs.data_ptr()
    else:
      d.q = q.data_ptr()
    ops.gqa_attn(d)
    torch.cuda.synchronize()
    return out

  # the two launches
  kc1, vc1 = kc0.clone(), vc0.clone()
  rd = L.RopeDesc()
  rd.B, rd.T, rd.S, rd.Hq, rd.Hkv, rd.dh = B, 1, S, Hq, Hkv, dh
  rd.rope_flavor, rd.rope_scale, rd.timescale, rd.qk_norm = L.TNX_ROPE_LLAMA, 1.0, ts.data_ptr(), -1
  q1 = torch.empty(B, Hq * dh, dtype=torch.bfloat16, device=gpu)
  rd.qkv, rd.positions, rd.pos_ld, rd.col_ptr = gq.data_ptr(), pos.data_ptr(), S, colp.data_ptr()
  rd.q_out, rd.kcache, rd.vcache = q1.data_ptr(), kc1.data_ptr(), vc1.data_ptr()
  ops.rope_kvwrite(rd)
  out1 = attn(q1, kc1, vc1, False)
  # the fused launch
  kc2, vc2 = kc0.clone(), vc0.clone()
  out2 = attn(None, kc2, vc2, True)
  assert torch.equal(kc1, kc2) and torch.equal(vc1, vc2)
  assert not torch.equal(kc2, kc0)
  assert out1.float().abs().max() > 0.05
  # one bf16 ulp of the larger of the two values (4e-3 below 1)
  d = (out1.float() - out2.float()).abs()
  ulp = 2.0 ** (torch.floor(torch.log2(torch.maximum(out1.float().abs(), out2.float().abs()).clamp_min(0.5))) - 7)
  assert (d <= ulp).all(), (d.max().item(), (d / ulp).max().item())


@pytest.mark.parametrize("family,dh,Hq,Hkv", [("llama3", 128, 8, 2), ("gemma3", 256, 4, 1), ("qwen3", 64, 6, 3)])
def test_rope_row_kernel_equals_the_per_head_kernel(gpu, family, dh, Hq, Hkv):
  """Rotation + cache write without q / k norm at many rows (512 in one call: the row kernel, 16-byte
  accesses, one sine / cosine per (row, i) for all heads) against the same rows in calls of 128
  (the per-head kernel): q and both caches bit for bit."""
  from tunix_amd import _lib as L
  from tunix_amd import ops
  from tunix_amd.model import _ROPE, rope_timescale
  B, T, S, col = 4, 128, 160, 9
  ld = (Hq + 2 * Hkv) * dh
  g = torch.Generator().manual_seed(96)
  qkv = torch.randn(B, T, ld, generator=g).to(torch.bfloat16).to(gpu)
  pos = torch.randint(0, 2000, (B, S), generator=g, dtype=torch.int32).to(gpu)
  ts = torch.from_numpy(rope_timescale(dh, 1e6)).to(gpu)
  colp = torch.tensor([col], dtype=torch.int32, device=gpu)

  def run(rows_per_call):
    q = torch.zeros(B, T, Hq * dh, dtype=torch.bfloat16, device=gpu)
    kc = torch.zeros(B, Hkv, S, dh, dtype=torch.bfloat16, device=gpu)
    vc = torch.zeros_like(kc)
    for b0 in range(0, B, rows_per_call):
      nb = min(rows_per_call, B - b0)
      rd = L.RopeDesc()
      rd.B, rd.T, rd.S, rd.Hq, rd.Hkv, rd.dh = nb, T, S, Hq, Hkv, dh
      rd.rope_flavor, rd.rope_scale, rd.timescale, rd.qk_norm = _ROPE[family], 8.0 if family == "gemma3" else 1.0, ts.data_ptr(), -1
      rd.q_prescale = dh ** -0.5 if family == "gemma3" else 0.0
      rd.qkv, rd.positions, rd.pos_ld, rd.col_ptr = qkv[b0:].data_ptr(), pos[b0:].data_ptr(), S, colp.data_ptr()
      rd.q_out, rd.kcache, rd.vcache = q[b0:].data_ptr(), kc[b0:].data_ptr(), vc[b0:].data_ptr()
      ops.rope_kvwrite(rd)
    torch.cuda.synchronize()
    return q, kc, vc

  one = run(B)        # 512 rows in one call
  four = run(1)       # 128 rows per call
  for name, x, y in zip(("q", "k cache", "v cache"), one, four):
    diff = (x.float() - y.float()).abs()
    assert torch.equal(x, y), (name, int((diff > 0).sum()), diff.max().item(), torch.nonzero(diff > 0)[:4].tolist())
  assert one[0].float().abs().max() > 0.1 and one[1][:, :, col: col + T].float().abs().max() > 0.5

@pytest.mark.parametrize("family,norm,Hq,Hkv,dh", [("qwen3", "qwen3", 32, 4, 128), ("gemma3", "gemma3", 4, 1, 256), ("llama3", "llama3", 3, 1, 16),
                                                   ("qwen3", "gemma3", 5, 2, 64), ("llama3", "qwen3", 2, 1, 512)])
def test_normed_heads_over_many_rows_equal_the_per_head_kernel(gpu, family, norm, Hq, Hkv, dh):
  """The fewest rows of the row kernel in one call (a head's squares summed over its own lanes) against a quarter per call (over a
  work-group): the fp32 sum runs in another order, so a rounded result may be the neighbouring bf16 value; columns that
  wrap around the cache included."""
  from tunix_amd import _lib as L
  from tunix_amd import ops
  from tunix_amd.model import _NORM, _ROPE, rope_timescale
  B = 4
  T = (384 + 5120 // (Hq + 2 * Hkv) + B - 1) // B
  S, col = T + 4, 9
  qkv = bf(rnd((B, T, (Hq + 2 * Hkv) * dh), 121)).to(gpu)
  pos = torch.randint(0, 2000, (B, col + T), generator=torch.Generator().manual_seed(122), dtype=torch.int32).to(gpu)
  ts = torch.from_numpy(rope_timescale(dh, 1e6)).to(gpu)
  wq, wk = bf(rnd((dh,), 123)).to(gpu), bf(rnd((dh,), 124)).to(gpu)
  colp = torch.tensor([col], dtype=torch.int32, device=gpu)

  def run(rows):
    q = torch.zeros(B, T, Hq * dh, dtype=torch.bfloat16, device=gpu)
    kc = torch.zeros(B, Hkv, S, dh, dtype=torch.bfloat16, device=gpu)
    vc = torch.zeros_like(kc)
    for b0 in range(0, B, rows):
      d = L.RopeDesc()
      d.B, d.T, d.S, d.Hq, d.Hkv, d.dh = rows, T, S, Hq, Hkv, dh
      d.rope_flavor, d.rope_scale, d.timescale = _ROPE[family], 8.0 if family == "gemma3" else 1.0, ts.data_ptr()
      d.qk_norm, d.norm_eps, d.q_norm_w, d.k_norm_w = _NORM[norm], 1e-6, wq.data_ptr(), wk.data_ptr()
      d.q_prescale = 0.25 if family == "gemma3" else 0.0
      d.qkv, d.positions, d.pos_ld, d.col_ptr = qkv[b0:].data_ptr(), pos[b0:].data_ptr(), pos.shape[1], colp.data_ptr()
      d.q_out, d.kcache, d.vcache = q[b0:].data_ptr(), kc[b0:].data_ptr(), vc[b0:].data_ptr()
      ops.rope_kvwrite(d)
    torch.cuda.synchronize()
    return q, kc, vc

  one, four = run(B), run(1)
  # a rotated element is x1 cos - x2 sin of normed elements that may each be one ulp off: ulps of the larger operand
  mag = float(max(one[0].abs().max(), one[1].abs().max()))
  for what, x, y in zip(("q", "k cache"), one, four):
    assert_bf16_close(x, y, min_equal=0.98, what=what, atol=2 * mag * 2.0 ** -7)
  assert torch.equal(one[2], four[2])



@pytest.mark.parametrize("family", ["llama3", "qwen3"])
def test_rope_from_splitk_planes_equals_finish_then_rope(gpu, family):
  """The rope / cache-write kernel fed with the partial planes of a split-k qkv linear against
  the finishing pass followed by the same kernel on its output: bit for bit."""
  from tunix_amd import _lib as L
  from tunix_amd import ops
  from tunix_amd.model import _NORM, _ROPE, rope_timescale
  B, T, S, Hq, Hkv, dh, K, g, split, col = 128, 1, 16, 4, 2, 64, 1024, 64, 4, 7
  N = (Hq + 2 * Hkv) * dh
  x, w = rnd((B, K), 84), rnd((K, N), 85, 0.02)
  c, s = ops.quantize_pack(bf(w).to(gpu), g, Q.NF4)
  gx = bf(x).to(gpu)
  ws = torch.empty(split * B * N, dtype=torch.float32, device=gpu)
  qkv = torch.empty(B, N, dtype=torch.bfloat16, device=gpu)
  ld = ops.make_qlinear_desc(M=B, K=K, N=N, group=g, qtype=Q.NF4, x=gx, codes=c, scales=s, y=qkv,
                             split_k=split, ws=ws)
  ops.qlinear(ld)                                  # planes + finishing pass -> qkv
  pos = torch.randint(0, 900, (B, S), generator=torch.Generator().manual_seed(86), dtype=torch.int32).to(gpu)
  ts = torch.from_numpy(rope_timescale(dh, 1e6)).to(gpu)
  qn, kn = bf(rnd((dh,), 87, 0.3) + 1).to(gpu), bf(rnd((dh,), 88, 0.3) + 1).to(gpu)
  colp = torch.tensor([col], dtype=torch.int32, device=gpu)
  outs = []
  for planes in (False, True):
    d = L.RopeDesc()
    d.B, d.T, d.S, d.Hq, d.Hkv, d.dh = B, T, S, Hq, Hkv, dh
    d.rope_flavor, d.rope_scale, d.timescale = _ROPE[family], 1.0, ts.data_ptr()
    if family != "llama3":
      d.qk_norm, d.norm_eps, d.q_norm_w, d.k_norm_w = _NORM[family], 1e-6, qn.data_ptr(), kn.data_ptr()
    else:
      d.qk_norm = -1
    qo = torch.zeros(B * T, Hq * dh, dtype=torch.bfloat16, device=gpu)
    kc = torch.zeros(B, Hkv, S, dh, dtype=torch.bfloat16, device=gpu)
    vc = torch.zeros_like(kc)
    d.positions, d.pos_ld, d.col_ptr = pos.data_ptr(), S, colp.data_ptr()
    d.q_out, d.kcache, d.vcache = qo.data_ptr(), kc.data_ptr(), vc.data_ptr()
    if planes:
      ops.qlinear(ld, finish=False)
      d.qkv_ws, d.split_k = ws.data_ptr(), split
    else:
      d.qkv = qkv.data_ptr()
    ops.rope_kvwrite(d)
    torch.cuda.synchronize()
    outs.append((qo, kc, vc))
  assert outs[0][0].float().abs().max() > 0
  for a, b in zip(*outs):
    assert torch.equal(a, b)


@pytest.mark.parametrize("M,F,r", [(128, 1024, 64), (200, 192, 32)])
def test_mul_epilogue_fuses_next_adapter_projection(gpu, M, F, r):
  """A gate|up linear with next_tpart: y equals the plain launch bit for bit, and
  tnx_lora_reduce over the planes equals bf16(y . A_next) (what tnx_lora_down gives)."""
  from tunix_amd import _lib as L
  from tunix_amd import ops
  K, g = 512, 64
  x = rnd((M, K), 90)
  wg, wu = rnd((K, F), 91, 0.05), rnd((K, F), 92, 0.05)
  a_next = rnd((F, r), 93, 0.02)
  c, s = ops.quantize_pack(bf(torch.cat([wg, wu], 1)).to(gpu), g, Q.NF4, True)
  gx = bf(x).to(gpu)
  y0 = torch.empty(M, F, dtype=torch.bfloat16, device=gpu)
  y1 = torch.full((M, F), 3.0, dtype=torch.bfloat16, device=gpu)
  base = dict(M=M, K=K, N=2 * F, group=g, qtype=Q.NF4, x=gx, codes=c, scales=s, epilogue=L.TNX_EPI_SILU_MUL)
  ops.qlinear(ops.make_qlinear_desc(y=y0, **base))
  ncb = math.ceil(2 * F / 128)
  tpart = torch.full((math.ceil(M / 128) * ncb * 8192,), float("nan"), dtype=torch.float32, device=gpu)
  a_t = bf(a_next).t().contiguous().to(gpu)
  ops.qlinear(ops.make_qlinear_desc(y=y1, next_a_t=a_t, next_rank=r, next_tpart=tpart, **base))
  t = torch.full((M, r + 16), 5.0, dtype=torch.bfloat16, device=gpu)
  ops.lora_reduce(tpart, M, ncb, r, t)
  torch.cuda.synchronize()
  assert torch.equal(y0, y1)
  want = Q.rb((y1.float().cpu().double() @ a_next.double()).float())
  assert_bf16_close(t[:, :r], want, what="fused next-adapter projection")
  assert (t[:, r:] == 5.0).all()
  t2 = torch.zeros(M, r, dtype=torch.bfloat16, device=gpu)
  ops.lora_down(y1, a_t, t2)
  assert (t[:, :r].float() - t2.float()).abs().max().item() <= 2.0 ** -7 * max(1e-3, t2.float().abs().max().item())


# (the second half of the shapes runs 256-row tiles, the first 128-row ones: what fills the device better)
PRE_SHAPES = [(65, 128, 16), (128, 256, 272), (129, 384, 48), (255, 128, 528), (769, 2048, 16304), (1024, 2048, 16384), (1023, 2176, 16144)]


@pytest.mark.parametrize("M,K,N", PRE_SHAPES)
def test_many_rows_from_the_expanded_copy(gpu, M, K, N):
  """Every form of the tile that qgemm_pre.h stores, at the edges of its row and column tiles, against 64-bit sums: fp32 results
  within the worst case of K roundings, bf16 ones within half an ulp more."""
  from tunix_amd import _lib as L
  from tunix_amd import ops
  g = torch.Generator(device=gpu).manual_seed(M)
  x = torch.randn(M, K, generator=g, device=gpu).bfloat16()
  w = (torch.randn(N, K, generator=g, device=gpu) * K ** -0.5).bfloat16()
  want = x.double() @ w.double().T
  err = K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)

  def run(wt, epilogue, n, dtype):
    y = torch.full((M + 1, n), 7.0, dtype=dtype, device=gpu)
    d = L.DenseDesc()
    d.M, d.K, d.N, d.dtype, d.batch, d.split_k = M, K, N, ops.DTYPES[torch.bfloat16], 1, 1
    d.x, d.ldx, d.w, d.epilogue, d.y, d.ldy = x.data_ptr(), K, ops.dense_expand(wt).data_ptr(), epilogue, y.data_ptr(), n
    ops.dense_linear(d)
    torch.cuda.synchronize()
    assert (y[M] == 7.0).all()      # nothing behind the last row
    return y[:M].double()

  for epilogue, ref, e, dtype in ((L.TNX_EPI_F32, want, err, torch.float32), (L.TNX_EPI_STORE, want, err, torch.bfloat16),
                                  (L.TNX_EPI_RELU2, want.clamp(min=0) ** 2, 2.1 * err * want.abs() + err ** 2, torch.bfloat16)):
    rounding = 0.0 if dtype == torch.float32 else 2.0 ** -8
    assert ((run(w, epilogue, N, dtype) - ref).abs() <= rounding * ref.abs() + e + 1e-30).all(), epilogue
  if N % 32:
    return
  half = N // 2
  paired = w.view(2, N // 32, 16, K).transpose(0, 1).reshape(N, K).contiguous()
  gate, up = want[:, :half], want[:, half:]
  for epilogue, act in ((L.TNX_EPI_SILU_MUL, torch.nn.functional.silu(gate)), (L.TNX_EPI_GELU_MUL, torch.nn.functional.gelu(gate, approximate="tanh"))):
    got = run(paired, epilogue, half, torch.bfloat16)
    assert ((got - act * up).norm() / (act * up).norm()) < 2.0 ** -8, epilogue


@pytest.mark.parametrize("M,K,N,rank,scale,residual", [
    (4000, 256, 1152, 32, 1.0, False),     # 128 columns in the last tile, a ragged last row block
    (3970, 640, 1152, 64, 0.75, True),     # an adapter's scale that is no power of two; two rows in the last block
    (4097, 128, 1040, 64, 0.5, True),      # 16 columns, one row, one k-tile
    (30000, 128, 144, 0, 1.0, False),      # one whole column tile's worth less: 144 = none whole, one of 144
    (33000, 128, 80, 32, 1.0, True),       # no whole tile at all
    (4100, 256, 1168, 32, 1.0, False),     # 144 columns in the last tile: no half
])
def test_last_column_tiles_of_half_the_width(gpu, M, K, N, rank, scale, residual):
  """Calls whose last column tile has at most 128 columns, from the converted copy: the bits of the codes, which go through whole tiles."""
  from tunix_amd import _lib as L
  from tunix_amd import ops
  g = torch.Generator(device=gpu).manual_seed(N + M)
  r = lambda *s: torch.randn(*s, generator=g, device=gpu)
  c, s = ops.quantize_pack((r(K, N) * 0.02).bfloat16(), 64, Q.NF4)
  x = r(M, K).bfloat16()
  kw = {}
  if residual:
    kw["residual"] = r(M, N).bfloat16()
  if rank:
    kw.update(lora_rank=rank, lora_nseg=1, lora_seg_end=[N], lora_seg_toff=[0], t=r(M, rank).bfloat16(), t_ld=rank, lora_b=(r(N, rank) * 0.1).bfloat16(), lora_scale=scale)
  outs = []
  for copy in (ops.qw_expand(c, s, K, N, 64, Q.NF4), None):
    y = torch.full((M + 1, N), 7.0, dtype=torch.bfloat16, device=gpu)
    ops.qlinear(ops.make_qlinear_desc(M=M, K=K, N=N, group=64, qtype=Q.NF4, x=x, codes=c, scales=s, y=y, w_expanded=copy,
                                      epilogue=L.TNX_EPI_RESIDUAL if residual else L.TNX_EPI_STORE, **kw))
    outs.append(y)
  torch.cuda.synchronize()
  assert torch.equal(outs[0][:M].view(torch.int16), outs[1][:M].view(torch.int16)) and bool((outs[0][M] == 7.0).all())


@pytest.mark.parametrize("M", [1000, 1025])
def test_expanded_copy_at_the_line_of_64_row_tiles(gpu, M):
  """256 tiles of 64 rows, one to a compute unit, and 272."""
  test_many_rows_from_the_expanded_copy(gpu, M, 256, 4096)


@pytest.mark.parametrize("K,rank,scale,residual", [(256, 64, 0.75, True), (128, 32, 1.0, False), (384, 0, 1.0, True)])
def test_linears_in_tiles_of_64_rows(gpu, K, rank, scale, residual):
  """A converted copy in tiles of 64 rows (234 of them, the last row block of one row), next to the codes in tiles of 128."""
  test_last_column_tiles_of_half_the_width(gpu, 513, K, 6656, rank, scale, residual)


@pytest.mark.parametrize("M,K,widths", [(600, 256, (3968, 4112, 16)), (1000, 2048, (8176, 4096, 4112))])
@pytest.mark.parametrize("rank", [32, 64])
@pytest.mark.parametrize("scale", [1.0, 0.25, 0.75])
def test_many_rows_adapter(gpu, M, K, widths, rank, scale):
  """The adapter behind the last k of 128- and 256-row tiles: scales that go into B (powers of two) and others, segments that begin
  inside a work-group's columns; against 64-bit sums of the same t."""
  from tunix_amd import ops
  N = sum(widths)
  g = torch.Generator(device=gpu).manual_seed(rank)
  r = lambda *s: torch.randn(*s, generator=g, device=gpu)
  x, w, t, b = r(M, K).bfloat16(), (r(K, N) * 0.02).bfloat16(), r(M, 3 * rank).bfloat16(), (r(N, rank) * 0.1).bfloat16()
  codes, scales = ops.quantize_pack(w, 64, Q.NF4)
  wd = ops.qw_dequant(codes, scales, K, N, 64, Q.NF4).double()
  ends = [int(v) for v in np.cumsum(widths)]
  want, size = x.double() @ wd, x.double().abs() @ wd.abs()
  for i, (a0, a1) in enumerate(zip([0] + ends[:-1], ends)):
    ti, bi = t[:, i * rank:(i + 1) * rank].double(), b[a0:a1].double().T
    want[:, a0:a1] += scale * (ti @ bi)
    size[:, a0:a1] += scale * (ti.abs() @ bi.abs())
  got = []
  for copy in (ops.qw_expand(codes, scales, K, N, 64, Q.NF4), None):
    y = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=gpu)
    ops.qlinear(ops.make_qlinear_desc(M=M, K=K, N=N, group=64, qtype=Q.NF4, x=x, codes=codes, scales=scales, y=y, lora_rank=rank, lora_nseg=3,
                                      lora_seg_end=ends, lora_seg_toff=[0, rank, 2 * rank], t=t, t_ld=3 * rank, lora_b=b, lora_scale=scale,
                                      w_expanded=copy))
    assert ((y.double() - want).abs() <= 2.0 ** -8 * want.abs() + (K + rank) * 2.0 ** -24 * size).all()
    got.append(y)
  assert torch.equal(got[0], got[1])   # from the copy and from the codes: the same sums


@pytest.mark.parametrize("K,N,counts", [(128, 272, (70, 0, 129, 40)), (4096, 272, (1300, 1255)), (4096, 3344, (1300, 1255)), (128, 528, (2200, 0, 1030, 8))])
def test_many_rows_experts_from_expanded_copies(gpu, K, N, counts):
  """Row blocks of 128 and (4096 -> 3344) of 256 routes: experts without rows, blocks that end inside a tile, experts of several groups of
  1024 rows."""
  from tunix_amd import _lib as L
  from tunix_amd import ops
  E, n = len(counts), sum(counts)
  g = torch.Generator(device=gpu).manual_seed(n)
  x = torch.randn(n, K, generator=g, device=gpu).bfloat16()
  w = (torch.randn(E, N, K, generator=g, device=gpu) * K ** -0.5).bfloat16()
  bank = torch.stack([ops.dense_expand(e) for e in w])
  route = torch.randperm(n, generator=torch.Generator().manual_seed(1)).to(torch.int32).to(gpu)
  offsets = torch.tensor([0] + [int(v) for v in np.cumsum(counts)], dtype=torch.int32, device=gpu)
  y = torch.full((n, N), float("nan"), dtype=torch.bfloat16, device=gpu)
  d = L.DenseDesc()
  d.M, d.K, d.N, d.dtype, d.batch, d.split_k = n, K, N, ops.DTYPES[torch.bfloat16], 1, 1
  d.x, d.ldx, d.w, d.w_stride, d.epilogue, d.y, d.ldy = x.data_ptr(), K, bank.data_ptr(), bank[0].numel(), L.TNX_EPI_STORE, y.data_ptr(), N
  d.n_experts, d.x_div, d.offsets, d.sorted_route = E, 1, offsets.data_ptr(), route.data_ptr()
  ops.dense_linear(d)
  for e, (a0, a1) in enumerate(zip(offsets.tolist()[:-1], offsets.tolist()[1:])):
    xe, we = x[route[a0:a1].long()].double(), w[e].double()
    want = xe @ we.T
    assert ((y[route[a0:a1].long()].double() - want).abs() <= 2.0 ** -8 * want.abs() + K * 2.0 ** -24 * (xe.abs() @ we.abs().T)).all()


def merged_and_apart(gpu, dh, Hkv, G, M, S, chunk, window, qtype, group, cache=None, positive=False):
  """(y, planes) of gqa_attn and the linear with its adapter inside, then of gqa_attn_parts and the linear that merges its chunks; cache(k, v, column): changes to
  the caches; positive: no weight below zero, so that an infinite value stays one."""
  from tunix_amd import _lib as L
  from tunix_amd import ops
  bf = torch.bfloat16
  g = torch.Generator(device=gpu).manual_seed(dh + M)
  K, N, rank = Hkv * G * dh, 272, 32
  r = lambda *s: torch.randn(*s, generator=g, device=gpu)
  w_of = lambda t: t.abs() + t.abs().mean() if positive else t
  col = S - 3
  tokens = torch.ones(M, S, dtype=torch.int32, device=gpu)
  for b in range(M):
    tokens[b, :(b * 37) % (col + 1)] = 0
  q, kc, vc = r(M, Hkv * G, dh).to(bf), r(M, Hkv, S, dh).to(bf), r(M, Hkv, S, dh).to(bf)
  if cache is not None:
    cache(kc, vc, col)
  n_chunks = -(-S // chunk)
  ws = torch.full((ops.attn_ws_bytes(M, 1, S, Hkv * G, dh, chunk) // 4,), float("nan"), device=gpu)
  out = torch.empty(M, K, dtype=bf, device=gpu)
  ad = L.AttnDesc()
  ad.B, ad.T, ad.S, ad.Hq, ad.Hkv, ad.dh = M, 1, S, Hkv * G, Hkv, dh
  ad.scale, ad.window, ad.pad_id, ad.kv_chunk = dh ** -0.5, window, 0, chunk
  at = torch.tensor([col], dtype=torch.int32, device=gpu)
  ad.q, ad.kcache, ad.vcache, ad.tokens, ad.tok_ld, ad.col_ptr = q.data_ptr(), kc.data_ptr(), vc.data_ptr(), tokens.data_ptr(), S, at.data_ptr()
  ad.ws, ad.out = ws.data_ptr(), out.data_ptr()
  split = {4096: 8, 768: 2}.get(K, K // 128)
  codes, scales = ops.quantize_pack(w_of(r(K, N) * 0.05).to(bf), group, qtype)
  a_t, b = w_of(r(rank, K) * K ** -0.5).to(bf), w_of(r(N, rank) * 0.3).to(bf)
  frag = ops.lora_frag(a_t)
  assert ops.qlinear_merged_ok(M, K, N, rank, split, dh, n_chunks)
  got = []
  for merged in (False, True):
    y = torch.full((M, N), float("nan"), dtype=bf, device=gpu)
    planes = torch.full((split, M, N), float("nan"), device=gpu)
    d = ops.make_qlinear_desc(M=M, K=K, N=N, group=group, qtype=qtype, x=out, codes=codes, scales=scales, y=y, lora_rank=rank, lora_nseg=1,
                              lora_seg_end=[N], lora_seg_toff=[0], lora_b=b, lora_scale=0.5, split_k=split, ws=planes)
    ws.fill_(float("nan"))
    if merged:   # (x is not read)
      out.fill_(float("nan"))
      ops.gqa_attn_parts(None, ad)
      ops.qlinear(d, a_frag=frag, parts=(ws, dh, n_chunks))
    else:
      ops.gqa_attn(ad)
      ops.qlinear(d, a_frag=frag)
    got += [y, planes]
  return got


@pytest.mark.parametrize("dh,Hkv,G,M,S,chunk,window,qtype,group", [
    (128, 8, 4, 1, 160, 32, 0, Q.NF4, 64),       # 5 chunks, 32 k-tiles in 8 splits of 4
    (128, 8, 4, 3, 384, 32, 100, Q.NF4, 64),     # 12, some before the window
    (128, 8, 4, 8, 128, 32, 0, Q.INT4, 32),      # 4
    (128, 8, 4, 9, 96, 64, 0, Q.INT4, 128),      # 2, rows of the next tile
    (128, 8, 4, 16, 64, 32, 20, Q.NF4, 32),
    (64, 2, 4, 33, 96, 32, 0, Q.INT4, 64),       # two heads a k-tile
    (64, 2, 4, 64, 64, 32, 40, Q.INT4, 64),
    (256, 1, 4, 17, 288, 96, 0, Q.INT4, 128),    # half a head a k-tile
    (256, 1, 4, 40, 64, 32, 0, Q.NF4, 64),
    (256, 1, 3, 2, 200, 32, 33, Q.INT4, 128),    # 6 k-tiles, three a split
])
def test_linear_that_merges_key_chunks(gpu, dh, Hkv, G, M, S, chunk, window, qtype, group):
  """gqa_attn_parts and a linear that merges its chunks against gqa_attn and the linear with its adapter inside, bit for bit: chunks without a key (padding in
  front, a window), whose outputs nobody writes, included."""
  got = merged_and_apart(gpu, dh, Hkv, G, M, S, chunk, window, qtype, group)
  assert got[0].isfinite().all()
  assert torch.equal(got[0], got[2]) and torch.equal(got[1], got[3])


@pytest.mark.parametrize("dh,Hkv,G,M,S,chunk,qtype,group", [
    (128, 8, 4, 3, 384, 32, Q.NF4, 64),       # 12 chunks, all of them at once
    (128, 8, 4, 9, 96, 64, Q.INT4, 128),      # 2, two pieces of a row at once
    (64, 2, 4, 33, 96, 32, Q.INT4, 64),
    (256, 1, 4, 17, 288, 96, Q.INT4, 128),
])
def test_linear_that_merges_key_chunks_keeps_infinities(gpu, dh, Hkv, G, M, S, chunk, qtype, group):
  """An infinite value in the cache (row 0), sums that overflow (row 1) and a key of NaN (row 2, by way of its maximum and sum) reach the output as they do through
  the pass that merges; no other row sees them."""
  def cache(kc, vc, col):
    vc[0, 0, col, 5] = float("inf")
    kc[1, -1], vc[1, -1, :, 7] = 0.0, 3.38e38
    kc[2, 0, col] = float("nan")

  y, planes, y_m, planes_m = merged_and_apart(gpu, dh, Hkv, G, M, S, chunk, 0, qtype, group, cache, positive=True)
  assert (y[:2] == float("inf")).all() and y[2].isnan().all() and y[3:].isfinite().all()
  same = lambda u, v: torch.testing.assert_close(u, v, rtol=0, atol=0, equal_nan=True)
  same(y_m, y)
  same(planes_m, planes)


@pytest.mark.parametrize("K,split,epilogue", [(128, 1, "TNX_EPI_STORE"), (512, 1, "TNX_EPI_RESIDUAL"), (512, 1, "TNX_EPI_F32"), (512, 4, "TNX_EPI_STORE")])
def test_linear_that_merges_key_chunks_beside_its_output(gpu, K, split, epilogue):
  """Partials that begin where the output ends, or end where it begins, give what they give anywhere else; an output that reaches into them raises."""
  from tunix_amd import _lib as L
  from tunix_amd import ops
  bf, M, N, dh, n_chunks, rank = torch.bfloat16, 4, 272, 128, 3, 32
  g = torch.Generator(device=gpu).manual_seed(K + split)
  r = lambda *s: torch.randn(*s, generator=g, device=gpu)
  parts = r(M, K // dh, n_chunks, dh + 4)
  parts[..., 1] = parts[..., 1].abs() + 1.0
  codes, scales = ops.quantize_pack((r(K, N) * 0.05).to(bf), 64, L.TNX_Q_INT4)
  frag, b, x = ops.lora_frag((r(rank, K) * K ** -0.5).to(bf)), (r(N, rank) * 0.3).to(bf), r(M, N).to(bf)
  wide = split > 1 or epilogue == "TNX_EPI_F32"
  out_bytes, part_bytes = split * M * N * (4 if wide else 2), parts.numel() * 4
  got = []
  for o0, p0, free in ((0, out_bytes, True), (part_bytes, 0, True), (part_bytes + 4096, 0, True), (part_bytes - 16, 0, False), (0, out_bytes - 16, False)):
    room = torch.zeros(part_bytes + out_bytes + 4096, dtype=torch.uint8, device=gpu)
    room[p0:p0 + part_bytes] = parts.view(torch.uint8).flatten()
    out = room[o0:o0 + out_bytes].view(torch.float32 if wide else bf)
    y = torch.empty(M, N, dtype=bf, device=gpu) if split > 1 else out
    d = ops.make_qlinear_desc(M=M, K=K, N=N, group=64, qtype=L.TNX_Q_INT4, x=x, codes=codes, scales=scales, y=y, epilogue=getattr(L, epilogue), residual=x, lora_rank=rank,
                              lora_nseg=1, lora_seg_end=[N], lora_seg_toff=[0], lora_b=b, lora_scale=0.5, split_k=split, ws=out if split > 1 else None)
    run = lambda: ops.qlinear(d, finish=False, a_frag=frag, parts=(room[p0:], dh, n_chunks))
    if free:
      run()
      got.append(out.clone())
      assert torch.equal(room[p0:p0 + part_bytes], parts.view(torch.uint8).flatten())
    else:
      with pytest.raises(ValueError, match="in the partials"):
        run()
  assert got[0].isfinite().all() and got[0].any() and all(torch.equal(got[0], v) for v in got[1:])


def test_linear_that_merges_key_chunks_refuses(gpu):
  """More rows, chunks or bytes than it takes."""
  from tunix_amd import ops
  ok = ops.qlinear_merged_ok
  assert ok(16, 4096, 4096, 64, 8, 128, 2) and not ok(32, 4096, 4096, 64, 8, 128, 2)      # bytes
  assert ok(1, 4096, 4096, 64, 8, 128, 12) and not ok(1, 4096, 4096, 64, 8, 128, 13)      # chunks
  assert not ok(1, 4096, 4096, 64, 4, 128, 2)        # eight k-tiles a split
  assert not ok(1, 4096, 4096, 48, 8, 128, 2) and not ok(1, 4096, 4096, 64, 8, 96, 2) and not ok(65, 1024, 1024, 32, 8, 256, 2)


@pytest.mark.parametrize("dh,Hkv,G,T,B,window,family,split", [
    (64, 2, 4, 5, 3, 0, "qwen3", 4),        # fewer positions than a tile pair; planes
    (64, 2, 4, 64, 4, 0, "qwen3", 1),       # two tiles a wave, prompts that begin inside a tile of the one before's last rows
    (64, 1, 3, 131, 3, 20, "qwen3", 1),
    (128, 2, 4, 3, 5, 0, "llama3", 2),
    (128, 2, 4, 200, 3, 0, "llama3", 1),    # work-groups of 32 positions
    (128, 1, 16, 97, 4, 33, "llama3", 1),
    (256, 1, 4, 70, 5, 16, "gemma3", 1),
    (256, 1, 4, 300, 2, 0, "gemma3", 1),
])
def test_prompts_without_their_padding(gpu, dh, Hkv, G, T, B, window, family, split):
  """Embedding, rotation with the cache write and attention of packed prompts against the padded ones, bit for bit in every row that is there; nothing else is
  written: prompts of all columns, of one, and such as begin at and around the edges of tiles."""
  from tunix_amd import _lib as L
  from tunix_amd import ops
  from tunix_amd.model import _NORM, _ROPE
  bf = torch.bfloat16
  g = torch.Generator(device=gpu).manual_seed(T)
  r = lambda *s: torch.randn(*s, generator=g, device=gpu)
  Hq, S, V = Hkv * G, T + 7, 50
  first = [0, T - 1, min(8, T - 2), min(33, T - 2), min(16, T - 1)][:B]
  lengths = [T - f for f in first]
  base = [sum(lengths[:b]) - first[b] for b in range(B)]
  M, W = sum(lengths), (Hq + 2 * Hkv) * dh
  at = torch.tensor([b * T + t for b in range(B) for t in range(first[b], T)], device=gpu)
  i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=gpu)
  starts, row_base, zero = i32(first), i32(base), i32([0])
  packed = ops.packed_rows(row_base, starts, M)
  ids = torch.randint(1, V, (B, S), generator=g, device=gpu, dtype=torch.int32)
  for b, f in enumerate(first):
    ids[b, :f] = 0
  positions = (torch.arange(S, device=gpu, dtype=torch.int32)[None] - starts[:, None]).clamp(min=0).contiguous()
  nan = lambda *s: torch.full(s, float("nan"), dtype=bf, device=gpu)
  table = r(V, 96).to(bf)
  e0, e1 = nan(B * T, 96), nan(M, 96)
  ops.embed(table, ids, zero, B, T, 1.5, e0)
  ops.embed(table, ids, zero, B, T, 1.5, e1, packed)
  assert torch.equal(e0[at], e1)
  src = r(split, B * T, W) * 0.5
  full, part = src.contiguous(), src[:, at].contiguous()
  wq, wk = r(dh).to(bf), r(dh).to(bf)
  scale = 0.0 if family == "gemma3" else dh ** -0.5
  ts = (10000.0 ** (torch.arange(dh // 2, device=gpu, dtype=torch.float32) * 2 / dh)).contiguous()
  got = []
  for rows, x, p in ((B * T, full, None), (M, part, packed)):
    q, out = nan(rows, Hq * dh), nan(rows, Hq * dh)
    kc, vc = torch.zeros(B, Hkv, S, dh, dtype=bf, device=gpu), torch.zeros(B, Hkv, S, dh, dtype=bf, device=gpu)
    y = x[0].to(bf).contiguous()
    rd = L.RopeDesc()
    rd.B, rd.T, rd.S, rd.Hq, rd.Hkv, rd.dh = B, T, S, Hq, Hkv, dh
    rd.rope_flavor, rd.rope_scale, rd.timescale = _ROPE[family], 1.0, ts.data_ptr()
    rd.qk_norm, rd.norm_eps, rd.q_norm_w, rd.k_norm_w = (-1 if family == "llama3" else _NORM[family]), 1e-6, wq.data_ptr(), wk.data_ptr()
    rd.q_prescale = dh ** -0.5 if family == "gemma3" else 0.0
    rd.qkv, rd.positions, rd.pos_ld, rd.col_ptr = y.data_ptr(), positions.data_ptr(), S, zero.data_ptr()
    if split > 1:
      rd.qkv_ws, rd.split_k = x.data_ptr(), split
    rd.q_out, rd.kcache, rd.vcache = q.data_ptr(), kc.data_ptr(), vc.data_ptr()
    ops.rope_kvwrite(rd, p)
    ad = L.AttnDesc()
    ad.B, ad.T, ad.S, ad.Hq, ad.Hkv, ad.dh, ad.scale, ad.window, ad.pad_id = B, T, S, Hq, Hkv, dh, scale, window, 0
    ad.q, ad.kcache, ad.vcache, ad.tokens, ad.tok_ld, ad.col_ptr, ad.out = (q.data_ptr(), kc.data_ptr(), vc.data_ptr(), ids.data_ptr(), S, zero.data_ptr(),
                                                                            out.data_ptr())
    ops.gqa_attn(ad, p)
    got.append((q, out, kc, vc))
  (q0, o0, k0, v0), (q1, o1, k1, v1) = got
  assert torch.equal(q0[at], q1) and o1.isfinite().all() and torch.equal(o0[at], o1)
  for b, f in enumerate(first):
    assert torch.equal(k0[b, :, f:], k1[b, :, f:]) and torch.equal(v0[b, :, f:], v1[b, :, f:])
    assert not k1[b, :, :f].any() and not v1[b, :, :f].any()


@pytest.mark.parametrize("E,x_div", [(1, 3), (64, 1), (65, 2), (256, 1), (257, 3), (520, 4)])
def test_many_rows_experts_are_found_among_any_number(gpu, E, x_div):
  """The search for a tile's expert, 256 of them at a time, and the rows of routes for divisors that are and are no powers of two: most experts
  without a row, some with several blocks, the first and the last with some."""
  from tunix_amd import _lib as L
  from tunix_amd import ops
  K, N = 128, 256
  rng = np.random.default_rng(E)
  counts = np.where(rng.random(E) < 0.6, 0, rng.integers(1, 300, size=E))
  counts[0], counts[-1] = 130, 257
  counts[0] += -int(counts.sum()) % x_div
  n = int(counts.sum())
  g = torch.Generator(device=gpu).manual_seed(n)
  x = torch.randn(n // x_div, K, generator=g, device=gpu).bfloat16()
  w = (torch.randn(E, N, K, generator=g, device=gpu) * K ** -0.5).bfloat16()
  bank = torch.stack([ops.dense_expand(e) for e in w])
  route = torch.randperm(n, generator=torch.Generator().manual_seed(2)).to(torch.int32).to(gpu)
  offsets = torch.tensor([0] + [int(v) for v in np.cumsum(counts)], dtype=torch.int32, device=gpu)
  y = torch.full((n, N), float("nan"), dtype=torch.bfloat16, device=gpu)
  d = L.DenseDesc()
  d.M, d.K, d.N, d.dtype, d.batch, d.split_k = n, K, N, ops.DTYPES[torch.bfloat16], 1, 1
  d.x, d.ldx, d.w, d.w_stride, d.epilogue, d.y, d.ldy = x.data_ptr(), K, bank.data_ptr(), bank[0].numel(), L.TNX_EPI_STORE, y.data_ptr(), N
  d.n_experts, d.x_div, d.offsets, d.sorted_route = E, x_div, offsets.data_ptr(), route.data_ptr()
  ops.dense_linear(d)
  for e, (a0, a1) in enumerate(zip(offsets.tolist()[:-1], offsets.tolist()[1:])):
    at = route[a0:a1].long()
    xe, we = x[at // x_div].double(), w[e].double()
    want = xe @ we.T
    assert ((y[at].double() - want).abs() <= 2.0 ** -8 * want.abs() + K * 2.0 ** -24 * (xe.abs() @ we.abs().T)).all()


@pytest.mark.parametrize("M,counts_scale,K,N", [(36, 1, 256, 512), (320, 1, 256, 512), (333, 2, 256, 512), (2601, 1, 4096, 2048)])
@pytest.mark.parametrize("qtype", [Q.INT4, Q.NF4])
def test_moe_from_the_experts_copies(gpu, M, counts_scale, K, N, qtype):
  """Experts read from their converted copies give the bits that they give from the codes, on both sides of the line between
  the two, with experts of very different sizes, in tiles of 128 and (2601 rows) of 256 rows."""
  from tunix_amd import _lib as L
  from tunix_amd import ops
  E, k, group = 4, 2, 64
  g = torch.Generator(device=gpu).manual_seed(M)
  w = (torch.randn(E, K, N, generator=g, device=gpu) * 0.05).bfloat16()
  packed = [ops.quantize_pack(e, group, qtype, True) for e in w]
  codes, scales = (torch.cat([p[i] for p in packed]) for i in (0, 1))
  bank = ops.qw_expand_bank(codes, scales, E, K, N, group, qtype)
  assert torch.equal(bank[2], ops.qw_expand(*packed[2], K, N, group, qtype))
  ids = torch.stack([(torch.arange(M, device=gpu) // counts_scale) % 3, torch.full((M,), 3, device=gpu)], 1).to(torch.int32)
  counts, offsets = torch.empty(E, dtype=torch.int32, device=gpu), torch.empty(E + 1, dtype=torch.int32, device=gpu)
  route = torch.empty(M * k, dtype=torch.int32, device=gpu)
  ops.moe_sort_routes(ids, E, counts, offsets, route)
  x = torch.randn(M, K, generator=g, device=gpu).bfloat16()
  got = []
  for copies in (None, bank):
    y = torch.full((M * k, N // 2), float("nan"), dtype=torch.bfloat16, device=gpu)
    d = L.MoeGmmDesc()
    d.n_routes, d.E, d.k, d.K, d.N, d.group, d.qtype, d.x, d.x_div = M * k, E, k, K, N, group, qtype, x.data_ptr(), k
    d.codes, d.scales, d.offsets, d.sorted_route = codes.data_ptr(), scales.data_ptr(), offsets.data_ptr(), route.data_ptr()
    d.epilogue, d.y = L.TNX_EPI_SILU_MUL, y.data_ptr()
    ops.moe_gmm(d, copies)
    got.append(y)
  assert got[0].isfinite().all() and torch.equal(got[0], got[1])


@pytest.mark.parametrize("qtype,K,N,rows", [(Q.INT4, 1024, 256, 144), (Q.INT4, 2048, 256, 176), (Q.INT4, 4096, 256, 304), (Q.INT4, 8320, 256, 0),
                                            (Q.NF4, 1152, 512, 144), (Q.NF4, 4096, 256, 176), (Q.NF4, 8320, 256, 242), (Q.NF4, 1024, 384, 0)])
def test_experts_copies_are_read_from_the_rows_on_that_pay(gpu, qtype, K, N, rows):
  """Copies that hold NaN show which calls read them: those with tnx_moe_expanded_rows rows per expert or more, and none where it
  says 0 (a contraction too long for int4, a width the many-row kernel does not take)."""
  from tunix_amd import _lib as L
  from tunix_amd import ops
  assert L.lib().tnx_moe_expanded_rows(K, N, qtype) == rows
  E, group = 2, 64
  g = torch.Generator(device=gpu).manual_seed(K)
  packed = ops.quantize_pack((torch.randn(K, N, generator=g, device=gpu) * 0.05).bfloat16(), group, qtype)
  codes, scales = (torch.cat([p, p]) for p in packed)
  bank = torch.full((E, L.lib().tnx_qw_expanded_bytes(K, N) // 2), float("nan"), dtype=torch.bfloat16, device=gpu)
  for avg in ((rows - 1, rows) if rows else (1024,)):
    n = E * avg
    x = torch.randn(n, K, generator=g, device=gpu).bfloat16()
    offsets = torch.tensor([0, avg, n], dtype=torch.int32, device=gpu)
    route = torch.arange(n, dtype=torch.int32, device=gpu)
    y = torch.zeros(n, N, dtype=torch.bfloat16, device=gpu)
    d = L.MoeGmmDesc()
    d.n_routes, d.E, d.k, d.K, d.N, d.group, d.qtype, d.x, d.x_div = n, E, 1, K, N, group, qtype, x.data_ptr(), 1
    d.codes, d.scales, d.offsets, d.sorted_route = codes.data_ptr(), scales.data_ptr(), offsets.data_ptr(), route.data_ptr()
    d.epilogue, d.y = L.TNX_EPI_STORE, y.data_ptr()
    ops.moe_gmm(d, bank)
    assert bool(torch.isnan(y).all()) == (avg == rows) and bool(torch.isnan(y).any()) == (avg == rows), avg


@pytest.mark.parametrize("D,F,wanted", [(384, 256, (True, False)), (384, 384, (True, False)), (128, 384, (True, False)), (256, 256, (True, True))])
def test_expert_bank_copies_what_calls_read(gpu, D, F, wanted):
  """A bank copies, counts and refreshes the weights whose copy some call reads, and no others."""
  import types

  from tunix_amd import ops
  from tunix_amd.model import ExpertBank
  cfg = types.SimpleNamespace(group=64, qtype=Q.INT4, int4_bound=7.0)
  E = 3

  def weights(seed):
    return {"p.e_gate": rnd((E, D, F), seed), "p.e_up": rnd((E, D, F), seed + 1), "p.e_down": rnd((E, F, D), seed + 2),
            "p.router": rnd((D, E), seed + 3)}
  bank = ExpertBank(cfg, weights(1), "p.", gpu)
  assert bank.wants_expansion() == wanted
  bank.expand()
  for seed in (1, 11):
    if seed > 1:
      bank.load_base(weights(seed))
    for copy, want, codes, scales, K, N in ((bank.gu_expanded, wanted[0], bank.gu_codes, bank.gu_scales, D, 2 * F),
                                            (bank.dn_expanded, wanted[1], bank.dn_codes, bank.dn_scales, F, D)):
      assert (copy is not None) == want
      if want:
        assert torch.equal(copy, ops.qw_expand_bank(codes, scales, E, K, N, 64, Q.INT4))
  assert bank.expanded_bytes() == 2 * sum(c.numel() for c in (bank.gu_expanded, bank.dn_expanded) if c is not None)


@pytest.mark.parametrize("epi", ["silu", "gelu", "residual"])
@pytest.mark.parametrize("scale", [0.5, 0.75])
def test_many_rows_gated_and_residual_in_tiles_of_256_rows(gpu, epi, scale):
  """Gated products of rounded halves with their two adapters, and sums with a residual, at the height of tiles that large passes take:
  against 64-bit sums, and codes against the copy bit for bit."""
  from tunix_amd import _lib as L
  from tunix_amd import ops
  M, K, N, rank, mul = 1023, 2048, 8480, 64, epi != "residual"
  g = torch.Generator(device=gpu).manual_seed(7)
  r = lambda *shape: torch.randn(*shape, generator=g, device=gpu)
  x, w, t, b = r(M, K).bfloat16(), (r(K, N) * 0.02).bfloat16(), r(M, 2 * rank).bfloat16(), (r(N, rank) * 0.1).bfloat16()
  res = r(M, N).bfloat16()
  plain = ops.quantize_pack(w, 64, Q.NF4)
  codes, scales = ops.quantize_pack(w, 64, Q.NF4, mul)
  lin = x.double() @ ops.qw_dequant(*plain, K, N, 64, Q.NF4).double()
  if mul:
    for i in range(2):
      lin[:, i * N // 2:(i + 1) * N // 2] += scale * (t[:, i * rank:(i + 1) * rank].double() @ b[i * N // 2:(i + 1) * N // 2].double().T)
    gate, up = (lin[:, i * N // 2:(i + 1) * N // 2].bfloat16().float() for i in range(2))
    act = (gate * torch.sigmoid(gate.double()).bfloat16().float()) if epi == "silu" else torch.nn.functional.gelu(gate.double(), approximate="tanh")
    # a gate or an up one ulp off moves the product by at most 1.13 (the slope of either activation) times that ulp of |gate up|
    want, mag = (act.bfloat16().float() * up).bfloat16(), (gate * up).abs()
    packed = torch.empty_like(b)
    packed[torch.from_numpy(Q.packed_col(np.arange(N), N, True)).to(gpu)] = b
    kw = dict(lora_nseg=-1, lora_seg_end=[N // 2, N], lora_seg_toff=[0, rank], lora_b=packed, epilogue=L.TNX_EPI_SILU_MUL if epi == "silu" else L.TNX_EPI_GELU_MUL)
  else:
    lin += scale * (t[:, :rank].double() @ b.double().T)
    want, mag = (lin.bfloat16().float() + res.float()).bfloat16(), torch.maximum(lin.abs().float(), res.float().abs())
    kw = dict(lora_nseg=1, lora_seg_end=[N], lora_seg_toff=[0], lora_b=b, residual=res, epilogue=L.TNX_EPI_RESIDUAL)
  got = []
  for copy in (ops.qw_expand(codes, scales, K, N, 64, Q.NF4), None):
    y = torch.full((M, N // 2 if mul else N), float("nan"), dtype=torch.bfloat16, device=gpu)
    ops.qlinear(ops.make_qlinear_desc(M=M, K=K, N=N, group=64, qtype=Q.NF4, x=x, codes=codes, scales=scales, y=y, lora_rank=rank, t=t, t_ld=2 * rank,
                                      lora_scale=scale, w_expanded=copy, **kw))
    got.append(y)
  assert torch.equal(got[0], got[1])
  assert_bf16_close(got[0], want, atol=1e-5, min_equal=0.9 if mul else 0.97, what=epi, mag=mag, ulps=3 if mul else 2)


@pytest.mark.parametrize("B,T,S,Hq,Hkv,col,window,seg,scale", [
    (2, 61, 61, 4, 1, 0, 0, False, 1.0),          # fewest tiles of the work-group form
    (3, 131, 333, 6, 2, 77, 0, False, 0.0),       # three query heads in lanes of four, queries from column 77, odd slots, no scaling
    (1, 259, 263, 4, 1, 3, 40, False, 0.0),       # a window inside two key blocks
    (2, 150, 150, 2, 2, 0, 0, True, 0.0625),      # a packed batch of several segments, one head per kv head
    (1, 45, 70, 16, 1, 5, 0, True, 0.0),           # sixteen heads per kv head: one position per tile
])
def test_gqa_attention_head_dim_256_many_positions(gpu, B, T, S, Hq, Hkv, col, window, seg, scale):
  """Keys and values of 256 dimensions through LDS: bit for bit what calls of a few positions give (every wave loads its own), and
  attention in 64 bits with the probabilities' bf16 rounding as the bound."""
  from tunix_amd import _lib as L
  from tunix_amd import ops
  dh, pad = 256, 0
  g = torch.Generator().manual_seed(190 + T)
  ids = torch.randint(1, 4 if seg else 100, (B, S), generator=g, dtype=torch.int32)
  ids = torch.sort(ids, dim=1).values if seg else ids
  if not seg:
    ids[0, :5] = pad
    ids[B - 1, 9] = pad
  q = bf(rnd((B, T, Hq * dh), 191) * dh ** -0.5).to(gpu)
  kc, vc = bf(rnd((B, Hkv, S, dh), 192)).to(gpu), bf(rnd((B, Hkv, S, dh), 193)).to(gpu)
  gids = ids.to(gpu).contiguous()

  def attn(t0, n):
    qs = q[:, t0:t0 + n].contiguous()
    out = torch.full((B, n, Hq * dh), 7.0, dtype=torch.bfloat16, device=gpu)
    colp = torch.tensor([col + t0], dtype=torch.int32, device=gpu)
    d = L.AttnDesc()
    d.B, d.T, d.S, d.Hq, d.Hkv, d.dh = B, n, S, Hq, Hkv, dh
    d.scale, d.window, d.pad_id = scale, window, pad
    d.q, d.kcache, d.vcache, d.out = qs.data_ptr(), kc.data_ptr(), vc.data_ptr(), out.data_ptr()
    if seg:
      d.segment_ids = gids.data_ptr()
    else:
      d.tokens = gids.data_ptr()
    d.tok_ld, d.col_ptr, d.kv_chunk = S, colp.data_ptr(), 0
    ops.gqa_attn(d)
    torch.cuda.synchronize()
    return out

  whole = attn(0, T)
  few = 3 * max(1, 16 // (1 << (Hq // Hkv - 1).bit_length()))       # three tiles of queries
  parts = torch.cat([attn(t0, min(few, T - t0)) for t0 in range(0, T, few)], dim=1)
  assert torch.equal(whole.view(torch.int16), parts.view(torch.int16))
  at, key = torch.arange(T)[:, None] + col, torch.arange(S)[None]
  mask = ((key <= at) & (at - key < window) if window else key <= at)[None] & \
      (ids[:, None, :] == ids[:, col:col + T, None] if seg else ids[:, None, :] != pad)
  valid = mask.any(-1) & (ids[:, col:col + T] != pad)
  heads = lambda x: x.cpu().repeat_interleave(Hq // Hkv, 1).double()
  score = q.cpu().view(B, T, Hq, dh).permute(0, 2, 1, 3).double() @ heads(kc).transpose(2, 3) * (scale or 1.0)
  ref = (torch.softmax(score.masked_fill(~mask[:, None], -1e30), -1) @ heads(vc)).permute(0, 2, 1, 3).reshape(B, T, -1).float()
  diff = (whole.float().cpu() - ref).abs()[valid]
  assert valid.float().mean() > 0.9 and diff.max().item() <= 2.0 ** -6 * max(1.0, ref[valid].abs().max().item()), diff.max().item()


@pytest.mark.parametrize("S,Hq,Hkv,dh,chunk,window", [
    (70, 8, 2, 128, 0, 0),        # three blocks for four waves; rows of ids read one by one
    (300, 16, 1, 128, 128, 0),    # sixteen heads on one, chunks of a block per wave, the last ones empty for most columns
    (300, 6, 2, 64, 0, 100),      # head_dim 64, three heads in lanes of four, a window over four or five blocks
    (1300, 4, 1, 128, 672, 0),    # odd and even block counts
    (300, 4, 1, 256, 128, 0),     # head_dim 256
    (200, 2, 2, 256, 0, 150),
])
@pytest.mark.parametrize("packed", [False, True])
def test_decode_attention_of_several_waves_per_chunk(gpu, S, Hq, Hkv, dh, chunk, window, packed):
  """One query position whose key blocks are shared among the waves of a work-group, at columns on both sides of every share, against
  attention in 64 bits (probabilities rounded to bf16: 2^-8 of values below 4)."""
  from tunix_amd import _lib as L
  from tunix_amd import ops
  B, pad = 3, 0
  g = torch.Generator().manual_seed(300 + S)
  ids = torch.sort(torch.randint(1, 4, (B, S), generator=g, dtype=torch.int32), 1).values if packed else \
      torch.randint(1, 100, (B, S), generator=g, dtype=torch.int32)
  if not packed:
    ids[0, :40] = pad
    ids[1, 7] = pad
  q = bf(rnd((B, Hq * dh), 301)).to(gpu)
  kc, vc = bf(rnd((B, Hkv, S, dh), 302)), bf(rnd((B, Hkv, S, dh), 303))
  gids = ids.to(gpu).contiguous()
  heads = lambda x: x.double().repeat_interleave(Hq // Hkv, 1)
  for col in sorted({min(c, S - 1) for c in (0, 31, 32, 63, 64, 95, 127, 128, 129, 160, 255, 256, 299, 671, 672, 703, 1299)}):
    kg, vg = kc.clone(), vc.clone()
    kg[:, :, col + 1:], vg[:, :, col + 1:] = 1e4, 1e4          # slots not written yet
    kg, vg = kg.to(gpu), vg.to(gpu)
    out = torch.full((B, Hq * dh), 7.0, dtype=torch.bfloat16, device=gpu)
    ws = torch.empty(max(ops.attn_ws_bytes(B, 1, S, Hq, dh, chunk) // 4, 1), dtype=torch.float32, device=gpu)
    colp = torch.tensor([col], dtype=torch.int32, device=gpu)
    d = L.AttnDesc()
    d.B, d.T, d.S, d.Hq, d.Hkv, d.dh = B, 1, S, Hq, Hkv, dh
    d.scale, d.window, d.pad_id = dh ** -0.5, window, pad
    d.q, d.kcache, d.vcache, d.out, d.ws = q.data_ptr(), kg.data_ptr(), vg.data_ptr(), out.data_ptr(), ws.data_ptr()
    if packed:
      d.segment_ids = gids.data_ptr()
    else:
      d.tokens = gids.data_ptr()
    d.tok_ld, d.col_ptr, d.kv_chunk = S, colp.data_ptr(), chunk
    ops.gqa_attn(d)
    torch.cuda.synchronize()
    lo = max(0, col - window + 1) if window else 0
    mask = torch.zeros(B, S, dtype=torch.bool)
    mask[:, lo:col + 1] = True
    mask &= (ids == ids[:, col:col + 1]) if packed else ids != pad
    score = (q.cpu().view(B, Hq, 1, dh).double() @ heads(kc).transpose(2, 3)) * dh ** -0.5
    ref = torch.softmax(score.masked_fill(~mask[:, None, None], -1e30), -1) @ heads(vc)
    live = mask.any(1)
    got = out.float().cpu().view(B, Hq, dh)
    diff = (got - ref[:, :, 0].float()).abs()[live]
    assert live.any() and diff.max().item() <= 2.0 ** -6 * max(1.0, ref[live].abs().max().item()), (col, diff.max().item())
    assert (got[~live] == 0).all()


@pytest.mark.parametrize("M,K,N,batch,ldx,ldy,relu2", [
    (1, 16, 1, 1, 16, 1, False),             # one turn of the k range, one row and column
    (16, 2048, 512, 1, 2048, 512, False),
    (33, 144, 75, 1, 148, 77, True),         # ragged everywhere, output rows off 16-byte alignment
    (70, 4112, 1000, 1, 4112, 1000, False),  # k turns that the waves do not share evenly
    (1300, 48, 1664, 1, 48, 1664, False),    # tiles of 128: half a step of k at the end
    (1537, 2064, 1025, 1, 2064, 1028, True),
    (400, 144, 1000, 1, 148, 1003, False),   # tiles of 64
    (129, 16, 4100, 1, 16, 4100, True),
    (1601, 80, 2050, 1, 80, 2053, True),     # tiles of 128 where those of 64 take four rounds
    (65, 48, 72, 130, 48, 72, False),
    (40, 64, 96, 9, 64, 96, False),          # a batch, few tiles and many
    (300, 256, 640, 9, 256, 640, False),
])
def test_dense_linear_in_32_bits(gpu, M, K, N, batch, ldx, ldy, relu2):
  """Few rows and many, against the products in 64 bits: every element within K roundings of its products' magnitudes."""
  from tunix_amd import _lib as L
  from tunix_amd import ops
  x, w = rnd((batch, M, ldx), 401).to(gpu), rnd((batch, N, K), 402).to(gpu)
  y = torch.full((batch, M, ldy), float("nan"), device=gpu)
  d = L.DenseDesc()
  d.M, d.K, d.N, d.dtype, d.split_k, d.batch = M, K, N, ops.DTYPES[torch.float32], 1, batch
  d.x, d.ldx, d.w, d.y, d.ldy = x.data_ptr(), ldx, w.data_ptr(), y.data_ptr(), ldy
  d.epilogue = L.TNX_EPI_RELU2 if relu2 else L.TNX_EPI_F32
  d.x_stride, d.w_stride, d.y_stride = M * ldx, N * K, M * ldy
  ops.dense_linear(d)
  xd, wd = x[..., :K].cpu().double(), w.cpu().double()
  want, size = xd @ wd.transpose(1, 2).contiguous(), xd.abs() @ wd.abs().transpose(1, 2).contiguous()
  bound = (K + 1) * 2.0 ** -24 * size
  if relu2:
    want, bound = want.clamp_min(0) ** 2, bound * (2 * want.abs() + bound) + 2.0 ** -23 * want ** 2
  got = y.cpu().double()
  assert ((got[..., :N] - want).abs() <= bound).all() and got[..., N:].isnan().all()


@pytest.mark.parametrize("K,N,counts,x_div", [
    (48, 75, (0, 3, 17, 0, 1), 1), (256, 512, (130, 0, 1, 301), 1), (2048, 256, (9, 40, 31, 0), 2),
    (48, 1000, (80, 64, 65, 0, 3) * 8, 2),                  # tiles of 64
    (80, 2040, (100, 96, 128, 129, 7, 99, 140, 101) * 2, 1),  # tiles of 128
])
def test_dense_experts_in_32_bits(gpu, K, N, counts, x_div):
  from tunix_amd import _lib as L
  from tunix_amd import ops
  E, n = len(counts), sum(counts)
  x, w = rnd(((n + x_div - 1) // x_div, K), 403).to(gpu), rnd((E, N, K), 404).to(gpu)
  route = torch.randperm(n, generator=torch.Generator().manual_seed(1)).to(torch.int32).to(gpu)
  offsets = torch.tensor([0] + [int(v) for v in np.cumsum(counts)], dtype=torch.int32, device=gpu)
  y = torch.full((n, N), float("nan"), device=gpu)
  d = L.DenseDesc()
  d.M, d.K, d.N, d.dtype, d.batch, d.split_k = n, K, N, ops.DTYPES[torch.float32], 1, 1
  d.x, d.ldx, d.w, d.w_stride, d.epilogue, d.y, d.ldy = x.data_ptr(), K, w.data_ptr(), N * K, L.TNX_EPI_F32, y.data_ptr(), N
  d.n_experts, d.x_div, d.offsets, d.sorted_route = E, x_div, offsets.data_ptr(), route.data_ptr()
  ops.dense_linear(d)
  for e, (a0, a1) in enumerate(zip(offsets.tolist()[:-1], offsets.tolist()[1:])):
    r = route[a0:a1].long()
    xe, we = x[r // x_div].cpu().double(), w[e].cpu().double()
    assert ((y[r].cpu().double() - xe @ we.T).abs() <= (K + 1) * 2.0 ** -24 * (xe.abs() @ we.abs().T)).all()


@pytest.mark.parametrize("family,dh,Hq,Hkv,split,chunk,window,R", [
    ("qwen3", 64, 8, 2, 4, 64, 0, 16),      # chunks of two key blocks, each by one wave
    ("qwen3", 128, 6, 2, 5, 0, 50, 32),     # a window of up to three
    ("qwen3", 64, 4, 2, 4, 0, 0, 32),       # half a wave per head
    ("qwen3", 128, 16, 2, 6, 96, 0, 16),    # ten heads of a pair of kv heads, split over chunks
    ("gemma3", 256, 4, 1, 5, 128, 100, 32),
    ("gemma3", 256, 16, 1, 8, 0, 0, 0),     # more heads than one batch of the waves takes, no adapter
    ("llama3", 128, 6, 2, 3, 0, 0, 16),     # no norms, three heads in lanes of four
    ("qwen3", 128, 8, 2, 9, 0, 0, 16),      # too many planes: the two launches
    ("qwen3", 128, 11, 1, 8, 64, 0, 16),    # of a few keys one head more than a batch of the waves: the two launches
])
def test_norms_rotation_and_attention_in_one_launch(gpu, family, dh, Hq, Hkv, split, chunk, window, R):
  """tnx_rope_gqa_attn_lora against the launches it stands for, at columns on both sides of the waves' shares: the cache bit for
  bit, the output to a bf16 ulp (the step's own key enters the softmax as a block of its own), of one wave's keys bit for bit too."""
  from tunix_amd import _lib as L
  from tunix_amd import ops
  from tunix_amd.model import rope_timescale
  B, S = 3, 300
  ld = (Hq + 2 * Hkv) * dh
  g = torch.Generator().manual_seed(700 + dh)
  ws = (torch.randn(split, B, ld, generator=g) * split ** -0.5).to(gpu)
  norms = [(torch.randn(dh, generator=g) * 0.1 + (0.0 if family == "gemma3" else 1.0)).to(torch.bfloat16).to(gpu) for _ in range(2)]
  ts = torch.from_numpy(rope_timescale(dh, 1e4)).to(gpu)
  pos = torch.randint(0, 900, (B, S), generator=g, dtype=torch.int32).to(gpu)
  tokens = torch.randint(1, 50, (B, S), generator=g, dtype=torch.int32)
  tokens[1, :9] = 0
  tokens = tokens.to(gpu)
  kc0, vc0 = (torch.randn(B, Hkv, S, dh, generator=g).to(torch.bfloat16).to(gpu) for _ in range(2))
  a_t = torch.randn(R, Hq * dh, generator=g).to(torch.bfloat16).to(gpu) if R else None
  for col in (0, 9, 31, 32, 127, 128, 160, 299):
    colp = torch.tensor([col], dtype=torch.int32, device=gpu)
    got = []
    for one in (False, True):
      kc, vc, q = kc0.clone(), vc0.clone(), torch.empty(B, Hq * dh, dtype=torch.bfloat16, device=gpu)
      out, t = torch.empty_like(q), torch.zeros(B, 32, dtype=torch.bfloat16, device=gpu)
      part = torch.empty(max(ops.attn_ws_bytes(B, 1, S, Hq, dh, chunk) // 4, 1), device=gpu)
      rd, d = L.RopeDesc(), L.AttnDesc()
      for x in (rd, d):
        x.B, x.T, x.S, x.Hq, x.Hkv, x.dh = B, 1, S, Hq, Hkv, dh
        x.kcache, x.vcache, x.col_ptr = kc.data_ptr(), vc.data_ptr(), colp.data_ptr()
      rd.rope_flavor, rd.rope_scale, rd.timescale = {"llama3": L.TNX_ROPE_LLAMA, "qwen3": L.TNX_ROPE_QWEN3, "gemma3": L.TNX_ROPE_GEMMA3}[family], 2.0, ts.data_ptr()
      rd.qk_norm = {"llama3": -1, "qwen3": L.TNX_NORM_QWEN3, "gemma3": L.TNX_NORM_GEMMA3}[family]
      rd.norm_eps, rd.q_norm_w, rd.k_norm_w = 1e-6, norms[0].data_ptr(), norms[1].data_ptr()
      rd.q_prescale = dh ** -0.5 if family == "gemma3" else 0.0
      rd.qkv_ws, rd.split_k, rd.positions, rd.pos_ld, rd.q_out = ws.data_ptr(), split, pos.data_ptr(), S, q.data_ptr()
      d.scale, d.window, d.q, d.out, d.ws = 0.0 if family == "gemma3" else dh ** -0.5, window, q.data_ptr(), out.data_ptr(), part.data_ptr()
      d.tokens, d.tok_ld, d.kv_chunk = tokens.data_ptr(), S, chunk
      if one:
        ops.rope_gqa_attn_lora(rd, d, a_t, t)
      else:
        ops.rope_kvwrite(rd)
        ops.gqa_attn(d)
      torch.cuda.synchronize()
      got.append((kc, vc, out.float(), t))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1]) and not torch.equal(got[0][0], kc0), col
    ref, out = got[0][2], got[1][2]
    ulp = 2.0 ** (torch.floor(torch.log2(torch.maximum(ref.abs(), out.abs()).clamp_min(0.5))) - 7)
    assert ((ref - out).abs() <= ulp).all(), (col, ((ref - out).abs() / ulp).max().item())
    if min(chunk or S, window or S) <= 64:
      assert torch.equal(ref, out), col
    if R:
      assert_down_projection(got[1][3][:, :R], got[1][2].to(torch.bfloat16), a_t)
