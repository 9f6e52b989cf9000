"""End-to-end parity of the HIP Sampler against the CPU oracle (through the C ABI).

Greedy ids: the oracle is teacher-forced with the ids the GPU produced; at every generated
position the GPU id must be the oracle's arg-max, or lie within two bf16 ulps of it (the logits
are bf16 values, so near-ties flip with the fp32 accumulation order; every such case is listed
with its top-2 margin, and the counts go to a summary file next to the run's other outputs).
Log-probs: <= 2e-2 absolute against the oracle's bf16 flow and against the fp32 reference mode.
"""
import numpy as np
import pytest
import torch

from oracle import model_ref as MR
from oracle import rl_ref
from oracle import sampler_ref as SR
from oracle import utils_ref as U
from tests import kezolix_cases, kuzezen_cases, lapevik_cases, nunezen_cases

pytestmark = pytest.mark.gpu


def _prompts(B, P, V, seed, ragged=True):
  rng = np.random.Generator(np.random.PCG64(seed))
  out = []
  for b in range(B):
    n = P if (not ragged or b % 3 == 0) else int(rng.integers(P // 2, P + 1))
    out.append(rng.integers(1, V, size=n).astype(np.int32))
  return out


def _oracle_full_logits(ref, token_buffer, pad_id):
  """Teacher-forced oracle logits for every column of the token buffer."""
  tb = np.asarray(token_buffer)
  B, L = tb.shape
  mask = tb != pad_id
  pos = U.build_positions_from_mask(mask)
  attn = U.make_causal_attn_mask(mask)
  cache = ref.init_cache(B, L)
  return ref(torch.from_numpy(tb.astype(np.int64)), torch.from_numpy(pos.astype(np.int64)), cache,
             torch.from_numpy(attn), 0)


NEAR_TIES = []   # (label, positions, ids that differ from the oracle arg-max, their margins in ulps)


def _write_near_tie_summary():
  """One line per checked rollout: how many greedy ids were not the oracle's arg-max and how far
  (in bf16 ulps of the top logit) the chosen logit lay below it."""
  import json
  import os
  root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
  out = os.path.join(root, "gpurun_out")
  try:
    os.makedirs(out, exist_ok=True)
    with open(os.path.join(out, "greedy_near_ties.json"), "w") as f:
      json.dump([{"case": c, "positions": n, "not_argmax": len(u), "margins_ulp": [round(x, 2) for x in u]}
                 for c, n, u in NEAR_TIES], f, indent=1)
  except OSError:
    pass


def _check_greedy(tb, logits, P, gpu_logprobs=None, lp_tol=2e-2, label=None, max_ulps=2.0):
  B, L = tb.shape
  report = []
  n = 0
  for b in range(B):
    for c in range(P, L):
      lg = logits[b, c - 1]
      best = int(torch.argmax(lg))
      tok = int(tb[b, c])
      n += 1
      if tok != best:
        margin = float(lg[best] - lg[tok])
        ulp = 2.0 ** (np.floor(np.log2(max(abs(float(lg[best])), 2.0 ** -120))) - 7)  # bf16 spacing
        report.append((b, c, tok, best, margin, margin / ulp))
  import inspect
  NEAR_TIES.append((label or inspect.stack()[1].function, n, [r[5] for r in report]))
  _write_near_tie_summary()
  for r in report:
    assert r[5] <= max_ulps, f"greedy id differs beyond a near-tie: {r}"
  if gpu_logprobs is not None:
    lp = torch.log_softmax(logits.float(), dim=-1)
    ref_lp = np.array([[float(lp[b, c - 1, int(tb[b, c])]) for c in range(P, L)] for b in range(B)])
    # 2e-2 absolute, the tolerance of the bf16 path; the logits are bf16 values, so where the
    # chosen logit exceeds 1 in magnitude two of its own ulps (2 * 2^(e-7)) are the floor
    mag = np.array([[abs(float(logits[b, c - 1, int(tb[b, c])])) for c in range(P, L)] for b in range(B)])
    tol = np.maximum(lp_tol, 2.0 * 2.0 ** (np.floor(np.log2(np.maximum(mag, 1e-30))) - 7))
    err = np.abs(np.asarray(gpu_logprobs)[:, P:L] - ref_lp)
    assert (err <= tol).all(), f"logprob error {err.max()} (largest allowed {tol.max()})"
  return report, n


@pytest.fixture(scope="module")
def tiny(gpu):
  from tunix_amd import config, dummy_model
  from tunix_amd.model import QLoRAModel
  cfg = config.tiny_qwen3()
  w = dummy_model.create_dummy_weights(cfg, seed=20251)
  return cfg, w, QLoRAModel(cfg, w, gpu)


def test_tiny_qwen3_greedy_decode(tiny, gpu):
  """The reference's own CPU-runnable case: 2 layers, B8, P64, 64 greedy steps + logprobs."""
  from tunix_amd.generate import CacheConfig, Sampler
  from tunix_amd.generate.utils import IdTokenizer
  cfg, w, model = tiny
  B, P, T = 8, 64, 64
  tok = IdTokenizer(cfg.vocab_size, pad_id=0, eos_id=1)
  sampler = Sampler(model, tok, CacheConfig(P + T, cfg.num_layers, cfg.num_kv_heads, cfg.head_dim))
  prompts = _prompts(B, P, cfg.vocab_size, 20251)
  out = sampler(prompts, max_generation_steps=T, max_prompt_length=P, return_logprobs=True,
                eos_tokens=[-1])
  st = sampler._last_state
  tb = st.token_buffer.cpu().numpy()
  assert all(len(t) == T for t in out.tokens)
  np.testing.assert_array_equal(out.padded_prompt_tokens, tb[:, :P])
  ref = MR.RefModel(cfg, w)
  logits = _oracle_full_logits(ref, tb, 0)
  report, n = _check_greedy(tb, logits, P, st.logprobs_buffer.cpu().numpy())
  print(f"greedy: {n - len(report)}/{n} ids equal the oracle arg-max; near-ties: {report}")
  # random N(0, 0.02) weights give nearly flat bf16 logits: a few per cent of the positions
  # have a top-2 margin of 0-2 ulps, where the accumulation order decides
  assert len(report) <= n // 20
  # sanity bound against the unrounded fp32 model: the distance is the bf16 rounding of the
  # whole network (both paths above already agree to 2e-2 with each other), so it only has to
  # stay of that order
  ref32 = MR.RefModel(cfg, w, bf16=False)
  lg32 = _oracle_full_logits(ref32, tb, 0)
  lp32 = torch.log_softmax(lg32.float(), -1)
  got = st.logprobs_buffer.cpu().numpy()
  err = max(abs(got[b, c] - float(lp32[b, c - 1, int(tb[b, c])])) for b in range(B) for c in range(P, P + T))
  assert err <= 5e-2, err
  # the oracle's own sampler loop reproduces the same buffer wherever no near-tie occurred
  if not report:
    ids = np.stack([U.pad_to_length(p, P, 0, left=True) for p in prompts])
    run = SR.run(ref, ids, T, 0, P + T, [-1])
    np.testing.assert_array_equal(run["token_buffer"], tb)


def test_graph_replay_equals_eager(tiny, gpu):
  from tunix_amd.generate import CacheConfig, Sampler
  from tunix_amd.generate.utils import IdTokenizer
  cfg, w, model = tiny
  tok = IdTokenizer(cfg.vocab_size, pad_id=0, eos_id=1)
  cc = CacheConfig(64, cfg.num_layers, cfg.num_kv_heads, cfg.head_dim)
  prompts = _prompts(4, 16, cfg.vocab_size, 7)
  a = Sampler(model, tok, cc, use_graph=True)(prompts, 40, return_logprobs=True, eos_tokens=[-1])
  b = Sampler(model, tok, cc, use_graph=False)(prompts, 40, return_logprobs=True, eos_tokens=[-1])
  for x, y in zip(a.tokens, b.tokens):
    np.testing.assert_array_equal(x, y)
  np.testing.assert_array_equal(np.asarray(a.logprobs), np.asarray(b.logprobs))


@pytest.mark.parametrize("rows", [3, 130])
@pytest.mark.parametrize("family,name,dtype", [("qlora", "tiny", "bf16")] + [
    (f, n, t) for f, cases in (("nunezen", nunezen_cases), ("lapevik", lapevik_cases), ("kuzezen", kuzezen_cases), ("kezolix", kezolix_cases))
    for n in sorted(cases.CONFIGS) for t in ("bf16", "fp32")])
def test_a_captured_step_allocates_nothing(tiny, gpu, family, name, dtype, rows):
  """Every buffer of a decode step is there before its capture: what the capture allocated (and filled) would be done again by
  every replay."""
  import importlib
  from tunix_amd.generate import CacheConfig, Sampler
  from tunix_amd.generate.utils import IdTokenizer
  if family == "qlora":
    model = tiny[2]
  else:
    model = importlib.import_module(f"tests.test_gpu_{family}").model_of(name, 3, torch.bfloat16 if dtype == "bf16" else torch.float32, gpu)[2]
  counts = []

  class Watched(Sampler):
    def _captured(self, step):
      def watched():
        count = lambda: torch.cuda.memory_stats(gpu)["allocation.all.allocated"]
        before = count()
        step()
        counts.append(count() - before)
      return super()._captured(watched)

  V = model.cfg.vocab_size
  prompts = [np.arange(2 + b % 5, 9, dtype=np.int32) % V for b in range(rows)]
  sampler = Watched(model, IdTokenizer(V, pad_id=0, eos_id=1), CacheConfig(64))
  for kw in (dict(return_logprobs=True), dict(temperature=1.0, top_p=1.0), dict(temperature=1.0, top_p=0.9, top_k=10)):
    sampler(prompts, 5, max_prompt_length=16, eos_tokens=[-1], **kw)
  assert counts == [0, 0, 0]


@pytest.mark.parametrize("free,given_back", [(64 << 20, True), (512 << 20, False)])
def test_a_capture_gives_the_cache_back_only_where_a_graph_has_no_room(tiny, gpu, monkeypatch, free, given_back):
  """A graph takes some MiB of the device, and no more than the room that a capture asks for."""
  from tunix_amd.generate import CacheConfig, Sampler
  from tunix_amd.generate.utils import IdTokenizer
  cfg, w, model = tiny
  taken, emptied = [], []

  class Watched(Sampler):
    def _captured(self, step):
      torch.cuda.synchronize(gpu)
      before = torch.cuda.mem_get_info(gpu)[0]
      with monkeypatch.context() as m:
        empty = torch.cuda.empty_cache
        m.setattr(torch.cuda, "mem_get_info", lambda device=None: (free, 288 << 30))
        m.setattr(torch.cuda, "empty_cache", lambda: (emptied.append(1), empty()))
        graph = super()._captured(step)
      taken.append(before - torch.cuda.mem_get_info(gpu)[0])
      return graph

  sampler = Watched(model, IdTokenizer(cfg.vocab_size, pad_id=0, eos_id=1), CacheConfig(64))
  prompts = _prompts(4, 16, cfg.vocab_size, 7)
  a = sampler(prompts, 20, eos_tokens=[-1])
  assert bool(emptied) == given_back and taken[0] < Sampler.CAPTURE_ROOM
  b = Sampler(model, sampler.tokenizer, CacheConfig(64), use_graph=False)(prompts, 20, eos_tokens=[-1])
  for x, y in zip(a.tokens, b.tokens):
    np.testing.assert_array_equal(x, y)


def test_sampler_contract(tiny, gpu):
  """Errors, eos truncation, echo, pad_output, return_logits (tunix/generate/sampler.py:868-1011)."""
  from tunix_amd.generate import CacheConfig, Sampler
  from tunix_amd.generate.utils import IdTokenizer
  cfg, w, model = tiny
  tok = IdTokenizer(cfg.vocab_size, pad_id=0, eos_id=1)
  sampler = Sampler(model, tok, CacheConfig(32, cfg.num_layers, cfg.num_kv_heads, cfg.head_dim))
  with pytest.raises(ValueError, match="must be less than the cache size"):
    sampler(["5 6 7"], max_generation_steps=40)
  out = sampler(["5 6 7", "9 10 11 12 13"], max_generation_steps=8, return_logits=True,
                return_logprobs=True, eos_tokens=[-1])
  assert out.padded_prompt_tokens.shape == (2, 8)          # next power of two of 5
  assert out.padded_prompt_tokens[0].tolist() == [0, 0, 0, 0, 0, 5, 6, 7]
  assert [len(t) for t in out.tokens] == [8, 8]
  assert out.logits[0].shape == (8, cfg.vocab_size)
  for b in range(2):
    np.testing.assert_array_equal(np.argmax(out.logits[b], -1), out.tokens[b])
    lp = torch.log_softmax(torch.from_numpy(out.logits[b]), -1).numpy()
    np.testing.assert_allclose(out.logprobs[b], lp[np.arange(8), out.tokens[b]], atol=2e-5)
  # an eos id truncates the row's output at its first occurrence
  eos = int(out.tokens[0][3])
  out2 = sampler(["5 6 7", "9 10 11 12 13"], max_generation_steps=8, eos_tokens=[eos])
  first = int(np.flatnonzero(out.tokens[0] == eos)[0])
  assert len(out2.tokens[0]) == first
  np.testing.assert_array_equal(out2.tokens[0], out.tokens[0][:first])
  out3 = sampler(["5 6 7"], max_generation_steps=4, echo=True, pad_output=True, eos_tokens=[-1])
  assert out3.tokens[0].shape == (4 + 4,) and out3.tokens[0][:3].tolist() == [5, 6, 7]
  with pytest.raises(NotImplementedError):
    sampler(["5"], 2, beam_size=2)


def test_single_step_forbidden_ids_and_prompt_length(tiny, gpu):
  """The cases of tests/generate/sampler_test.py:412-466 (one generation step: the decode loop
  adds nothing after the prefill), :632-665 (forbidden ids never appear, in greedy mode and when
  drawing) and :100-152 (an explicit max_prompt_length at least as long as the prompts is used
  as given, a shorter one is replaced by the next power of two)."""
  from tunix_amd.generate import CacheConfig, Sampler
  from tunix_amd.generate.utils import IdTokenizer
  cfg, w, model = tiny
  V = cfg.vocab_size
  tok = IdTokenizer(V, pad_id=0, eos_id=1)
  sampler = Sampler(model, tok, CacheConfig(64, cfg.num_layers, cfg.num_kv_heads, cfg.head_dim))
  prompts = ["5 6 7", "9 10 11 12 13"]
  ref = sampler(prompts, max_generation_steps=6, eos_tokens=[-1])
  one = sampler(prompts, max_generation_steps=1, eos_tokens=[-1], return_logprobs=True)
  assert [len(t) for t in one.tokens] == [1, 1]
  assert [int(t[0]) for t in one.tokens] == [int(t[0]) for t in ref.tokens]
  assert all(len(lp) == 1 and np.isfinite(lp).all() for lp in one.logprobs)

  allowed = V // 4
  forbidden = set(range(allowed, V)) | {tok.eos_id()}
  steps = 40
  for kw in (dict(temperature=1.0, seed=123),                       # greedy: no top_p given
             dict(temperature=1.0, top_p=1.0, seed=123),             # categorical draw in the head
             dict(temperature=0.8, top_p=0.9, top_k=20, seed=7)):    # top-k / top-p kernel
    out = sampler(["5 6 7"], max_generation_steps=steps, forbidden_tokens=forbidden, **kw)
    assert len(out.tokens[0]) == steps, kw
    assert not (set(out.tokens[0].tolist()) & forbidden), kw

  wide = sampler(prompts, max_generation_steps=4, max_prompt_length=16, eos_tokens=[-1])
  assert wide.padded_prompt_tokens.shape == (2, 16)
  assert wide.padded_prompt_tokens[1].tolist() == [0] * 11 + [9, 10, 11, 12, 13]
  short = sampler(prompts, max_generation_steps=4, max_prompt_length=2, eos_tokens=[-1])
  assert short.padded_prompt_tokens.shape == (2, 8)
  # left padding is masked out: the continuation does not depend on the padded width
  for b in range(2):
    np.testing.assert_array_equal(wide.tokens[b], ref.tokens[b][:4])
    np.testing.assert_array_equal(short.tokens[b], ref.tokens[b][:4])


@pytest.mark.parametrize("top_k,top_p", [(50, 0.95), (None, 0.9), (None, 1.0)])
def test_top_p_sampling_against_oracle(tiny, gpu, top_k, top_p):
  """temperature / top-k / top-p, top-p over the whole vocabulary (no top-k) and the plain
  categorical draw (the reference's default rollout configuration: top_p 1.0, no top-k).  The draw depends on the RANK of every candidate (the noise is
  indexed by sorted position), so one bf16 ulp in one logit re-deals the noise: ids are checked
  exactly against the oracle's draw from the logits the GPU itself produced, and those logits
  against the teacher-forced oracle within bf16 resolution."""
  from oracle import threefry as TF
  from tunix_amd.generate import CacheConfig, Sampler
  from tunix_amd.generate.utils import IdTokenizer
  cfg, w, model = tiny
  B, P, T = 4, 16, 12
  tok = IdTokenizer(cfg.vocab_size, pad_id=0, eos_id=1)
  sampler = Sampler(model, tok, CacheConfig(P + T, cfg.num_layers, cfg.num_kv_heads, cfg.head_dim))
  prompts = _prompts(B, P, cfg.vocab_size, 99, ragged=False)
  temp = 0.8
  out = sampler(prompts, T, max_prompt_length=P, temperature=temp, top_p=top_p, top_k=top_k, seed=42,
                return_logprobs=True, return_logits=True, eos_tokens=[-1])
  tb = sampler._last_state.token_buffer.cpu().numpy()
  ref = MR.RefModel(cfg, w)
  logits = _oracle_full_logits(ref, tb, 0)
  key = TF.prng_key(42)
  for c in range(P, P + T):
    gpu_lg = torch.from_numpy(np.stack([out.logits[b][c - P] for b in range(B)]))   # raw logits
    t_ref, lp_ref = SR.sample_top_p(gpu_lg, TF.fold_in(key, c - 1), temp, top_p, top_k)
    np.testing.assert_array_equal(t_ref.numpy(), tb[:, c])
    got_lp = np.array([out.logprobs[b][c - P] for b in range(B)])
    np.testing.assert_allclose(got_lp, lp_ref.numpy(), atol=2e-5)
    diff = (gpu_lg - logits[:, c - 1]).abs()
    assert diff.max().item() <= 2.0 ** -6 * max(1.0, logits[:, c - 1].abs().max().item())
    lp_full = torch.log_softmax(logits[:, c - 1].float() / temp, -1)
    for b in range(B):
      assert abs(out.logprobs[b][c - P] - float(lp_full[b, tb[b, c]])) <= 2e-2
  # the graph-replayed path draws the same ids; another seed changes them
  out_b = sampler(prompts, T, max_prompt_length=P, temperature=temp, top_p=top_p, top_k=top_k,
                  seed=42, eos_tokens=[-1])
  out_c = sampler(prompts, T, max_prompt_length=P, temperature=temp, top_p=top_p, top_k=top_k,
                  seed=43, eos_tokens=[-1])
  assert all(np.array_equal(x, y) for x, y in zip(out.tokens, out_b.tokens))
  assert not all(np.array_equal(x, y) for x, y in zip(out.tokens, out_c.tokens))


def test_lora_update_changes_output_and_checks_structure(tiny, gpu):
  """LoRA-only weight sync (tunix/generate/sampler.py:333-352)."""
  from tunix_amd.generate import CacheConfig, Sampler
  from tunix_amd.generate.utils import IdTokenizer
  cfg, w, model = tiny
  tok = IdTokenizer(cfg.vocab_size, pad_id=0, eos_id=1)
  sampler = Sampler(model, tok, CacheConfig(32, cfg.num_layers, cfg.num_kv_heads, cfg.head_dim))
  lora = {k: v for k, v in w.items() if ".lora_" in k}
  base = sampler(["3 4 5 6"], 8, return_logprobs=True, eos_tokens=[-1])
  zero_b = {k: (torch.zeros_like(v) if k.endswith("lora_b") else v) for k, v in lora.items()}
  sampler.update_lora(zero_b)
  changed = sampler(["3 4 5 6"], 8, return_logprobs=True, eos_tokens=[-1])
  assert np.abs(np.asarray(base.logprobs) - np.asarray(changed.logprobs)).max() > 0
  # B = 0 equals the model without LoRA (qwix zero-init invariant)
  w_nolora = {k: v for k, v in w.items() if ".lora_" not in k}
  ref = MR.RefModel(cfg, {**w_nolora, **zero_b})
  tb = sampler._last_state.token_buffer.cpu().numpy()
  _check_greedy(tb, _oracle_full_logits(ref, tb, 0), 4,
                sampler._last_state.logprobs_buffer.cpu().numpy())
  sampler.update_lora(lora)
  again = sampler(["3 4 5 6"], 8, return_logprobs=True, eos_tokens=[-1])
  np.testing.assert_array_equal(np.asarray(base.logprobs), np.asarray(again.logprobs))
  bad = dict(lora)
  bad.pop(next(iter(bad)))
  with pytest.raises(ValueError, match="same structure"):
    sampler.update_lora(bad)


def test_full_state_replacement_requantises_in_place(tiny, gpu):
  """Full-state replacement (tunix/generate/sampler.py:322-325): new base weights are re-quantised
  and re-packed into the buffers the model already holds; afterwards the model is bit-identical
  to one built from the new weights, and a partial state that splits a fused projection, or has
  another shape, raises."""
  from tunix_amd import dummy_model
  from tunix_amd.generate import CacheConfig, Sampler
  from tunix_amd.generate.utils import IdTokenizer
  from tunix_amd.model import QLoRAModel
  cfg, w, _ = tiny
  model = QLoRAModel(cfg, w, gpu)
  w2 = dummy_model.create_dummy_weights(cfg, seed=777)
  fresh = QLoRAModel(cfg, w2, gpu)
  ptr = model.layers[0]["qkv"].codes.data_ptr()
  tok = IdTokenizer(cfg.vocab_size, pad_id=0, eos_id=1)
  cc = CacheConfig(32, cfg.num_layers, cfg.num_kv_heads, cfg.head_dim)
  sampler = Sampler(model, tok, cc)
  before = sampler(["3 4 5 6"], 8, return_logprobs=True, eos_tokens=[-1])
  sampler.update_params(w2)                       # base + LoRA leaves
  assert model.layers[0]["qkv"].codes.data_ptr() == ptr
  for a, b in zip(model.layers, fresh.layers):
    for key in ("qkv", "o", "gu", "down"):
      assert torch.equal(a[key].codes, b[key].codes) and torch.equal(a[key].scales, b[key].scales)
      assert torch.equal(a[key].a_t, b[key].a_t) and torch.equal(a[key].b_t, b[key].b_t)
    assert torch.equal(a["attn_norm"], b["attn_norm"])
  assert torch.equal(model.embed, fresh.embed) and torch.equal(model.head_w, fresh.head_w)
  after = sampler(["3 4 5 6"], 8, return_logprobs=True, eos_tokens=[-1])
  want = Sampler(fresh, tok, cc)(["3 4 5 6"], 8, return_logprobs=True, eos_tokens=[-1])
  np.testing.assert_array_equal(after.tokens[0], want.tokens[0])
  np.testing.assert_array_equal(np.asarray(after.logprobs), np.asarray(want.logprobs))
  assert np.abs(np.asarray(before.logprobs) - np.asarray(after.logprobs)).max() > 0
  # base weights only: the adapters stay
  base_only = {k: v for k, v in w.items() if ".lora_" not in k}
  sampler.update_params(base_only)
  assert torch.equal(model.layers[0]["qkv"].a_t, fresh.layers[0]["qkv"].a_t)
  with pytest.raises(ValueError, match="same structure"):
    sampler.update_params({"l0.wq": w["l0.wq"]})                       # wk / wv of the fused projection missing
  with pytest.raises(ValueError, match="same shape"):
    sampler.update_params({"embed": w["embed"][:, :8]})
  with pytest.raises(ValueError, match="same structure"):
    sampler.update_params({"no_such_leaf": w["embed"]})


def test_rejected_state_leaves_the_model_untouched(tiny, gpu):
  """A state that is refused must not have changed anything: every name, fused-member set and
  shape is checked before the first copy (the reference validates before it replaces,
  tunix/generate/sampler.py:280-284, :322-325)."""
  from tunix_amd import dummy_model
  from tunix_amd.model import QLoRAModel
  cfg, w, _ = tiny
  model = QLoRAModel(cfg, w, gpu)
  w2 = dummy_model.create_dummy_weights(cfg, seed=4242)
  snap = {"embed": model.embed.clone(), "final_norm": model.final_norm.clone(),
          "qkv0": model.layers[0]["qkv"].codes.clone(), "o0": model.layers[0]["o"].codes.clone(),
          "a0": model.layers[0]["qkv"].a_t.clone(), "norm0": model.layers[0]["attn_norm"].clone()}

  def untouched():
    return (torch.equal(snap["embed"], model.embed) and torch.equal(snap["final_norm"], model.final_norm)
            and torch.equal(snap["qkv0"], model.layers[0]["qkv"].codes)
            and torch.equal(snap["o0"], model.layers[0]["o"].codes)
            and torch.equal(snap["a0"], model.layers[0]["qkv"].a_t)
            and torch.equal(snap["norm0"], model.layers[0]["attn_norm"]))

  # valid leaves first in iteration order, the offending one last
  with pytest.raises(ValueError, match="same structure"):   # wk / wv of the fused q|k|v missing
    model.update_params({"embed": w2["embed"], "final_norm": w2["final_norm"], "l0.wo": w2["l0.wo"],
                         "l0.attn_norm": w2["l0.attn_norm"], "l1.wq": w2["l1.wq"]})
  assert untouched()
  with pytest.raises(ValueError, match="same shape"):
    model.update_params({"embed": w2["embed"], "l0.wo": w2["l0.wo"], "l1.wo": w2["l1.wo"][:, :64]})
  assert untouched()
  with pytest.raises(ValueError, match="same shape"):       # a LoRA leaf of another rank, after valid base leaves
    model.update_params({"embed": w2["embed"], "l0.wq.lora_a": w2["l0.wq.lora_a"][:, :4],
                         "l0.wq.lora_b": w2["l0.wq.lora_b"][:4]})
  assert untouched()
  lora2 = {k: v for k, v in w2.items() if ".lora_" in k}
  bad = dict(lora2)
  last = sorted(k for k in bad if k.endswith(".lora_b"))[-1]
  bad[last] = bad[last][:, :8]
  with pytest.raises(ValueError, match="same shape"):       # LoRA-only swap, one wrong shape at the end
    model.update_lora(bad)
  assert untouched()
  model.update_params({"embed": w2["embed"]})                # and a valid partial state goes through
  assert not torch.equal(snap["embed"], model.embed)


def test_top_k_equal_to_the_vocabulary_sorts_the_row(tiny, gpu):
  """top_k == V is a real top-k in the reference (jax.lax.top_k(k = V): the row is sorted and the
  draw runs over sorted positions, tunix/generate/sampler.py:118-134), also with top_p = 1.0, so
  its ids differ from those of top_k = None for the same seed; top_k > V raises."""
  from oracle import threefry as TF
  from tunix_amd.generate import CacheConfig, Sampler
  from tunix_amd.generate.utils import IdTokenizer
  cfg, w, model = tiny
  B, P, T = 4, 16, 6
  V = cfg.vocab_size
  tok = IdTokenizer(V, pad_id=0, eos_id=1)
  sampler = Sampler(model, tok, CacheConfig(P + T, cfg.num_layers, cfg.num_kv_heads, cfg.head_dim))
  prompts = _prompts(B, P, V, 5, ragged=False)
  out = sampler(prompts, T, max_prompt_length=P, temperature=0.8, top_p=1.0, top_k=V, seed=3,
                return_logprobs=True, return_logits=True, eos_tokens=[-1])
  tb = sampler._last_state.token_buffer.cpu().numpy()
  key = TF.prng_key(3)
  for c in range(P, P + T):
    gpu_lg = torch.from_numpy(np.stack([out.logits[b][c - P] for b in range(B)]))
    t_ref, lp_ref = SR.sample_top_p(gpu_lg, TF.fold_in(key, c - 1), 0.8, 1.0, V)
    np.testing.assert_array_equal(t_ref.numpy(), tb[:, c])
    np.testing.assert_allclose(np.array([out.logprobs[b][c - P] for b in range(B)]), lp_ref.numpy(), atol=2e-5)
  plain = sampler(prompts, T, max_prompt_length=P, temperature=0.8, top_p=1.0, top_k=None, seed=3, eos_tokens=[-1])
  assert not all(np.array_equal(x, y) for x, y in zip(out.tokens, plain.tokens))
  with pytest.raises(ValueError, match="top_k"):
    sampler(prompts, T, max_prompt_length=P, temperature=0.8, top_p=1.0, top_k=V + 1, seed=3)


def test_captures_of_a_thread_share_a_stream(tiny, gpu):
  """One stream per thread to capture on, whatever became of the capture before."""
  import threading
  from tunix_amd.generate.sampler import CacheConfig, Sampler, _capture_stream
  from tunix_amd.generate.utils import IdTokenizer
  cfg, _, model = tiny[:3]
  sampler = Sampler(model, IdTokenizer(cfg.vocab_size), CacheConfig(32))
  generate = lambda: sampler([[5, 6, 7]], 8, max_prompt_length=8, eos_tokens=[-1]).tokens[0]
  want = generate()
  mine, other = _capture_stream(gpu), []
  x = torch.zeros(4, device=gpu)

  def fails():
    x.add_(1.0)
    raise ValueError("a step that fails")

  with pytest.raises(ValueError, match="a step that fails"):
    sampler._captured(fails)
  assert np.array_equal(generate(), want) and _capture_stream(gpu) is mine
  t = threading.Thread(target=lambda: other.extend([_capture_stream(gpu), generate()]))
  t.start()
  t.join()
  assert other[0] is not mine and np.array_equal(other[1], want)


@pytest.mark.parametrize("name,kw,P,lens,rows", [
    ("tiny_qwen3", {}, 64, (64, 40, 1, 57, 0), 16384),
    ("tiny_qwen3", {}, 64, (3, 40, 64, 57, 33), 130),          # groups of two prompts
    ("gemma3_1b", dict(num_layers=2, vocab_size=2048), 40, (40, 17, 33), 16384),
    ("llama31_8b", dict(num_layers=2, vocab_size=2048), 300, (290, 300), 16384),
    ("qwen3_30b_a3b", dict(num_layers=1, vocab_size=2048, num_experts=16), 33, (9, 30, 33), 16384),
])
def test_prompts_packed_and_padded_give_the_same(gpu, monkeypatch, name, kw, P, lens, rows):
  """The prompts' forward pass over their tokens alone and over the padded rows: the same tokens and the same bits of their log-probabilities.  (Groups of so few
  rows that the linears take another kernel: the first token's log-probability within what the greedy tests allow against the oracle.)"""
  from tunix_amd import config, dummy_model
  from tunix_amd.generate.sampler import CacheConfig, Sampler
  from tunix_amd.generate.utils import IdTokenizer
  from tunix_amd.model import QLoRAModel
  cfg = getattr(config, name)(**kw)
  model = QLoRAModel(cfg, dummy_model.create_dummy_weights(cfg, seed=3), "cuda:0")
  rng = np.random.default_rng(P)
  prompts = [rng.integers(2, cfg.vocab_size, size=n).astype(np.int32) for n in lens]
  sampler = Sampler(model, IdTokenizer(cfg.vocab_size), CacheConfig(P + 6), prefill_rows=rows)
  outs, packed = [], []
  monkeypatch.setattr(Sampler, "PACK_FROM", 0)
  packs = Sampler.packs
  for on in (True, False):
    monkeypatch.setattr(Sampler, "packs", staticmethod(lambda st, r: packed.append(packs(st, r)) or (packed[-1] and on)))
    outs.append(sampler(prompts, 6, max_prompt_length=P, return_logprobs=True, eos_tokens=[-1]))
  assert packed == [True, True]
  first = [np.asarray([lp[0] for lp in o.logprobs]) for o in outs]
  assert np.abs(first[0] - first[1]).max() <= 2e-2
  if rows > 1000:
    for a, b in zip(*(list(zip(o.tokens, o.logprobs)) for o in outs)):
      assert np.array_equal(a[0], b[0]) and np.array_equal(np.asarray(a[1]), np.asarray(b[1]))
