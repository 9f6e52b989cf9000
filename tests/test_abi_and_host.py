"""CPU checks of the boundary and the host logic: the shared library loads and exports every
entry point include/tunix_hip.h declares (no compute call is made here), the ctypes table covers
the same set with matching arity and struct sizes, argument checking works without a GPU where
it happens before any launch, and the host helpers agree with the oracle / the reference's
literal vectors."""
import ctypes
import os
import re
import subprocess

import numpy as np
import pytest

from oracle import utils_ref as U
from tunix_amd import _lib as L
from tunix_amd import config
from tunix_amd.generate import utils as G

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "tunix_hip.h")

DECL = re.compile(r"^(?:int|int64_t|size_t|const char\*)\s+(tnx_[a-z0-9_]+)\s*\(([^;]*)\)\s*;", re.M | re.S)


def _declared():
  text = open(HEADER).read()
  text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
  out = {}
  for m in DECL.finditer(text):
    args = m.group(2).strip()
    n = 0 if args in ("", "void") else len([a for a in args.split(",") if a.strip()])
    out[m.group(1)] = n
  return out


def test_header_declares_the_expected_entry_points():
  d = _declared()
  assert len(d) >= 23
  for name in ("tnx_qlinear_lora", "tnx_gqa_attn", "tnx_qknorm_rope_kvwrite", "tnx_rmsnorm",
               "tnx_lmhead_logp", "tnx_moe_int4_gmm", "tnx_sample_topk", "tnx_grpo_ratio"):
    assert name in d


def test_library_exports_every_declared_symbol():
  assert os.path.exists(L.LIB_PATH), "libtunix_hip.so is not built (run __graft_entry__.build())"
  handle = ctypes.CDLL(L.LIB_PATH)
  for name in _declared():
    assert hasattr(handle, name), f"{name} is declared in include/tunix_hip.h but not exported"
  # and nothing beyond the declared ABI leaks out with the tnx_ prefix (tnx_set_error is the
  # library-internal error setter shared by its translation units)
  nm = subprocess.run(["nm", "-D", "--defined-only", L.LIB_PATH], capture_output=True, text=True).stdout
  exported = {ln.split()[-1] for ln in nm.splitlines() if " T " in ln and ln.split()[-1].startswith("tnx_")}
  assert exported - set(_declared()) <= {"tnx_set_error"}, exported - set(_declared())


def test_ctypes_table_matches_header():
  d = _declared()
  assert set(L.SIGNATURES) == set(d)
  for name, (_, args) in L.SIGNATURES.items():
    assert len(args) == d[name], f"{name}: header has {d[name]} parameters, ctypes table {len(args)}"


def test_version_and_argument_errors_without_gpu():
  lib = L.lib()
  # the library, the header and the ctypes binding name one and the same ABI version
  hdr = open(HEADER).read()
  major = int(re.search(r"#define TNX_ABI_VERSION_MAJOR (\d+)", hdr).group(1))
  minor = int(re.search(r"#define TNX_ABI_VERSION_MINOR (\d+)", hdr).group(1))
  assert lib.tnx_version() == (major << 16) | minor
  assert L.ABI_VERSION == (major, minor)
  cb, sb = ctypes.c_size_t(), ctypes.c_size_t()
  assert lib.tnx_qw_sizes(4096, 4096, 64, ctypes.byref(cb), ctypes.byref(sb)) == 0
  assert cb.value == 4096 * 4096 // 2
  assert sb.value == (4096 // 16) * (4096 // 128) * 2 * 16 * 2 + 16
  rc = lib.tnx_qw_sizes(100, 4096, 64, ctypes.byref(cb), ctypes.byref(sb))
  assert rc == -22 and b"128" in lib.tnx_last_error()
  with pytest.raises(ValueError, match="128"):
    L.check(rc, "qw_sizes")
  assert lib.tnx_qw_sizes(4096, 4096, 48, None, None) == -22
  assert lib.tnx_lmhead_nblocks(128256) > 0


def test_struct_layouts_match_the_header(tmp_path):
  # the descriptor structs cross the C ABI by pointer: the ctypes mirrors must have the sizes and
  # the field offsets a C compiler gives the header's structs
  pairs = {"tnx_qlinear_desc": L.QLinearDesc, "tnx_rope_desc": L.RopeDesc,
           "tnx_attn_desc": L.AttnDesc, "tnx_lmhead_desc": L.LmHeadDesc, "tnx_moe_gmm_desc": L.MoeGmmDesc,
           "tnx_rows_src": L.RowsSrc, "tnx_dense_desc": L.DenseDesc, "tnx_residual_norm_desc": L.ResidualNormDesc,
           "tnx_part_rope_desc": L.PartRopeDesc, "tnx_sink_attn_desc": L.SinkAttnDesc, "tnx_lightning_desc": L.LightningDesc,
           "tnx_gated_norm_desc": L.GatedNormDesc, "tnx_logits_desc": L.LogitsDesc, "tnx_short_conv_desc": L.ShortConvDesc,
           "tnx_ssd_desc": L.SsdDesc, "tnx_latent_prep_desc": L.LatentPrepDesc, "tnx_latent_q_desc": L.LatentQDesc,
           "tnx_latent_kv_desc": L.LatentKvDesc, "tnx_latent_attn_desc": L.LatentAttnDesc, "tnx_gate_mul_desc": L.GateMulDesc,
           "tnx_parallel_step_desc": L.ParallelStepDesc, "tnx_conv_kvwrite_desc": L.ConvKvDesc, "tnx_mixed_attn_desc": L.MixedAttnDesc,
           "tnx_memory_desc": L.MemoryDesc, "tnx_rownorm_kvwrite_desc": L.RowNormKvDesc, "tnx_gated_state_desc": L.GatedStateDesc,
           "tnx_norm_lora_desc": L.NormLoraDesc, "tnx_commit_desc": L.CommitDesc, "tnx_embed_desc": L.EmbedDesc}
  lines = ['#include <stdio.h>', '#include <stddef.h>', '#include "tunix_hip.h"', 'int main(void) {']
  for cname, cls in pairs.items():
    lines.append(f'  printf("{cname} %zu\\n", sizeof({cname}));')
    for fname, _ in cls._fields_:
      lines.append(f'  printf("{cname}.{fname} %zu\\n", offsetof({cname}, {fname}));')
  lines += ['  return 0;', '}']
  src = tmp_path / "layout.c"
  src.write_text("\n".join(lines))
  exe = tmp_path / "layout"
  subprocess.run(["gcc", "-I", os.path.join(ROOT, "include"), str(src), "-o", str(exe)], check=True)
  got = dict(ln.split() for ln in subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout.splitlines())
  for cname, cls in pairs.items():
    assert int(got[cname]) == ctypes.sizeof(cls), cname
    for fname, _ in cls._fields_:
      assert int(got[f"{cname}.{fname}"]) == getattr(cls, fname).offset, f"{cname}.{fname}"


def test_host_utils_match_oracle_and_reference_vectors():
  assert [G.next_power_of_2(x) for x in (0, 2, 3, 4, 5)] == [1, 2, 4, 4, 8]
  x = np.array([1, 2, 3])
  np.testing.assert_array_equal(G.pad_to_length(x, 5, 0, left=True), U.pad_to_length(x, 5, 0, left=True))
  for ids in ([1, 2, 3, 4, 5, 6], [0, 0, 1, 2, 3, 4], [0, 1, 2, 3, 0, 0]):
    assert G.np_find_first_non_pad_idx(np.array(ids), 0) == U.find_first_non_pad_idx(np.array(ids), 0)
  for ids in ([1, 2, 3, 4, 5, -1], [1, 2, -1, 4, -1, 0], [1, 2, 3, 4, 5, 6]):
    assert G.np_find_first_eos_idx(np.array(ids), -1) == U.find_first_eos_idx(np.array(ids), -1)
  m = np.array([[1, 1, 1, 1], [0, 1, 1, 1], [1, 1, 1, 0], [0, 1, 1, 0]])
  np.testing.assert_array_equal(G.build_positions_from_mask(m), [[0, 1, 2, 3], [0, 0, 1, 2], [0, 1, 2, 2], [0, 0, 1, 1]])


def test_sampling_mode_conflict_message():
  cur = [None]
  G.check_sampling_mode_conflict(cur, "top_p")
  with pytest.raises(ValueError, match="Conflicts setting sampling_mode"):
    G.check_sampling_mode_conflict(cur, "greedy")


def test_id_tokenizer():
  t = G.IdTokenizer(100, pad_id=0, eos_id=1, bos_id=2)
  assert t.encode("5 6 7") == [5, 6, 7] and t.decode([5, 6]) == "5 6"
  assert t.dedup_bos_ids([2, 2, 2, 9]) == [2, 9]
  assert (t.pad_id(), t.eos_id(), t.bos_id()) == (0, 1, 2)


def test_config_presets():
  c = config.llama31_8b()
  assert (c.num_layers, c.embed_dim, c.hidden_dim, c.num_heads, c.num_kv_heads, c.head_dim, c.vocab_size) == (
      32, 4096, 14336, 32, 8, 128, 128256)
  assert c.qtype == config.Q_NF4 and c.group == 64 and c.lora_rank == 64
  g = config.gemma3_1b()
  assert [g.is_local_layer(i) for i in range(6)] == [True] * 5 + [False]
  assert g.rope_params(0) == (10_000.0, 1.0) and g.rope_params(5) == (1_000_000.0, 1.0)
  m = config.qwen3_30b_a3b()
  assert m.num_experts == 128 and m.num_experts_per_tok == 8
  assert "l0.e_gate" in m.quantized_names() and "l0.wq" in m.lora_names() and "l0.e_gate" not in m.lora_names()
  with pytest.raises(ValueError):
    config.ModelConfig(family="gpt2", num_layers=1, vocab_size=8, embed_dim=8, hidden_dim=8, num_heads=1,
                       num_kv_heads=1, head_dim=8)


def test_product_does_not_import_the_oracle():
  """The oracle is test infrastructure: nothing under tunix_amd/ may reference it."""
  pkg = os.path.join(ROOT, "tunix_amd")
  for dirpath, _, files in os.walk(pkg):
    for f in files:
      if f.endswith((".py", ".hip", ".h")):
        text = open(os.path.join(dirpath, f)).read()
        assert not re.search(r"^\s*(from|import)\s+oracle\b", text, re.M), os.path.join(dirpath, f)


def test_ffi_handlers_cover_the_documented_targets_and_call_declared_entry_points():
  """csrc/tunix_ffi.cc (the jax.ffi handlers, built only where jaxlib's headers exist) defines the
  twelve targets INTEGRATION.md lists and calls nothing the header does not declare."""
  src = open(os.path.join(ROOT, "tunix_amd", "csrc", "tunix_ffi.cc")).read()
  targets = set(re.findall(r"XLA_FFI_DEFINE_HANDLER_SYMBOL\((tnx_\w+_ffi)", src))
  doc = open(os.path.join(ROOT, "INTEGRATION.md")).read()
  documented = set(re.findall(r"`(tnx_\w+_ffi)`", doc))
  assert targets == documented and len(targets) == 12, (targets ^ documented)
  called = set(re.findall(r"\b(tnx_[a-z0-9_]+)\s*\(", src)) - {t for t in targets}
  assert called <= set(_declared()), called - set(_declared())


def test_binding_refuses_another_abi_version(monkeypatch):
  """A library of another major version (or an older minor one) must not be called."""
  major, minor = L.ABI_VERSION
  monkeypatch.setattr(L, "_lib", None)
  monkeypatch.setattr(L, "ABI_VERSION", (major + 1, 0))
  with pytest.raises(ImportError, match="ABI version"):
    L.lib()
  monkeypatch.setattr(L, "_lib", None)
  monkeypatch.setattr(L, "ABI_VERSION", (major, minor + 1))   # the real major, a newer minor
  with pytest.raises(ImportError, match="ABI version"):
    L.lib()


def test_missing_library_fails_loudly(monkeypatch):
  monkeypatch.setattr(L, "_lib", None)
  monkeypatch.setattr(L, "LIB_PATH", "/nonexistent/libtunix_hip.so")
  with pytest.raises(ImportError, match="no CPU fallback"):
    L.lib()


def test_sampling_plan_uses_one_predicate_for_path_and_workspace():
  """top_k None / <= 0 mean "no top-k"; top_k == V is a real top-k of the whole row in the
  reference (jax.lax.top_k(k = V), draw over sorted positions: tunix/generate/sampler.py:118-134)
  and takes the full sort whatever top_p; top_k > V raises as jax.lax.top_k does.  The same
  predicate decides the workspace: a full sort must get the full-row sort's workspace, not the
  (much smaller) segmented top-k one."""
  from tunix_amd.generate.sampler import sampling_plan
  V = 1000
  assert sampling_plan(None, 1.0, V) == (0, "head_draw")
  assert sampling_plan(0, 1.0, V) == (0, "head_draw")
  assert sampling_plan(V, 1.0, V) == (V, "fullsort")
  assert sampling_plan(V, 0.9, V) == (V, "fullsort")
  with pytest.raises(ValueError, match="top_k"):
    sampling_plan(V + 5, 0.9, V)
  assert sampling_plan(None, 0.9, V) == (0, "fullsort")
  assert sampling_plan(50, 0.9, V) == (50, "topk")
  assert sampling_plan(V - 1, 1.0, V) == (V - 1, "topk")
  lib = L.lib()
  # the library treats k >= V like k = 0 when it sizes the segmented workspace: that size is far
  # below what the full sort needs, which is why the host must not pair it with top_p < 1
  B, Vbig = 128, 128256
  small = lib.tnx_sample_topk_ws_bytes(B, Vbig, Vbig)
  assert small == lib.tnx_sample_topk_ws_bytes(B, Vbig, 0)
  assert small < 4 * B * Vbig


def test_threefry_seed_mirrors_jax_with_32_bit_integers():
  from tunix_amd.generate.sampler import _threefry_seed
  assert _threefry_seed(0) == (0, 0)
  assert _threefry_seed(7) == (0, 7)
  assert _threefry_seed(-1) == (0, 0xFFFFFFFF)
  assert _threefry_seed(-2 ** 31) == (0, 0x80000000)
  assert _threefry_seed(2 ** 32 + 5) == (0, 5)


def test_split_k_choice_of_the_decode_linears():
  """The k split the model picks per linear (host logic, no GPU): shapes that fill the device
  run unsplit, few-block shapes split up to 8 ways, and a gate|up linear stays unsplit when the
  split would save at most 7 k-tiles (its epilogue then replaces the finishing pass and the next
  linear's LoRA down-projection); the override wins over everything."""
  import types
  from tunix_amd.model import Runner
  m = Runner.__new__(Runner)
  m.split_k_override = {}
  lin = lambda name, K, N, il=False: types.SimpleNamespace(names=[f"layers.0.{name}"], K=K, N=N, interleave2=il)
  assert m._split_k(lin("wq", 4096, 6144), 128) == 5            # Llama-3.1-8B q|k|v: 48 column blocks
  assert m._split_k(lin("wo", 4096, 4096), 128) == 8
  assert m._split_k(lin("w_down", 14336, 4096), 128) == 8
  assert m._split_k(lin("w_gate", 4096, 28672, True), 128) == 1  # 224 blocks fill the device
  assert m._split_k(lin("w_gate", 1152, 13824, True), 64) == 1   # Gemma3-1B: 108 blocks, a 2-way split saves 4 k-tiles
  assert m._split_k(lin("w_gate", 4096, 2048, True), 64) == 8    # 16 blocks: the split saves 28 k-tiles
  assert m._split_k(lin("wq", 4096, 6144), 8192) == 1            # many rows
  m.split_k_override = {"w_gate": 3}
  assert m._split_k(lin("w_gate", 1152, 13824, True), 64) == 3


@pytest.mark.parametrize("override", [{}, {"wq": 4}])
@pytest.mark.parametrize("rows", [1, 64, 127, 128, 129, 160, 1024, 16384])
def test_partial_planes_have_room_at_every_row_count_of_a_runner(rows, override):
  """A runner of many rows is called with fewer (the last group of prompts): the planes of a linear that splits there fit."""
  import types
  from tunix_amd.model import Runner
  lin = lambda name, K, N, il=False: types.SimpleNamespace(names=[f"l0.{name}"], K=K, N=N, interleave2=il)
  layers = [dict(qkv=lin("wq", 4096, 6144), o=lin("wo", 4096, 4096), gu=lin("w_gate", 4096, 28672, True), down=lin("w_down", 14336, 4096)),
            dict(qkv=lin("wq", 512, 768), o=lin("wo", 512, 512), gu=lin("w_gate", 4096, 2048, True))]
  r = Runner.__new__(Runner)
  r.split_k_override, r.M, r.model = override, rows, types.SimpleNamespace(layers=layers)
  room = r._split_floats()
  for ly in layers:
    for f in ly.values():
      for M in list(range(1, min(rows, 300) + 1)) + [rows]:
        split = r._split_k(f, M)
        assert split == 1 or split * M * f.N <= room, (f.names, M, split)


@pytest.mark.parametrize("groups,S,head_dim,chunks", [
    (1, 4000, 128, 32), (1, 65, 128, 1), (64, 1000, 128, 4), (128, 129, 64, 2), (129, 4000, 128, 1), (255, 4000, 128, 1), (256, 1025, 128, 2), (257, 1024, 64, 1),
    (400, 4000, 64, 2), (401, 4000, 64, 1), (128, 4000, 256, 2), (129, 257, 256, 3), (129, 256, 256, 1), (171, 1025, 256, 4), (171, 1024, 256, 1),
    (200, 3000, 256, 6), (256, 3000, 256, 1), (264, 700, 256, 4), (384, 700, 256, 3), (512, 3000, 256, 1), (513, 700, 256, 3), (640, 700, 256, 2), (901, 3000, 256, 1)])
def test_key_chunks_of_a_decode_step(groups, S, head_dim, chunks):
  from tunix_amd.model import Runner
  assert Runner._key_chunks(groups, S, head_dim) == chunks


@pytest.mark.parametrize("groups,S,head_dim,chunks", [
    (1, 256, 128, 1), (1, 257, 128, 3), (128, 256, 128, 1), (128, 257, 128, 2), (1, 384, 64, 1), (1, 385, 64, 4), (128, 384, 64, 1), (128, 385, 64, 2),
    (1, 256, 256, 2), (64, 288, 256, 3), (256, 1025, 128, 2), (200, 3000, 256, 6)])
def test_key_chunks_of_a_decode_step_without_an_adapter_behind(groups, S, head_dim, chunks):
  """Short contexts are not cut where the merging pass would have nothing else to do; longer ones as ever."""
  from tunix_amd.model import Runner
  assert Runner._key_chunks(groups, S, head_dim, adapter_behind=False) == chunks


def test_chunks_that_a_linear_merges():
  from tunix_amd import ops
  from tunix_amd.model import Runner
  ok = lambda n: ops.qlinear_merged_ok(1, 4096, 4096, 64, 8, 128, n)
  assert ok(Runner.MERGED_CHUNKS) and not ok(Runner.MERGED_CHUNKS + 1)


@pytest.mark.parametrize("M,heads,kv_heads,head_dim,D,S,rank,chunks", [
    (1, 32, 8, 128, 4096, 1536, 64, 12), (1, 32, 8, 128, 4096, 3000, 64, 12), (1, 32, 8, 128, 4096, 8192, 64, 12), (1, 32, 8, 128, 4096, 8193, 64, 29),   # (of 288)
    (1, 32, 8, 128, 4096, 16384, 64, 32), (2, 32, 8, 128, 4096, 16384, 64, 12), (2, 32, 8, 128, 4096, 16385, 64, 16), (3, 32, 8, 128, 4096, 16384, 64, 10),
    (1, 8, 2, 64, 512, 16384, 32, 12), (1, 8, 2, 64, 512, 32768, 32, 12), (1, 8, 2, 64, 512, 32769, 32, 114), (2, 8, 2, 64, 512, 16384, 32, 12), (2, 8, 2, 64, 512, 16385, 32, 57),
    (3, 8, 2, 64, 512, 8192, 32, 12), (3, 8, 2, 64, 512, 8193, 32, 37),
    (1, 32, 8, 128, 4096, 3000, 0, 24),       # no adapter: the merging pass runs
    (1, 32, 8, 128, 4096, 256, 0, 1),
    (1, 64, 8, 128, 8192, 3000, 64, 24),      # sixteen k-tiles a split
    (4, 32, 4, 128, 2048, 3000, 64, 16),      # twelve are more bytes than it merges
    (4, 32, 4, 128, 2048, 1600, 64, 10),      # ... ten, of 160 keys, are not
    (1, 4, 1, 256, 1152, 3000, 32, 24),       # heads of 256
    (1, 32, 8, 128, 4096, 65, 64, 1),
])
def test_key_chunks_in_front_of_the_linear_that_merges_them(M, heads, kv_heads, head_dim, D, S, rank, chunks):
  """Twelve where o merges that many by itself and they are not too long; otherwise as many as fill the device."""
  import math
  import types
  from tunix_amd.model import FusedLinear, Runner
  o = FusedLinear.__new__(FusedLinear)
  o.names, o.K, o.N, o.rp, o.has_lora, o.head, o.interleave2 = ["l0.wo"], heads * head_dim, D, rank, rank > 0, False, False
  r = Runner.__new__(Runner)
  r.split_k_override, r.cfg, r.S = {}, types.SimpleNamespace(num_kv_heads=kv_heads, head_dim=head_dim), S
  r.kv_chunk, r.attn_ws = r._decode_chunk(o, M, S), None
  assert (math.ceil(S / r.kv_chunk) if r.kv_chunk else 1) == chunks
  assert r.kv_chunk % 32 == 0 and (r.merges(o, M) is not None) == (rank > 0 and 1 < chunks <= 12 and o.K < 8192)


@pytest.mark.parametrize("groups,S,width,chunks", [
    (1, 4000, 256, 32), (40, 300, 512, 4), (40, 300, 256, 1), (60, 1000, 512, 4), (85, 2500, 512, 3), (86, 2500, 512, 5), (102, 1025, 512, 5), (96, 1024, 512, 2),
    (103, 2500, 512, 2), (128, 4000, 256, 2), (129, 2500, 512, 3), (129, 1024, 512, 1), (171, 1500, 512, 4), (171, 1500, 256, 1), (171, 2500, 256, 4),
    (32, 256, 512, 8), (8, 256, 320, 8), (8, 256, 256, 1), (33, 256, 512, 2), (32, 224, 512, 2), (32, 257, 512, 3), (193, 4000, 512, 1), (256, 4000, 512, 1), (257, 1000, 512, 3), (257, 100, 128, 1), (340, 600, 512, 3), (341, 1500, 512, 2), (381, 4000, 512, 1)])
def test_key_chunks_of_a_layer_list_step(groups, S, width, chunks):
  from tunix_amd.stack_model import StackRunner
  assert StackRunner._key_chunks(groups, S, width) == chunks


@pytest.mark.parametrize("name,P,first,group,packs", [
    ("tiny_qwen3", 16, (0, 1), 2, False), ("tiny_qwen3", 16, (0, 15), 2, False), ("tiny_qwen3", 256, (0,) * 30 + (200, 200), 32, False),
    ("tiny_qwen3", 256, (0,) * 30 + (240, 240), 32, True),
    ("gemma3_1b", 256, (0, 4), 2, False), ("gemma3_1b", 256, (0, 5), 2, True), ("gemma3_1b", 256, (0, 5), 1, False), ("gemma3_1b", 256, (3, 6), 1, True),
    ("llama31_8b", 128, (0, 1), 2, True), ("llama31_8b", 128, (0, 0), 2, False), ("llama31_8b", 128, (1,), 1, True),
])
def test_prompts_are_packed_where_their_padding_is_worth_a_launch(name, P, first, group, packs):
  import types
  from tunix_amd.generate.sampler import Sampler
  from tunix_amd.model import Runner
  r = Runner.__new__(Runner)
  r.cfg = getattr(config, name)()
  st = types.SimpleNamespace(padded=any(first), first=np.array(first), group=group, num_input_tokens=P)
  assert Sampler.packs(st, r) is packs
  assert not Sampler.packs(st, object())      # a runner that knows padded rows alone


def test_split_k_leaves_no_empty_split_and_goes_on_for_long_contractions():
  import math
  import types
  from tunix_amd.model import Runner
  m = Runner.__new__(Runner)
  m.split_k_override = {}
  lin = lambda name, K, N: types.SimpleNamespace(names=[f"l0.{name}"], K=K, N=N, interleave2=False)
  assert m._split_k(lin("wq", 1152, 1536), 64) == 5            # nine k-tiles, two per split
  assert m._split_k(lin("w_down", 6912, 1152), 64) == 14       # nine column blocks: 126 of 256 compute units, four k-tiles each
  assert m._split_k(lin("w_down", 16384, 1152), 64) == 16
  assert m._split_k(lin("wq", 8192, 512), 1) == 8              # the attention kernel takes eight planes in one round trip
  for kt in range(1, 130):
    for n in (128, 640, 1152, 4096, 12800):
      s = m._split_k(lin("wo", 128 * kt, n), 8)
      assert 1 <= s <= 16 and (s - 1) * math.ceil(kt / s) < kt


def test_a_metric_takes_a_term_with_a_gradient_in_place():
  """What aggregate_loss returns is added to in place by terms that ask for a gradient, and carries it."""
  import torch
  from tunix_amd.rl import common as C
  aux = torch.tensor(2.0, requires_grad=True)
  m = C._metric(torch.tensor([3.0, 4.0]), 1.0)
  m.unreduced_sum += 0.5 * aux
  total = m.compute()
  assert total.item() == 1.0
  total.backward()
  assert aux.grad.item() == 0.125


def test_a_metric_that_left_the_device_is_computed_where_it_is():
  """A saved metric whose numbers are loaded to the host (or were there, or changed their type) takes the tensor operations."""
  import io
  import torch
  from tunix_amd.rl import common as C
  m = C._metric(torch.tensor([3.0, 4.0]), 1.0)
  assert m.compute().item() == 0.75
  f = io.BytesIO()
  torch.save(m, f)
  f.seek(0)
  assert torch.load(f, weights_only=False, map_location="cpu").compute().item() == 0.75   # (written above by this test)
  m.unreduced_sum.data = m.unreduced_sum.data.double()
  assert m.compute().item() == 0.75 and m.compute().dtype == torch.float64
