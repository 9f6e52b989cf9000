"""Wait states around vector instructions that are written in assembly, in the listing of the built library: the MFMAs of qgemm_pre.h, and the
maxima of attention.hip, which lane swaps read.

The compiler does not look inside assembly: it keeps no distance between such an MFMA and the vector instructions that it places around
it itself (copies of an operand, reads of a finished accumulator), nor between such a maximum and a swap.  Required, in instruction slots of
which `s_nop N` is N + 1: two between a vector write and an MFMA that reads it, eight between a 16x16x32 bf16 MFMA (four passes) and anything
else that reads or overwrites its result, three until its addend's registers are overwritten; two between a vector write and a permlane swap
of the register.  These are the distances that the compiler keeps around its own instructions.
"""
import os
import re
import shutil
import subprocess
from collections import defaultdict

import pytest

from tunix_amd import _lib

OBJDUMP = shutil.which("llvm-objdump") or "/opt/rocm/llvm/bin/llvm-objdump"
KERNELS = ("qgemm_pre_kernel", "attn_wg_kernel")
VALU_TO_MFMA, MFMA_TO_OTHER, ADDEND_TO_WRITE, VALU_TO_SWAP = 2, 8, 3, 2

LINE = re.compile(r"^\s+([a-z_]\w+)\s*(.*?)\s*//\s*([0-9A-Fa-f]+):")
TARGET = re.compile(r"<[^>+]+(?:\+0x([0-9a-f]+))?>\s*$")


def registers(operand):
  m = re.fullmatch(r"-?\|?([va])(\d+)\|?", operand)
  if m:
    return {(m[1], int(m[2]))}
  m = re.fullmatch(r"-?\|?([va])\[(\d+):(\d+)\]\|?", operand)
  return {(m[1], i) for i in range(int(m[2]), int(m[3]) + 1)} if m else set()


class Instruction:
  def __init__(self, line, op, operands, address):
    self.text, self.op, self.address = line.split("//")[0].strip(), op, address
    ops = [registers(o.split(" ")[0]) for o in re.split(r",\s*(?![^\[]*\])", operands)] if operands else []
    self.mfma = op.startswith("v_mfma")
    self.valu = op.startswith("v_") and not self.mfma
    load = ("load" in op or "read" in op) and not self.valu and " lds" not in operands
    writes_first = self.mfma or load or (self.valu and not op.startswith(("v_cmp", "v_readfirstlane", "v_readlane", "v_nop")))
    self.writes = set(ops[0]) if writes_first and ops else set()
    if "swap" in op and self.valu:
      self.writes |= ops[1]
    # (an accumulator that is a source too, or a swap's, is in both sets)
    self.reads = set().union(*(ops[1:] if writes_first else ops)) if ops else set()
    if "swap" in op or op.startswith(("v_fmac", "v_mac", "v_dot")):
      self.reads |= self.writes
    self.ab, self.addend = (ops[1] | ops[2], ops[3]) if self.mfma else (set(), set())
    self.slots = int(operands, 0) + 1 if op == "s_nop" else 1
    m = TARGET.search(line) if op.startswith(("s_branch", "s_cbranch")) else None
    self.target = int(m[1] or "0", 16) if m else None   # bytes behind the function's first instruction


def parse(listing):
  out = []
  for line in listing.splitlines():
    m = LINE.match(line)
    if m:
      out.append(Instruction(line, m[1], m[2], int(m[3], 16)))
  return out


def too_close(code):
  """[(slots between, slots needed, first, second)] over all paths through the function."""
  at = {c.address: i for i, c in enumerate(code)}
  before = defaultdict(list)
  for i, c in enumerate(code):
    if c.target is not None:
      before[at[code[0].address + c.target]].append(i)
    if c.op not in ("s_branch", "s_endpgm", "s_setpc_b64") and i + 1 < len(code):
      before[i + 1].append(i)
  found = []
  for i, c in enumerate(code):
    if not (c.mfma or c.writes or c.reads):
      continue
    touches, seen, paths = c.writes | c.reads, {}, [(j, 0) for j in before[i]]
    while paths:
      j, slots = paths.pop()
      if seen.get(j, 99) <= slots:
        continue
      seen[j] = slots
      p = code[j]
      need = 0
      if c.mfma and p.valu and p.writes & (c.ab | c.addend):
        need = VALU_TO_MFMA
      elif p.mfma and not c.mfma:
        if p.writes & touches:
          need = MFMA_TO_OTHER
        elif p.addend & c.writes:
          need = ADDEND_TO_WRITE
      elif p.mfma and c.mfma and p.writes & c.ab:
        need = MFMA_TO_OTHER
      elif c.op.startswith("v_permlane") and p.valu and p.writes & touches:
        need = VALU_TO_SWAP
      if slots < need:
        found.append((slots, need, p.text, c.text))
      if slots + p.slots < MFMA_TO_OTHER:
        paths += [(k, slots + p.slots) for k in before[j]]
  return found


@pytest.fixture(scope="module")
def listings(tmp_path_factory):
  if not os.path.exists(OBJDUMP):
    pytest.skip("no llvm-objdump")
  where = tmp_path_factory.mktemp("code")
  shutil.copy(_lib.LIB_PATH, where / "lib.so")
  subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=where, check=True, stdout=subprocess.DEVNULL)
  out = {}
  for f in sorted(where.glob("*gfx950")):
    names = [n for n in re.findall(r"(\S+)$", subprocess.run([OBJDUMP, "--syms", str(f)], check=True, capture_output=True, text=True).stdout, re.M)
             if any(k in n for k in KERNELS) and not n.endswith(".kd")]
    if names:
      text = subprocess.run([OBJDUMP, "-d", "--mcpu=gfx950", "--disassemble-symbols=" + ",".join(names), str(f)],
                            check=True, capture_output=True, text=True).stdout
      for part in re.split(r"^(?=[0-9a-f]{8,} <)", text, flags=re.M)[1:]:
        out[re.match(r"[0-9a-f]+ <(\S+)>", part)[1]] = part
  return out


@pytest.mark.parametrize("kernel", KERNELS)
def test_wait_states_around_assembly_mfmas(listings, kernel):
  mine = {n: t for n, t in listings.items() if kernel in n}
  assert mine
  for name, text in mine.items():
    code = parse(text)
    assert sum(c.mfma for c in code) >= 32, name
    assert kernel != "attn_wg_kernel" or sum(c.op.startswith("v_permlane") for c in code) >= 4, name
    assert not too_close(code), (name, too_close(code)[:3])


@pytest.mark.parametrize("what,lines,bad", [
    ("copy of an operand", ["v_accvgpr_read_b32 v7, a73", "s_lshl_b32 s16, s16, 7", "v_mfma_f32_16x16x32_bf16 a[4:7], v[4:7], v[62:65], a[4:7]"], 1),
    ("the same with its wait", ["v_accvgpr_read_b32 v7, a73", "s_nop 1", "v_mfma_f32_16x16x32_bf16 a[4:7], v[4:7], v[62:65], a[4:7]"], 0),
    ("addend written", ["v_mul_f32_e32 v5, v1, v2", "v_mfma_f32_16x16x32_bf16 v[4:7], v[8:11], v[12:15], v[4:7]"], 1),
    ("result read", ["v_mfma_f32_16x16x32_bf16 a[0:3], v[0:3], v[4:7], a[0:3]", "s_nop 6", "v_accvgpr_read_b32 v9, a3"], 1),
    ("result read late", ["v_mfma_f32_16x16x32_bf16 a[0:3], v[0:3], v[4:7], a[0:3]", "s_nop 7", "v_accvgpr_read_b32 v9, a3"], 0),
    ("result overwritten", ["v_mfma_f32_16x16x32_bf16 v[0:3], v[4:7], v[8:11], 0", "s_nop 3", "v_add_u32_e32 v2, v30, v31"], 1),
    ("result stored", ["v_mfma_f32_16x16x32_bf16 v[0:3], v[4:7], v[8:11], 0", "ds_write_b128 v20, v[0:3] offset:16"], 1),
    ("result an operand", ["v_mfma_f32_16x16x32_bf16 v[0:3], v[4:7], v[8:11], 0", "v_mfma_f32_16x16x32_bf16 v[12:15], v[0:3], v[8:11], 0"], 1),
    ("accumulators in turn", ["v_mfma_f32_16x16x32_bf16 a[0:3], v[4:7], v[8:11], a[0:3]"] * 3, 0),
    ("operand reloaded", ["v_mfma_f32_16x16x32_bf16 a[0:3], v[4:7], v[8:11], a[0:3]", "ds_read_b128 v[4:7], v20"], 0),
    ("addend reused", ["v_mfma_f32_16x16x32_bf16 v[0:3], v[4:7], v[8:11], v[12:15]", "s_nop 1", "v_mov_b32_e32 v12, v40"], 1),
    ("swap of a maximum", ["v_max_f32 v8, v1, v2", "v_permlane16_swap_b32_e32 v8, v9"], 1),
    ("swap with its copy", ["v_max3_f32 v8, v1, v2, v3", "v_mov_b32_e32 v9, v8", "s_nop 0", "v_permlane32_swap_b32_e32 v8, v9"], 1),
    ("the same with its wait", ["v_max3_f32 v8, v1, v2, v3", "v_mov_b32_e32 v9, v8", "s_nop 1", "v_permlane32_swap_b32_e32 v8, v9"], 0),
    ("swap of other registers", ["v_max_f32 v8, v1, v2", "v_permlane16_swap_b32_e32 v10, v9"], 0),
    ("round a loop", ["v_mfma_f32_16x16x32_bf16 a[0:3], v[4:7], v[8:11], a[0:3]", "v_add_u32_e32 v4, v20, v21",
                      "s_cbranch_scc1 65533 // 0000000000000008: BF85FFFD <f>"], 1),
])
def test_planted_distances_are_found(what, lines, bad):
  listing = "\n".join("\t" + (l if "//" in l else f"{l} // {4 * i:016X}: 00000000") for i, l in enumerate(lines))
  assert bool(too_close(parse(listing))) == bool(bad), what
