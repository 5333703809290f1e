"""Guards for the inline-assembly loads of csrc/qgemm_dma.hip and csrc/qgemm_wp.hip (CPU only: the files are compiled to gfx950 assembly and read as text).

The kernel requests activations with `global_load_dwordx4` written as inline assembly and waits for them with a hand-counted `s_waitcnt vmcnt(n)`, so
that weight pieces issued behind them stay in flight.  The compiler takes the destination registers for valid as soon as the request is issued: if it
ever copies or reuses one of them between the request and the wait, the kernel computes with stale data and nothing fails loudly.  These checks read
the generated code in layout order, which is how the requests, the wait and the first use follow each other in every build so far; a failure means
"look at the assembly", not necessarily "wrong code"."""
import os, pathlib, re, subprocess, tempfile
import pytest
from tinygrad_amd import build as tb

SOURCES = {"qgemm_dma.hip": (r"^(_Z16qgemm_dma_kernelI\w+EEv5QArgsii):", 19), "qgemm_wp.hip": (r"^(_Z15qgemm_wp_kernelI\w+EEv5QArgsii):", 12)}

def _regs(line: str) -> set:
  out, code = set(), line.split(";")[0]
  for m in re.finditer(r"\bv\[(\d+):(\d+)\]", code): out.update(range(int(m.group(1)), int(m.group(2)) + 1))
  for m in re.finditer(r"\bv(\d+)\b", code): out.add(int(m.group(1)))
  return out

@pytest.fixture(scope="module", params=sorted(SOURCES))
def kernels(request):
  try: hipcc = tb._hipcc()
  except RuntimeError: pytest.skip("hipcc not found")
  pattern, at_least = SOURCES[request.param]
  with tempfile.TemporaryDirectory() as d:
    out = pathlib.Path(d) / (request.param + ".s")
    r = subprocess.run([hipcc, *tb.HIPCC_FLAGS, "--cuda-device-only", "-S", str(tb.CSRC / request.param), "-o", str(out)], capture_output=True, text=True)
    if r.returncode != 0: pytest.fail(f"hipcc -S failed:\n{r.stderr[-2000:]}")
    text = out.read_text()
  ks = {}
  for name in re.findall(pattern, text, re.M):
    ks[name] = text[text.index("\n" + name + ":"):text.index(".set " + name + ".uses_flat_scratch")].split("\n")
  assert len(ks) >= at_least, sorted(ks)
  return text, ks

def test_no_scratch(kernels):
  """The register sets that hold requests in flight must be registers: a kernel that spills keeps them in memory."""
  text, ks = kernels
  for name in ks:
    m = re.search(r"\.set " + re.escape(name) + r"\.private_seg_size, (\d+)", text)
    assert m and int(m.group(1)) == 0, (name, m and m.group(1))

def _touches_in_flight(L):
  """Forward data flow over the kernel's basic blocks: a request (`global_load_dwordx4 v[a:b]`, only written as inline assembly in this file) puts its destination
  registers in flight; the source passes them through an asm statement marked "; landed" right behind the hand-counted wait, which lands them all (the wait itself is a
  switch over immediates that the compiler lowers to a tree of branches with paths no run takes, so it cannot serve as the landing point of a path-insensitive
  analysis); an instruction that names a register in flight - other than a request that overwrites it - is a finding.  Returns the findings as (line number, text)."""
  ins = []                                                                     # (line index, text) of instructions; labels -> index of the next instruction
  labels = {}
  in_asm, has_marks = False, any(l.strip().startswith(";;#ASMSTART") for l in L)   # (hand-made listings carry no ASMSTART / ASMEND: every request counts there)
  for i, l in enumerate(L):
    m = re.match(r"(\.LBB\d+_\d+):", l)
    if m: labels[m.group(1)] = len(ins); continue
    if l.strip().startswith(";;#ASMSTART"): in_asm = True; continue
    if l.strip().startswith(";;#ASMEND"): in_asm = False; continue
    if l.strip() == "; landed": ins.append((i, "; landed")); continue
    t = l.split(";")[0].strip()
    if not l.startswith("\t") or not t or t.startswith("."): continue
    # a 16-byte load that the compiler wrote (it places that load's wait itself) is an ordinary instruction here, not a request
    if has_marks and not in_asm and t.startswith("global_load_dwordx4"): t = "compiler_" + t
    ins.append((i, t))
  n = len(ins)
  succ = [[] for _ in range(n)]
  for k, (_, t) in enumerate(ins):
    op = t.split()[0]
    if op == "s_endpgm": continue
    if op == "s_branch": succ[k].append(labels[t.split()[1]]); continue
    if op.startswith("s_cbranch"): succ[k].append(labels[t.split()[1]])
    if k + 1 < n: succ[k].append(k + 1)
  state = [None] * n                                                           # registers in flight BEFORE instruction k
  state[0] = frozenset()
  work, found = [0], {}
  while work:
    k = work.pop()
    cur, (li, t) = state[k], ins[k]
    m = re.match(r"global_load_dwordx4 v\[(\d+):(\d+)\]", t)
    if m: out = cur | frozenset(range(int(m.group(1)), int(m.group(2)) + 1))   # (its address registers are read at issue: not a use of data in flight)
    elif t == "; landed": out = frozenset()
    else:
      if _regs(t) & cur: found[li + 1] = t
      out = cur
    for j in succ[k]:
      new = out if state[j] is None else state[j] | out
      if new != state[j]: state[j] = new; work.append(j)
  return sorted(found.items())

def test_requests_in_flight_are_not_touched(kernels):
  """Every kernel of the file, K <= 4096 (requests in the prologue) and K > 4096 (one request site in the stage loop, waited for in the next pass)."""
  _, ks = kernels
  for name, L in ks.items():
    assert any("global_load_dwordx4" in l for l in L), name
    bad = _touches_in_flight(L)
    assert not bad, (name, bad[:5])

def test_the_check_itself():
  """The data-flow check on hand-made listings: a copy of a register in flight is found on a straight path, around a loop's back edge and behind a branch; uses behind
  the landing mark and reuse of the request's address registers are not."""
  ok = ["\tglobal_load_dwordx4 v[4:7], v[4:5], off", "\ts_cbranch_scc1 .LBB0_2", "\tv_mov_b32_e32 v9, v1", ".LBB0_2:", "\ts_waitcnt vmcnt(0)", "\t; landed", "\tv_mov_b32_e32 v8, v5", "\ts_endpgm"]
  assert _touches_in_flight(ok) == []
  straight = ["\tglobal_load_dwordx4 v[4:7], v[2:3], off", "\tv_mov_b32_e32 v8, v5", "\t; landed", "\ts_endpgm"]
  assert [t for _, t in _touches_in_flight(straight)] == ["v_mov_b32_e32 v8, v5"]
  branch = ["\tglobal_load_dwordx4 v[4:7], v[2:3], off", "\ts_cbranch_scc1 .LBB0_2", "\t; landed", "\ts_branch .LBB0_3", ".LBB0_2:", "\tv_add_u32_e32 v6, v1, v2", "\t; landed", ".LBB0_3:", "\ts_endpgm"]
  assert [t for _, t in _touches_in_flight(branch)] == ["v_add_u32_e32 v6, v1, v2"]
  loop = [".LBB0_1:", "\tv_mov_b32_e32 v9, v4", "\t; landed", "\tds_write_b128 v1, v[4:7]", "\tglobal_load_dwordx4 v[4:7], v[2:3], off", "\ts_cbranch_scc1 .LBB0_1", "\t; landed", "\ts_endpgm"]
  assert [t for _, t in _touches_in_flight(loop)] == ["v_mov_b32_e32 v9, v4"]

def test_wave_private_loop_keeps_its_ring_in_flight(kernels):
  """qgemm_wp.hip counts its direct-to-LDS pieces by hand; a compiler-placed `s_waitcnt vmcnt(0)` inside the row-group loop (it puts one in front of an LDS atomic
  builtin, for instance, because it cannot tell the counters from the rings) would empty the ring once per group.  Inside the loop of the SwiGLU
  instantiations every vector-memory wait must be one of the source's own (between ASMSTART / ASMEND); the others also hold the residual load of the
  summing wave, which the compiler waits for."""
  _, ks = kernels
  names = [n for n in ks if "qgemm_wp_kernel" in n]
  if not names: pytest.skip("not the wave-private source")
  checked = 0
  for name in names:
    m = re.match(r"_Z15qgemm_wp_kernelILi\d+ELb([01])ELb([01])E", name)
    if m.group(2) == "0": continue                                           # (plain, residual, q / k / v)
    L = ks[name]
    start = max(i for i, l in enumerate(L) if "This Loop Header: Depth=1" in l)
    inside_asm, bad = False, []
    for i in range(start, len(L)):
      t = L[i].strip()
      if t.startswith(";;#ASMSTART"): inside_asm = True
      elif t.startswith(";;#ASMEND"): inside_asm = False
      elif t.startswith("s_waitcnt") and "vmcnt" in t and not inside_asm and i < len(L) - 6: bad.append((i, t))
    assert not bad, (name, bad)
    checked += 1
  assert checked >= 4

def _wide_loop(L):
  """Instructions of a wide-tile kernel's loop over K, [(text, written by hand)]: the backward branch whose span holds sixteen requests into LDS."""
  ins, by_hand, at = [], False, {}
  for l in L:
    t = l.strip()
    m = re.match(r"(\.LBB\d+_\d+):", t)
    if m: at[m.group(1)] = len(ins)
    elif t.startswith(";;#ASMSTART"): by_hand = True
    elif t.startswith(";;#ASMEND"): by_hand = False
    elif t and not t.startswith((";", ".")):
      ins.append((t.split(";")[0].strip(), by_hand))
      m = re.match(r"s_cbranch\w+ (\.LBB\d+_\d+)$", ins[-1][0])
      if m and m.group(1) in at and sum(" lds" in x for x, _ in ins[at[m.group(1)]:]) == 16: return ins[at[m.group(1)]:]
  raise AssertionError("no loop with sixteen requests into LDS")

def _wide_findings(ins):
  """What would break or empty the loop's pipeline: spills, a wait of the compiler's that a request of this half has to land for, a half without its eight requests into LDS and its hand-written
  wait for all of them in front of the barrier."""
  bad, issued, into_lds, halves, waited = [], 0, 0, [], False
  for t, by_hand in ins:
    if t.startswith("scratch_"): bad.append(t)
    elif t.startswith("buffer_load"): issued += 1; into_lds += " lds" in t; waited = False
    elif t.startswith("s_waitcnt") and "vmcnt" in t:
      n = int(re.search(r"vmcnt\((\d+)\)", t).group(1))
      if by_hand: waited = n == 0 and "lgkmcnt(0)" in t; issued = 0 if n == 0 else issued
      elif issued > n: bad.append(f"{t} behind {issued} requests")
    elif t == "s_barrier":
      if not (by_hand and waited): bad.append("a barrier without its wait")
      halves.append(into_lds); into_lds = 0
  if halves != [8, 8] or into_lds: bad.append(f"requests into LDS per half: {halves}, {into_lds} behind the last barrier")
  return bad

def test_wide_tiles_keep_their_requests_in_flight():
  """qgemm_wide_kernel (csrc/qgemm_rows.h) fills one half of its LDS by requests that write it themselves while it reads the other, and waits for them by hand in front of each of its two barriers."""
  try: hipcc = tb._hipcc()
  except RuntimeError: pytest.skip("hipcc not found")
  with tempfile.TemporaryDirectory() as d:
    out = pathlib.Path(d) / "rows.s"
    r = subprocess.run([hipcc, *tb.HIPCC_FLAGS, "--cuda-device-only", "-S", str(tb.CSRC / "qgemm_rows_a.hip"), "-o", str(out)], capture_output=True, text=True)
    if r.returncode != 0: pytest.fail(f"hipcc -S failed:\n{r.stderr[-2000:]}")
    text = out.read_text()
  names = re.findall(r"^(_Z17qgemm_wide_kernelI\w+):", text, re.M)
  assert len(names) == 2, names
  for name in names:
    ins = _wide_loop(text[text.index("\n" + name + ":"):text.index(".set " + name + ".uses_flat_scratch")].split("\n"))
    assert sum(t.startswith("v_mfma") for t, _ in ins) == 256, name
    assert not (bad := _wide_findings(ins)), (name, bad[:5])
  good = ins
  at = next(i for i, (t, _) in enumerate(good) if t == "s_barrier")
  assert _wide_findings(good[:at - 1] + good[at:])                                  # (the wait gone)
  assert _wide_findings(good[:at - 1] + [("s_waitcnt vmcnt(3)", False)] + good[at - 1:])
  assert _wide_findings(good[:9] + [("scratch_load_dword v1, off, off", False)] + good[9:])

def test_tall_tiles_wait_only_by_hand():
  """qgemm_tall_kernel (csrc/qgemm_tall.hip): its loop over K holds no spill and no wait for vector memory but the four in front of its barriers, which leave the younger requests under way; a request
  into LDS never follows the write of m0, where it goes, directly (one wait state lies between them, which the compiler sees to in its own code and not in inline assembly)."""
  try: hipcc = tb._hipcc()
  except RuntimeError: pytest.skip("hipcc not found")
  with tempfile.TemporaryDirectory() as d:
    out = pathlib.Path(d) / "tall.s"
    r = subprocess.run([hipcc, *tb.HIPCC_FLAGS, "--cuda-device-only", "-S", str(tb.CSRC / "qgemm_tall.hip"), "-o", str(out)], capture_output=True, text=True)
    if r.returncode != 0: pytest.fail(f"hipcc -S failed:\n{r.stderr[-2000:]}")
    text = out.read_text()
  names = re.findall(r"^(_Z17qgemm_tall_kernelI\w+):", text, re.M)
  assert len(names) == 4, names
  for name in names:
    lines = [l.split(";")[0].strip() for l in text[text.index("\n" + name + ":"):text.index(".set " + name + ".uses_flat_scratch")].split("\n")]
    at = {l[:-1]: i for i, l in enumerate(lines) if re.match(r"\.LBB\d+_\d+:$", l)}
    loops = [lines[at[m.group(1)]:i] for i, l in enumerate(lines) if (m := re.match(r"s_cbranch\w+ (\.LBB\d+_\d+)$", l)) and at.get(m.group(1), i) < i]
    loops = [x for x in loops if sum(t.startswith("v_mfma") for t in x) == 256]
    assert len(loops) == 1, name
    assert [t for t in loops[0] if "vmcnt" in t] == ["s_waitcnt vmcnt(%d)" % n for n in (14, 15, 3, 2)], name
    assert not any(t.startswith("scratch_") for t in loops[0]) and sum(t == "s_barrier" for t in loops[0]) == 4 and sum(" lds" in t for t in loops[0]) == 21, name
    code = [l for l in lines if l and not l.startswith((".", "s_waitcnt"))]
    after = [t for m0, t in zip(code, code[1:]) if re.search(r"\bm0\b", m0)]
    assert len(after) == sum(t.endswith(" lds") for t in code) >= 21 and not any(t.endswith(" lds") for t in after), name      # (and m0 has no other use)
