"""The C-ABI library loads and exports every symbol include/tinygrad_amd.h declares (no GPU call is made)."""
import ctypes, pathlib, re
import pytest
from decode_helpers import many_tile

ROOT = pathlib.Path(__file__).resolve().parent.parent

def _declared():
  text = (ROOT / "include" / "tinygrad_amd.h").read_text()
  text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
  return sorted(set(re.findall(r"\b(tga_\w+)\s*\(", text)))

def test_header_declares_entry_points():
  names = _declared()
  assert "tga_qlinear" in names and "tga_dequant" in names and "tga_grouped_mxfp8_gemm" in names and len(names) >= 30

def test_library_exports_every_declared_symbol():
  lib_path = ROOT / "tinygrad_amd" / "libtinygrad_amd.so"
  if not lib_path.exists(): pytest.fail(f"{lib_path} is missing: run `python -m tinygrad_amd.build`")
  lib = ctypes.CDLL(str(lib_path))
  missing = [n for n in _declared() if not hasattr(lib, n)]
  assert not missing, f"declared in the header but not exported: {missing}"

def test_python_binding_covers_the_header():
  from tinygrad_amd import runtime as rt
  lib = rt.load_library()
  for n in _declared(): assert getattr(lib, n).restype is not None

def test_missing_library_fails_loudly(monkeypatch, tmp_path):
  from tinygrad_amd import runtime as rt
  monkeypatch.setattr(rt, "_lib", None); monkeypatch.setattr(rt, "_LIB_PATH", tmp_path / "nope.so")
  with pytest.raises(RuntimeError, match="no fallback"): rt.load_library()

def test_host_side_argument_checks_without_gpu():
  from tinygrad_amd import moe
  import numpy as np
  assert moe.m_max_for(4096, 8, 128) == 65536                                     # (ceil(T*k/256) + E) * 256, moe_routing.py:89-90
  b = moe.to_bf16_bits(np.array([1.0, 1.00390625, -2.5, 1.01171875], np.float32))     # 1 + 2^-8 ties to even (1.0); 1 + 3*2^-8 rounds up
  np.testing.assert_array_equal(moe.from_bf16_bits(b), np.array([1.0, 1.0, -2.5, 1.015625], np.float32))

def test_moe_feed_forward_refuses_operands_of_other_sizes(monkeypatch):
  """Every operand of the fused feed-forward is looked at before the native call, which reads what the sizes ask for: logits of another width or fewer rows, weights of another K or
  number of experts, and scales, biases or activations that are too small are AssertionErrors; a down projection to another width takes the single steps, which return that width."""
  import numpy as np
  from tinygrad_amd import moe, runtime as rt
  class Lib:
    def tga_moe_feed_forward_plan(self, T, D, I, E, k, need): need._obj.value = 256; return 0
    def tga_malloc(self, p, n): p._obj.value = 1 << 20; return 0
    def tga_moe_feed_forward(self, *a): calls.append("fused"); return 0
    def tga_moe_route(self, *a): calls.append("single"); return 1
  calls, lib = [], Lib()
  monkeypatch.setattr(rt, "lib", lambda: lib)
  monkeypatch.setattr(rt.Buffer, "__del__", lambda self: None)
  T, D, I, E, k = 40, 512, 256, 8, 2
  def buf(shape, dtype): return rt.Buffer(shape, dtype, ptr=4096)
  good = dict(inp=((T, D), np.uint16), logits=((T, E), np.float32), gq=((E, 2 * I, D), np.uint8), ge=((E, 2 * I, D // 32), np.uint8), gb=((E, 2 * I), np.float32),
              dq=((E, D, I), np.uint8), de=((E, D, I // 32), np.uint8), db=((E, D), np.float32))
  def call(**other):
    b = {n: buf(*v) for n, v in {**good, **other}.items()}
    return moe.moe_feed_forward(b["inp"], b["logits"], k, (b["gq"], b["ge"]), b["gb"], (b["dq"], b["de"]), b["db"])
  assert call().shape == (T, D) and calls == ["fused"]
  for other in (dict(logits=((T, E // 2), np.float32)), dict(logits=((T - 1, E), np.float32)), dict(logits=((T, E), np.float16)), dict(inp=((T, D), np.uint8)),
                dict(gq=((E, 2 * I, D // 2), np.uint8)), dict(dq=((E, D, I // 2), np.uint8)), dict(dq=((E // 2, D, I), np.uint8)), dict(dq=((E, D, 2 * I), np.uint8)),
                dict(ge=((E, 2 * I, D // 64), np.uint8)), dict(de=((E // 2, D, I // 32), np.uint8)), dict(gb=((E, I), np.float32)), dict(db=((E // 2, D), np.float32))):
    with pytest.raises(AssertionError): call(**other)
  assert calls == ["fused"]
  with pytest.raises(RuntimeError): call(dq=((E, 256, I), np.uint8))               # (the library above refuses the single steps' first call)
  assert calls == ["fused", "single"]

def test_prefill_step_refuses_what_its_kernels_cannot_address():
  """Rows whose activations lie beyond 2^32 values, expert counts and gating kinds that do not exist and expert formats without a kernel are errors before anything is launched (pointers here lead nowhere)."""
  from tinygrad_amd import runtime as rt
  L = rt.load_library()
  NAMES = "NBLOCKS DIM HEADS KV HD MAXCTX EMB EMB_TYPE ROPE EXPERTS TOPK GATING NORM_TOPK QKNORM HIDDEN DENSE_HIDDEN EPS_BITS SCALE_BITS".split()
  good = dict(NBLOCKS=1, DIM=2048, HEADS=16, KV=16, HD=128, MAXCTX=1 << 20, EMB=4096, EMB_TYPE=2, ROPE=4096, EXPERTS=64, TOPK=8, GATING=1, NORM_TOPK=0, QKNORM=0, HIDDEN=1024, DENSE_HIDDEN=0, EPS_BITS=0, SCALE_BITS=0)
  def call(rows, words, types=(39, 39), **other):
    m = (ctypes.c_int64 * len(NAMES))(*[{**good, **other}[n] for n in NAMES])
    b = (ctypes.c_int64 * 21)(*([4096] * 6 + [1] + [4096] * 8 + [1, 1, 1, 1, *types]))
    assert L.tga_prefill_step(m, b, 4096, 1, rows, 0, 4096, 4096, None) != 0
    assert words in L.tga_last_error().decode(), L.tga_last_error()
  call((1 << 20) - 1, "more than a step takes")                                    # 2^20 rows x 8 experts x 1024 values
  call((1 << 19) + 8, "more than a step takes")
  call((1 << 19) + 8, "more than a step takes", EXPERTS=0, HIDDEN=8192)
  call(1 << 19, "more than a step takes", DIM=8192, HIDDEN=256)
  call(32, "of 64 experts", TOPK=0); call(32, "of 4 experts", EXPERTS=4)
  call(32, "ExpertGating 0", GATING=0); call(32, "ExpertGating 5", GATING=5)
  call(32, "experts of block 0", types=(39, 22)); call(32, "experts of block 0", types=(12, 39), DIM=2048 + 128)

@pytest.mark.gpu
def test_freed_blocks_are_kept_and_given_back(gpu):
  """tga_free keeps a block for later requests of its size class, never hands it out while kernels may still use it, and tga_trim gives everything back: results computed into
  blocks that were freed and allocated again many times over are right, and the library still allocates afterwards."""
  import numpy as np
  n = 3 << 20
  src = [gpu.Buffer.from_numpy(np.full(n, i, np.uint8)) for i in range(4)]
  streams = [gpu.Stream() for _ in range(2)]
  for r in range(40):                                                              # more rounds than dirty blocks are collected before they are settled
    outs = [gpu.Buffer((n,), np.uint8) for _ in range(4)]
    for i, o in enumerate(outs): gpu.check(gpu.lib().tga_copy_kernel(o.ptr, src[(i + r) % 4].ptr, n, streams[i % 2].handle))
    if r % 7 == 0:
      gpu.synchronize()
      for i, o in enumerate(outs): assert (o.numpy() == (i + r) % 4).all()
  gpu.check(gpu.lib().tga_trim())
  b = gpu.Buffer((n,), np.uint8); gpu.check(gpu.lib().tga_copy_kernel(b.ptr, src[3].ptr, n, None)); gpu.synchronize()
  assert (b.numpy() == 3).all()

@pytest.mark.gpu
def test_a_capture_gets_no_block(gpu):
  """A block that tga_free keeps is never handed to a thread whose own capture is open: the recorded launches would use it after the call that took it gave it back."""
  import numpy as np
  n = 5 << 20
  stream, src, dst = gpu.Stream(), gpu.Buffer((4096,), np.uint8).zero_(), gpu.Buffer((4096,), np.uint8)
  bufs = [gpu.Buffer((n,), np.uint8) for _ in range(9)]
  kept = {b.ptr for b in bufs}
  bufs.clear()
  gpu.Buffer((n,), np.uint8)                                                       # (settles the class: its blocks may be handed out from here on)
  with pytest.raises(RuntimeError, match="captures"):
    with gpu.Graph(stream):
      gpu.check(gpu.lib().tga_copy_kernel(dst.ptr, src.ptr, 4096, stream.handle))
      gpu.Buffer((n,), np.uint8)
  gpu.check(gpu.lib().tga_copy_kernel(dst.ptr, src.ptr, 4096, stream.handle)); stream.synchronize()
  assert gpu.Buffer((n,), np.uint8).ptr in kept                                    # the capture is over: kept blocks are handed out again

@pytest.mark.parametrize("t", [2, 12], ids=["Q4_0", "Q4_K"])
def test_tall_tiles_have_rows_of_1024_values_or_more(t):
  """Shorter rows are outside what the rule was measured on, and rows of 256 values shorter than what the kernel's touches bring (their address lay in front of the row)."""
  for k in (256, 512, 768): assert many_tile(t, (28672,), 1023, k)[0] != (512, 128) and many_tile(t, (14336, 14336), 2047, k, 2)[0] != (512, 128)
  assert many_tile(t, (28672,), 1023, 1024) == ((512, 128), 1)

@pytest.mark.parametrize("t,m,n,k,epi,tall", [(2, 1261, 9296, 1280, 2, False), (2, 1023, 17312, 1280, 2, False), (2, 1024, 12464, 1024, 2, True), (2, 2047, 8784, 1536, 2, True), (2, 1024, 22768, 1024, 0, False),
                                              (12, 1024, 18896, 1024, 2, False), (12, 768, 24288, 1536, 2, False), (12, 1024, 18672, 2048, 2, True)])
def test_tall_tiles_of_several_rounds_and_few_steps(t, m, n, k, epi, tall):
  """Two and more rounds of tall tiles of few steps, the last one less than 75 or 78 % full, were 2 - 7 % slower than the other tiles: taken from there on."""
  assert (many_tile(t, (n, n) if epi == 2 else (n,), m, k, epi)[0] == (512, 128)) == tall
