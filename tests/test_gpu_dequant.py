"""GPU block dequant vs the oracle: bit-exact (the bar for ggml_data_to_tensor, tinygrad/llm/gguf.py:23-119)."""
import numpy as np, pytest
from oracle import ggml as og
from tinygrad_amd import synth
from tinygrad_amd.runtime import GGML_QUANT

pytestmark = pytest.mark.gpu
TYPES = [2, 3, 6, 7, 8, 12, 13, 14, 18, 21, 22, 23, 39, 41]

def _gpu_dequant(gpu, data, n, t, dtype=np.float32):
  from tinygrad_amd.gguf import ggml_data_to_tensor
  return ggml_data_to_tensor(data, n, t, out_dtype=dtype).numpy()

from conftest import golden_kats

@pytest.mark.parametrize("name,t,n,block,exp", golden_kats(), ids=[k[0] for k in golden_kats()])
def test_golden_fixture_vectors(gpu, name, t, n, block, exp):
  """The committed fixture of the reference tests' vectors through the device kernel, bit for bit."""
  assert _gpu_dequant(gpu, block, n, t).tobytes() == exp.tobytes()

def test_q8_0_reference_kat(gpu):
  # test/unit/test_gguf.py:36-40
  block = np.frombuffer(np.float16(2.0).tobytes() + np.arange(1, 33, dtype=np.int8).tobytes(), dtype=np.uint8).copy()
  np.testing.assert_array_equal(_gpu_dequant(gpu, block, 32, 8), np.arange(1, 33, dtype=np.float32) * 2.0)

def test_mxfp4_reference_kats(gpu):
  # test/unit/test_gguf.py:42-48
  block = np.array([0x80] + list(range(16)), dtype=np.uint8)
  exp = np.array([0., 1., 2., 3., 4., 6., 8., 12., -0., -1., -2., -3., -4., -6., -8., -12.] + [0.] * 16, dtype=np.float32)
  out = _gpu_dequant(gpu, block, 32, 39)
  assert out.tobytes() == exp.tobytes()          # includes the sign of -0.0
  # test/unit/test_gguf.py:89-105 (a real GLM-4.7-Flash block)
  block = np.array([0x7a, 0x29, 0xab, 0x61, 0x10, 0x21, 0x02, 0x4a, 0x15, 0xca, 0x05, 0x01, 0x9b, 0x39, 0x0b, 0x0b, 0x1c], dtype=np.uint8)
  exp = np.array([-0.015625, -0.046875, 0.015625, 0.0, 0.015625, 0.03125, -0.03125, 0.09375, -0.03125, 0.09375, 0.015625, -0.046875,
                  -0.015625, -0.046875, -0.046875, -0.0625, 0.03125, -0.03125, 0.125, 0.015625, 0.03125, 0.0, 0.0625, 0.015625,
                  -0.0625, 0.0, 0.0, -0.015625, 0.046875, 0.0, 0.0, 0.015625], dtype=np.float32)
  np.testing.assert_array_equal(_gpu_dequant(gpu, block, 32, 39), exp)

@pytest.mark.parametrize("t", TYPES)
def test_random_blocks_bit_exact(gpu, t):
  rng = np.random.default_rng(100 + t)
  nel, nby = GGML_QUANT[t]
  nb = 4096 + 37
  data = rng.integers(0, 256, size=(nb, nby), dtype=np.uint8)       # every byte random: includes NaN/Inf/subnormal fp16 scales
  if t == 39: data[:8, 0] = [0, 1, 2, 3, 254, 255, 127, 128]       # E8M0 corner cases incl. the two fp32-subnormal scales
  with np.errstate(all="ignore"): ref = og.ggml_data_to_tensor(data, nb * nel, t)
  out = _gpu_dequant(gpu, data, nb * nel, t)
  same = (out.view(np.uint32) == ref.view(np.uint32)) | (np.isnan(out) & np.isnan(ref))
  assert same.all(), f"type {t}: {np.count_nonzero(~same)} of {same.size} elements differ"

@pytest.mark.parametrize("t", TYPES)
def test_model_path_fp16_cast(gpu, t):
  """TGA_F16 output == RNE fp16 cast of the float32 dequant (the HALF=1 cast at tinygrad/llm/model.py:376)."""
  rng = np.random.default_rng(200 + t)
  data = synth.random_blocks(rng, t, 64, 1024)
  ref = og.ggml_data_to_tensor(data, 64 * 1024, t).astype(np.float16)
  out = _gpu_dequant(gpu, data, 64 * 1024, t, np.float16)
  assert out.tobytes() == ref.tobytes()

def test_empty_and_unknown_type(gpu):
  from tinygrad_amd.gguf import ggml_data_to_tensor
  assert ggml_data_to_tensor(np.zeros(0, dtype=np.uint8), 0, 2).numpy().size == 0
  with pytest.raises(ValueError): ggml_data_to_tensor(np.zeros(512, dtype=np.uint8), 256, 1337)   # test/unit/test_gguf.py:114-116

def test_lm_head_sized_q6_k(gpu):
  """A full-size slice property: dequant of the first and last 64 rows of a 128256x4096 Q6_K tensor addressed inside one big buffer."""
  rng = np.random.default_rng(7)
  rows, k = 2048, 4096
  data = synth.random_blocks(rng, 14, rows, k)
  out = _gpu_dequant(gpu, data, rows * k, 14)
  ref = og.ggml_data_to_tensor(data, rows * k, 14)
  assert out.tobytes() == ref.tobytes()

def test_synth_q4_k_writer_produces_valid_blocks(gpu):
  """tga_synth_weights(Q4_K): the blocks decode (oracle) to within one quantization step of U(-amp, amp) values: max |w| <= amp * (1 + 1/15)
  and the values are spread (not a constant), i.e. a valid block stream of the right magnitude."""
  n, amp = 256 * 64, 0.02
  buf = gpu.Buffer((n // 256 * 144,), np.uint8)
  gpu.check(gpu.lib().tga_synth_weights(12, buf.ptr, n, 77, amp, None))
  w = og.ggml_data_to_tensor(buf.numpy(), n, 12)
  assert np.isfinite(w).all() and np.abs(w).max() <= amp * 1.1 and w.std() > amp * 0.4
  assert _gpu_dequant(gpu, buf.numpy(), n, 12).tobytes() == w.tobytes()

@pytest.mark.parametrize("t", TYPES)
@pytest.mark.parametrize("f16", [True, False])
def test_large_results_are_those_of_their_parts(gpu, t, f16):
  """Results of 16 MB and more leave past the caches: the bits of the same blocks in runs below that, at the smallest such size, one block more, and (fp16) an output that starts two bytes
  off a dword; the bytes around it stay."""
  nel, nby = GGML_QUANT[t]
  n = (16 << 20) // (2 if f16 else 4) + nel
  n -= n % nel
  rng = np.random.default_rng(t)
  data = np.tile(synth.random_blocks(rng, t, 64, 1024), -(-n // 65536))[:n // nel * nby]
  src, sz, L = gpu.Buffer.from_numpy(data), 2 if f16 else 4, gpu.lib()
  half = n // nel // 2
  ref = gpu.Buffer((n * sz,), np.uint8)
  for b0, nb in ((0, half), (half, n // nel - half)):
    gpu.check(L.tga_dequant(t, src.ptr + b0 * nby, nb * nel, ref.ptr + b0 * nel * sz, gpu.dtype_code(np.float16 if f16 else np.float32), None))
  ref = ref.numpy()
  for off in ((16, 18) if f16 else (16,)):
    out = gpu.Buffer((n * sz + 64,), np.uint8)
    gpu.check(L.tga_memset(out.ptr, 0xAB, out.nbytes, None))
    gpu.check(L.tga_dequant(t, src.ptr, n, out.ptr + off, gpu.dtype_code(np.float16 if f16 else np.float32), None))
    got = out.numpy()
    assert (got[off:off + n * sz] != ref).sum() == 0 and (got[:off] == 0xAB).all() and (got[off + n * sz:] == 0xAB).all(), off

@pytest.mark.parametrize("t", TYPES)
def test_ragged_last_workgroups_and_unaligned_blocks(gpu, t):
  """One block, a block less and more than a workgroup's run of 2048 or 4096 values, and block bytes that start two past a 16-byte boundary: the
  oracle's bits in float32 and their cast in fp16, the byte behind the result untouched."""
  nel, nby = GGML_QUANT[t]
  rng = np.random.default_rng(100 + t)
  for nb in sorted({1, 2048 // nel - 1, 2048 // nel + 1, 4096 // nel - 1, 4096 // nel, 4096 // nel + 1, 3 * 4096 // nel + 2} - {0}):
    data = synth.random_blocks(rng, t, 1, nb * nel)
    ref = og.ggml_data_to_tensor(data, nb * nel, t)
    for at in (0, 2):
      src = gpu.Buffer.from_numpy(np.concatenate([np.zeros(at, np.uint8), data]))
      for f16, sz in ((True, 2), (False, 4)):
        out = gpu.Buffer((nb * nel * sz + 16,), np.uint8)
        gpu.check(gpu.lib().tga_memset(out.ptr, 0xAB, out.nbytes, None))
        gpu.check(gpu.lib().tga_dequant(t, src.ptr + at, nb * nel, out.ptr, gpu.dtype_code(np.float16 if f16 else np.float32), None))
        got, exp = out.numpy(), (ref.astype(np.float16) if f16 else ref)
        assert got[:nb * nel * sz].tobytes() == exp.tobytes() and (got[nb * nel * sz:] == 0xAB).all(), (nb, at, f16)
