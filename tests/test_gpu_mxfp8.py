"""MXFP8 MoE prefill path on the GPU vs the oracle: quantize_mxfp8 bit-exact, route/dispatch/combine exact (integer / byte work),
grouped GEMM within the reference's own error bars (test/backend/test_asm_gemm.py:310-313: mean-rel-err < 1e-2 vs dequant-matmul)."""
import numpy as np, pytest
from oracle import mxfp8 as omx, moe as omoe

pytestmark = pytest.mark.gpu

def test_quantize_mxfp8_bit_exact(gpu):
  from tinygrad_amd import moe
  rng = np.random.default_rng(1)
  x = (rng.standard_normal((300, 512)) * np.exp2(rng.integers(-20, 12, size=(300, 1)))).astype(np.float32)
  x[0, :32] = 0; x[1, :64] = 2.0 ** -3; x[2, 5] = 448.0; x[3, :32] = 1e-30
  q, e8, packed = moe.quantize_mxfp8(gpu.Buffer.from_numpy(x))
  rq, re8 = omx.quantize_mxfp8(x)
  np.testing.assert_array_equal(e8.numpy(), re8)
  np.testing.assert_array_equal(q.numpy(), rq)
  np.testing.assert_array_equal(packed.numpy(), omx.mx_pack(re8))
  # bf16 input
  xb = moe.to_bf16_bits(x)
  q2, e82, _ = moe.quantize_mxfp8(gpu.Buffer.from_numpy(xb))
  rq2, re82 = omx.quantize_mxfp8(moe.from_bf16_bits(xb))
  np.testing.assert_array_equal(e82.numpy(), re82); np.testing.assert_array_equal(q2.numpy(), rq2)

@pytest.mark.parametrize("M,N", [(256, 512), (96, 64), (384, 320)])
def test_transpose_quantize_mxfp8_bit_exact(gpu, M, N):
  """transpose_quantize_mxfp8(g) == quantize_mxfp8(g.T) (extra/llama_kernels/transpose_quantize_mxfp8/__init__.py:24-25): bit-exact against the
  oracle and against this library's own row-wise quantizer fed the transposed matrix; M = 96 has a partial 128-row tile and no packed scales."""
  from tinygrad_amd import moe
  rng = np.random.default_rng(M + N)
  g = (rng.standard_normal((M, N)) * np.exp2(rng.integers(-20, 12, size=(1, N)))).astype(np.float32)
  g[:32, 0] = 0; g[32:64, 1] = 2.0 ** -3; g[5, 2] = 448.0; g[:32, 3] = 1e-30
  gb = moe.to_bf16_bits(g)
  q, e8, si = moe.transpose_quantize_mxfp8(gpu.Buffer.from_numpy(gb))
  rq, re8, rsi = omx.transpose_quantize_mxfp8(moe.from_bf16_bits(gb))
  assert q.shape == (N, M) and e8.shape == (N, M // 32)
  np.testing.assert_array_equal(e8.numpy(), re8); np.testing.assert_array_equal(q.numpy(), rq)
  if M % 128 == 0: np.testing.assert_array_equal(si.numpy(), rsi)
  else: assert si is None and rsi is None
  q2, e82, si2 = moe.quantize_mxfp8(gpu.Buffer.from_numpy(np.ascontiguousarray(gb.T)))
  np.testing.assert_array_equal(q2.numpy(), q.numpy()); np.testing.assert_array_equal(e82.numpy(), e8.numpy())
  if M % 128 == 0: np.testing.assert_array_equal(si2.numpy(), si.numpy())

def test_fused_silu_mul_quantize_mxfp8(gpu):
  """silu(x_w1) * x_w3 quantized without an intermediate tensor (extra/llama_kernels/fused_silu_mul_quantize_mxfp8).  The product is
  formed in float32 from exp2; where the device's exp2 differs from numpy's in the last ulp an E4M3 code may land on the other side of
  a rounding boundary, so the bar is: block exponents equal, codes equal except for a < 1e-4 fraction, and those within one code."""
  from tinygrad_amd import moe
  rng = np.random.default_rng(4)
  w1 = (rng.standard_normal((256, 768)) * 3).astype(np.float32); w3 = rng.standard_normal((256, 768)).astype(np.float32)
  w1[0, :32] = 0; w1[1, :32] = -40.0; w1[2, :32] = 30.0
  b1, b3 = moe.to_bf16_bits(w1), moe.to_bf16_bits(w3)
  q, e8, packed = moe.fused_silu_mul_quantize_mxfp8(gpu.Buffer.from_numpy(b1), gpu.Buffer.from_numpy(b3))
  rq, re8 = omx.silu_mul_quantize_mxfp8(moe.from_bf16_bits(b1), moe.from_bf16_bits(b3))
  ge8, gq = e8.numpy(), q.numpy()
  assert np.mean(ge8 != re8) < 1e-4 and np.abs(ge8.astype(int) - re8.astype(int)).max() <= 1
  same_block = np.repeat(ge8 == re8, 32, axis=-1)
  diff = (gq != rq) & same_block
  assert diff.mean() < 1e-4
  mag = lambda c: (c & 0x7F).astype(int)
  assert (np.abs(mag(gq[diff]) - mag(rq[diff])) <= 1).all()
  np.testing.assert_array_equal(packed.numpy(), omx.mx_pack(ge8))
  # against the unfused chain on the GPU itself (float32 product quantized by tga_quantize_mxfp8): same bar
  act = moe.from_bf16_bits(b1); act = (act * (1.0 / (1.0 + np.exp2(act * np.float32(-1.4426950408889634)))) * moe.from_bf16_bits(b3)).astype(np.float32)
  q2, e82, _ = moe.quantize_mxfp8(gpu.Buffer.from_numpy(act))
  assert np.mean(q2.numpy() != gq) < 1e-4

@pytest.mark.parametrize("T,E,k", [(300, 16, 4), (4096, 128, 8), (7, 5, 5)])
def test_route_dispatch_combine(gpu, T, E, k):
  from tinygrad_amd import moe
  rng = np.random.default_rng(T + E)
  logits = rng.standard_normal((T, E)).astype(np.float32)
  if T > 10: logits[3, 2] = logits[3, 7] = 9.0                                   # a tie inside the top-k
  if E == 128: logits[:, :64] -= 3.0                                             # skewed load, some experts (nearly) empty
  r = moe.route(gpu.Buffer.from_numpy(logits), k, E)
  ref = omoe.route(logits, k, E)
  np.testing.assert_array_equal(r.topi.numpy(), ref["topi"])
  np.testing.assert_array_equal(r.off.numpy(), ref["off"])
  np.testing.assert_array_equal(r.dest_row.numpy(), ref["dest_row"])
  np.testing.assert_allclose(r.weights.numpy(), ref["weights"], rtol=2e-6, atol=1e-8)
  assert r.m_l == ref["m_l"]
  # invariants: dest_row is injective into expert-contiguous 256-padded ranges
  d = r.dest_row.numpy(); off = r.off.numpy(); e = r.topi.numpy().reshape(-1)
  assert len(set(d.tolist())) == T * k and (off % 256 == 0).all() and ((d >= off[e]) & (d < off[e + 1])).all()
  D = 64
  x = moe.to_bf16_bits(rng.standard_normal((T, D)).astype(np.float32))
  xg = moe.dispatch(gpu.Buffer.from_numpy(x), r)
  np.testing.assert_array_equal(xg.numpy(), omoe.dispatch(x, ref, k))
  # identity experts: combine(dispatch(x)) = x * sum(weights) = x (up to bf16 rounding of the products)
  out = moe.combine(xg, r, T, k)
  xf = moe.from_bf16_bits(x)
  wb = moe.from_bf16_bits(moe.to_bf16_bits(ref["weights"]))
  exp = moe.to_bf16_bits(moe.from_bf16_bits(moe.to_bf16_bits(xf[:, None, :] * wb[:, :, None])).sum(1))
  np.testing.assert_array_equal(out.numpy(), exp)

@pytest.mark.parametrize("E,N,K,rows", [(4, 256, 128, [256, 0, 512, 256]), (8, 512, 2048, [256] * 8), (3, 256, 768, [512, 256, 0])])
def test_grouped_mxfp8_gemm(gpu, E, N, K, rows):
  from tinygrad_amd import moe
  rng = np.random.default_rng(N + K)
  off = np.concatenate([[0], np.cumsum(rows)]).astype(np.int32)
  M = int(off[-1]) + 256                                                          # one tile beyond expert_off[E]: expert E - 1's by rows_e (moe_routing.py:98-104)
  x = (rng.standard_normal((M, K)) * 0.5).astype(np.float32)
  w = (rng.standard_normal((E, N, K)) * 0.5).astype(np.float32)
  xq, xe8 = omx.quantize_mxfp8(x); wq, we8 = omx.quantize_mxfp8(w)
  C = gpu.Buffer((M, N), np.uint16).zero_()
  bufs = [gpu.Buffer.from_numpy(a) for a in (xq, wq, xe8, we8, off)]
  gpu.check(gpu.lib().tga_grouped_mxfp8_gemm(C.ptr, bufs[0].ptr, bufs[1].ptr, None, None, bufs[2].ptr, bufs[3].ptr, bufs[4].ptr, M, N, K, E, None))
  got = moe.from_bf16_bits(C.numpy())
  ref = omx.grouped_mx_gemm_ref(xq, xe8, wq, we8, off)
  used = M
  err_mx = np.abs(got[:used] - ref[:used]).mean() / np.abs(ref[:used]).mean()
  assert err_mx < 1e-2, err_mx                                                    # the reference's bar
  # tighter: bf16 output of a float32 accumulation of exactly representable products: within one bf16 ulp of the oracle
  np.testing.assert_allclose(got[:used], ref[:used], rtol=2 ** -7, atol=1e-3 * np.abs(ref).max())
  # the routed-only variant writes the same values below expert_off[E] and nothing beyond
  C2 = gpu.Buffer((M, N), np.uint16).zero_()
  gpu.check(gpu.lib().tga_grouped_mxfp8_gemm_routed(C2.ptr, bufs[0].ptr, bufs[1].ptr, bufs[2].ptr, bufs[3].ptr, bufs[4].ptr, M, N, K, E, None))
  np.testing.assert_array_equal(C2.numpy()[:off[-1]], C.numpy()[:off[-1]]); assert (C2.numpy()[off[-1]:] == 0).all()
  # the pointer-argument kernel a Tensor.custom_kernel PROGRAM would bind (arguments in sink order, then the scalars), launched like
  # HIPProgram.__call__ does: 512 threads x (M / 256) (N / 256) workgroups
  import ctypes
  fn = ctypes.c_void_p()
  gpu.check(gpu.lib().tga_kernel_symbol(b"tga_grouped_mxfp8_gemm_kernel", ctypes.byref(fn)))
  C3 = gpu.Buffer((M, N), np.uint16).zero_()
  vals = [ctypes.c_void_p(C3.ptr), ctypes.c_void_p(bufs[0].ptr), ctypes.c_void_p(bufs[1].ptr), ctypes.c_void_p(None), ctypes.c_void_p(None), ctypes.c_void_p(bufs[2].ptr),
          ctypes.c_void_p(bufs[3].ptr), ctypes.c_void_p(bufs[4].ptr), ctypes.c_int(M), ctypes.c_int(N), ctypes.c_int(K), ctypes.c_int(E)]
  args = (ctypes.c_void_p * len(vals))(*[ctypes.cast(ctypes.pointer(v), ctypes.c_void_p) for v in vals])
  grid, block = (ctypes.c_uint32 * 3)((M // 256) * (N // 256), 1, 1), (ctypes.c_uint32 * 3)(512, 1, 1)
  gpu.check(gpu.lib().tga_launch_kernel(fn, grid, block, args, None)); gpu.synchronize()
  np.testing.assert_array_equal(C3.numpy(), C.numpy())
  assert gpu.lib().tga_kernel_symbol(b"no_such_kernel", ctypes.byref(fn)) != 0
  # against the unquantized product: the reference's second bar (< 6e-2)
  full = np.zeros_like(ref)
  for e in range(E): full[off[e]:off[e + 1]] = x[off[e]:off[e + 1]] @ w[e].T
  full[off[-1]:] = x[off[-1]:] @ w[E - 1].T
  assert np.abs(got[:used] - full[:used]).mean() / np.abs(full[:used]).mean() < 6e-2

def test_dense_mx_gemm_and_expert_bias(gpu):
  """The dense MXFP8 GEMM (one expert owning every row) against the oracle's matmul_mx semantics, then the per-expert bias add of
  gpt_oss.py:219-224 on a grouped result (bias cast to bf16, bf16 add), bit for bit."""
  from tinygrad_amd import moe
  rng = np.random.default_rng(12)
  M, N, K = 512, 256, 256
  x = moe.to_bf16_bits((rng.standard_normal((M, K)) * 0.5).astype(np.float32))
  w = (rng.standard_normal((N, K)) * 0.5).astype(np.float32)
  wq, we8 = omx.quantize_mxfp8(w)
  out = moe.mx_gemm(gpu.Buffer.from_numpy(x), (gpu.Buffer.from_numpy(wq), gpu.Buffer.from_numpy(we8)))
  xq, xe8 = omx.quantize_mxfp8(moe.from_bf16_bits(x))
  ref = omx.grouped_mx_gemm_ref(xq, xe8, wq[None], we8[None], np.array([0, M], np.int32))
  got = moe.from_bf16_bits(out.numpy())
  np.testing.assert_allclose(got, ref, rtol=2 ** -7, atol=1e-3 * np.abs(ref).max())
  # bias by expert on three experts' tiles; the last tile lies beyond expert_off[E] and takes the last expert's bias (rows_e)
  E = 3
  off = np.array([0, 256, 256, 512], dtype=np.int32)                 # expert 1 owns no rows
  h = moe.to_bf16_bits(rng.standard_normal((768, N)).astype(np.float32))
  bias = rng.standard_normal((E, N)).astype(np.float32)
  hb = gpu.Buffer.from_numpy(h)
  moe.add_expert_bias(hb, gpu.Buffer.from_numpy(bias), gpu.Buffer.from_numpy(off))
  exp = omx.add_expert_bias(moe.from_bf16_bits(h), bias, off)
  np.testing.assert_array_equal(hb.numpy(), moe.to_bf16_bits(exp))
  assert (hb.numpy()[512:] != h[512:]).any()                         # rows beyond expert_off[E] got expert E - 1's bias

def test_swiglu_interleaved(gpu):
  """The clamped interleaved SwiGLU between the two grouped GEMMs (examples/mlperf/models/gpt_oss.py:94-98) on bf16 rows, bit for bit against the
  oracle's bf16 chain except where the device's exp differs by an ulp before the bf16 rounding (at most one bf16 ulp, a handful of elements)."""
  from tinygrad_amd import moe
  rng = np.random.default_rng(21)
  h = moe.to_bf16_bits((rng.standard_normal((300, 512)) * 4).astype(np.float32))
  h[0, :8] = moe.to_bf16_bits(np.array([100, 100, -100, -100, 7, -7, 0, 0], np.float32))
  y = moe.swiglu(gpu.Buffer.from_numpy(h)).numpy()
  ref = omx.swiglu_interleaved(moe.from_bf16_bits(h))
  got = moe.from_bf16_bits(y)
  assert y.shape == (300, 256)
  np.testing.assert_allclose(got, ref, rtol=2 ** -7, atol=1e-30)
  assert (moe.to_bf16_bits(ref) == y).mean() > 0.99

def test_moe_feed_forward_composition(gpu):
  """moe.moe_feed_forward (route -> dispatch -> grouped GEMM + bias -> SwiGLU -> grouped GEMM + bias -> combine, gpt_oss.py:213-226) against the
  reference's per-expert loop (gpt_oss.py:227-238) restated in the oracle; the reference has no test of its own for either branch, the
  loop is the definition (oracle pinned in tests/test_oracle_pins.py).  Bar: the reference's MXFP8 GEMM bar (mean rel-err < 1e-2), since the two
  branches round to bf16 at different points (the loop weighs and sums bf16 contributions expert by expert, the grouped branch weighs rows)."""
  from tinygrad_amd import moe
  rng = np.random.default_rng(33)
  T, D, I, E, k = 96, 256, 256, 6, 2
  inp = moe.to_bf16_bits(rng.standard_normal((T, D)).astype(np.float32))
  logits = rng.standard_normal((T, E)).astype(np.float32); logits[:, 4] = -30.0       # expert 4 is never selected: an empty range
  wgu, wdn = (rng.standard_normal((E, 2 * I, D)) * D ** -0.5).astype(np.float32), (rng.standard_normal((E, D, I)) * I ** -0.5).astype(np.float32)
  bgu, bdn = (rng.standard_normal((E, 2 * I)) * 0.1).astype(np.float32), (rng.standard_normal((E, D)) * 0.1).astype(np.float32)
  (gq, ge), (dq, de) = omx.quantize_mxfp8(wgu), omx.quantize_mxfp8(wdn)
  B = gpu.Buffer.from_numpy
  ref = omx.moe_feed_forward_loop(moe.from_bf16_bits(inp), logits, k, gq, ge, bgu, dq, de, bdn)
  for routed_only in (True, False):
    out = moe.moe_feed_forward(B(inp), B(logits), k, (B(gq), B(ge)), B(bgu), (B(dq), B(de)), B(bdn), routed_only=routed_only)
    got = moe.from_bf16_bits(out.numpy())
    assert got.shape == (T, D) and np.isfinite(got).all()
    err = np.abs(got - ref).mean() / np.abs(ref).mean()
    print(f"moe_feed_forward vs per-expert loop (routed_only={routed_only}): mean rel-err {err:.2e}")
    assert err < 1e-2
    np.testing.assert_allclose(got, ref, rtol=0.05, atol=0.02 * np.abs(ref).max())

def test_grouped_gemm_with_counts_skips_padding(gpu):
  """tga_grouped_mxfp8_gemm_counts: routed rows equal the routed-tiles product bit for bit; padding rows inside an expert's range come out as zeros even
  when A holds garbage there; rows beyond expert_off[E] keep their contents.  Experts of 1, 16, 17, 128, 129, 255, 256 and 300 rows and an empty one."""
  rng = np.random.default_rng(41)
  counts = np.array([1, 16, 17, 0, 128, 129, 255, 256, 300], np.int32)
  E, N, K = len(counts), 512, 384
  off = np.concatenate([[0], np.cumsum((counts + 255) // 256 * 256)]).astype(np.int32)
  M = int(off[-1]) + 512                                              # two tiles beyond the routed range
  def rand_mx(rows):
    q = rng.integers(0, 256, size=(rows, K), dtype=np.uint8); q[(q & 0x7F) == 0x7F] = 0x38
    return q, rng.integers(121, 126, size=(rows, K // 32), dtype=np.uint8)
  xq, xe = rand_mx(M); wq, we = rand_mx(E * N)                         # padding rows of A are random too: they must not reach the output
  bufs = [gpu.Buffer.from_numpy(a) for a in (xq, wq, xe, we)]
  offb, cntb = gpu.Buffer.from_numpy(off), gpu.Buffer.from_numpy(counts)
  C1, C2 = gpu.Buffer((M, N), np.uint16), gpu.Buffer((M, N), np.uint16)
  for C in (C1, C2): gpu.check(gpu.lib().tga_memset(C.ptr, 0xAB, C.nbytes, None))
  gpu.check(gpu.lib().tga_grouped_mxfp8_gemm_routed(C1.ptr, bufs[0].ptr, bufs[1].ptr, bufs[2].ptr, bufs[3].ptr, offb.ptr, M, N, K, E, None))
  gpu.check(gpu.lib().tga_grouped_mxfp8_gemm_counts(C2.ptr, bufs[0].ptr, bufs[1].ptr, bufs[2].ptr, bufs[3].ptr, offb.ptr, cntb.ptr, M, N, K, E, None))
  c1, c2 = C1.numpy(), C2.numpy()
  for e in range(E):
    lo, n, hi = int(off[e]), int(counts[e]), int(off[e + 1])
    np.testing.assert_array_equal(c2[lo:lo + n], c1[lo:lo + n], err_msg=f"routed rows of expert {e}")
    pad16 = lo + (n + 15) // 16 * 16                                  # rows of a 16-row group that also holds routed rows are multiplied like them
    np.testing.assert_array_equal(c2[lo + n:pad16], c1[lo + n:pad16])
    assert (c2[pad16:hi] == 0).all(), f"padding rows of expert {e}"
  assert (c2[off[-1]:] == 0xABAB).all()

@pytest.mark.parametrize("rows,K", [(1, 32), (3, 96), (5, 160), (257, 128), (33, 1056), (2048, 4096)])
def test_quantize_rows_of_any_length(gpu, rows, K):
  """Four lanes per block: single blocks, rows that end inside a wave, several trips per thread; float32 and bf16 rows, with and without the packed scales, bit for bit."""
  from tinygrad_amd import moe
  rng = np.random.default_rng(rows + K)
  x = (rng.standard_normal((rows, K)) * np.exp2(rng.integers(-20, 12, size=(rows, 1)))).astype(np.float32)
  bits = moe.to_bf16_bits(x)
  for src, ref in ((x, x), (bits, moe.from_bf16_bits(bits))):
    q, e8, packed = moe.quantize_mxfp8(gpu.Buffer.from_numpy(src))
    rq, re8 = omx.quantize_mxfp8(ref)
    np.testing.assert_array_equal(e8.numpy(), re8); np.testing.assert_array_equal(q.numpy(), rq)
    assert (packed is None) == (K % 128 != 0)
    if packed is not None: np.testing.assert_array_equal(packed.numpy(), re8.reshape(rows, K // 128, 4).view(np.uint32)[..., 0].T)

def test_large_quantized_results_are_those_of_their_parts(gpu):
  """Results of 16 MB and more leave past the caches: rows of float32, of bf16, of the fused SwiGLU and of the transposed form against the same rows in parts below that."""
  from tinygrad_amd import moe
  rows, K = 4100, 4096
  rng = np.random.default_rng(9)
  x = rng.standard_normal((rows, K), dtype=np.float32) * np.exp2(rng.integers(-20, 12, size=(rows, 1))).astype(np.float32)
  bits, up = moe.to_bf16_bits(x), moe.to_bf16_bits(x[::-1])
  B = gpu.Buffer.from_numpy
  for whole, part in ((lambda: moe.quantize_mxfp8(B(x)), lambda a, b: moe.quantize_mxfp8(B(x[a:b]))), (lambda: moe.quantize_mxfp8(B(bits)), lambda a, b: moe.quantize_mxfp8(B(bits[a:b]))),
                      (lambda: moe.fused_silu_mul_quantize_mxfp8(B(bits), B(up)), lambda a, b: moe.fused_silu_mul_quantize_mxfp8(B(bits[a:b]), B(up[a:b])))):
    q, e8, packed = (b.numpy() for b in whole())
    for a, b in ((0, 2050), (2050, rows)):
      rq, re8, rp = (v.numpy() for v in part(a, b))
      assert (q[a:b] != rq).sum() == 0 and (e8[a:b] != re8).sum() == 0 and (packed[:, a:b] != rp).sum() == 0
  g = bits[:4096]                                                      # (columns of the source are rows of the result)
  q, e8, packed = (b.numpy() for b in moe.transpose_quantize_mxfp8(B(g)))
  for a, b in ((0, 2048), (2048, K)):
    rq, re8, rp = (v.numpy() for v in moe.transpose_quantize_mxfp8(B(np.ascontiguousarray(g[:, a:b]))))
    assert (q[a:b] != rq).sum() == 0 and (e8[a:b] != re8).sum() == 0 and (packed[:, a:b] != rp).sum() == 0

@pytest.mark.parametrize("M,N", [(32, 64), (96, 128), (128, 64), (160, 192), (512, 256)])
def test_transpose_quantize_of_ragged_row_counts(gpu, M, N):
  """Row counts that end inside a 128-row tile (no packed scales there) against quantize_mxfp8 of the transposed matrix, bit for bit."""
  from tinygrad_amd import moe
  bits = moe.to_bf16_bits(np.random.default_rng(M + N).standard_normal((M, N)).astype(np.float32) * 3)
  q, e8, packed = moe.transpose_quantize_mxfp8(gpu.Buffer.from_numpy(bits))
  rq, re8 = omx.quantize_mxfp8(np.ascontiguousarray(moe.from_bf16_bits(bits).T))
  np.testing.assert_array_equal(q.numpy(), rq); np.testing.assert_array_equal(e8.numpy(), re8)
  if packed is not None: np.testing.assert_array_equal(packed.numpy(), re8.reshape(N, M // 128, 4).view(np.uint32)[..., 0].T)

def test_swiglu_beyond_one_trip_and_off_alignment(gpu):
  """More outputs than one pass of the grid holds, a length that is no multiple of four, and operands that start off a 16-byte boundary: the same values as small aligned calls."""
  from tinygrad_amd import moe
  rng = np.random.default_rng(5)
  unit = moe.to_bf16_bits((rng.standard_normal((1, 2 * 4099)) * 4).astype(np.float32))
  ref = omx.swiglu_interleaved(moe.from_bf16_bits(unit))[0]
  rows = (1 << 24) // 4099 + 300                                       # > 2^24 outputs, rows of an odd length
  y = moe.swiglu(gpu.Buffer.from_numpy(np.tile(unit, (rows, 1)))).numpy()
  np.testing.assert_allclose(moe.from_bf16_bits(y[0]), ref, rtol=2 ** -7, atol=1e-30)
  assert (y == y[0]).all()
  off = gpu.Buffer.from_numpy(np.concatenate([np.zeros(1, np.uint16), unit[0]])).view(2, (1, 2 * 4099), np.uint16)
  np.testing.assert_array_equal(moe.swiglu(off).numpy()[0], y[0])

@pytest.mark.parametrize("T,D,I,E,k", [(1, 256, 256, 8, 1), (1, 512, 256, 128, 8), (33, 256, 512, 3, 3), (64, 512, 256, 16, 4), (65, 256, 256, 65, 2), (129, 256, 256, 200, 5), (300, 512, 256, 4, 2), (700, 256, 256, 2, 1)])
def test_moe_feed_forward_at_tile_edges(gpu, T, D, I, E, k):
  """The fused feed-forward at one token, one and two routing workgroups, more experts than a wave has lanes, experts of no rows, of fewer rows than a tile and of several tiles (both
  tile heights), against the reference's per-expert loop restated in the oracle.  Bar as in the composition test above: the two branches round to bf16 at different points."""
  from tinygrad_amd import moe
  rng = np.random.default_rng(T + E)
  inp = moe.to_bf16_bits(rng.standard_normal((T, D)).astype(np.float32))
  logits = rng.standard_normal((T, E)).astype(np.float32) + np.linspace(0, 3, E, dtype=np.float32)
  wgu, wdn = (rng.standard_normal((E, 2 * I, D)) * D ** -0.5).astype(np.float32), (rng.standard_normal((E, D, I)) * I ** -0.5).astype(np.float32)
  bgu, bdn = (rng.standard_normal((E, 2 * I)) * 0.1).astype(np.float32), (rng.standard_normal((E, D)) * 0.1).astype(np.float32)
  (gq, ge), (dq, de) = omx.quantize_mxfp8(wgu), omx.quantize_mxfp8(wdn)
  B = gpu.Buffer.from_numpy
  ref = omx.moe_feed_forward_loop(moe.from_bf16_bits(inp), logits, k, gq, ge, bgu, dq, de, bdn)
  got = moe.from_bf16_bits(moe.moe_feed_forward(B(inp), B(logits), k, (B(gq), B(ge)), B(bgu), (B(dq), B(de)), B(bdn)).numpy())
  assert np.isfinite(got).all() and np.abs(got - ref).mean() / np.abs(ref).mean() < 1e-2
  np.testing.assert_allclose(got, ref, rtol=0.05, atol=0.02 * np.abs(ref).max())

def _single_steps(moe, inp, logits, k, gate_up, b_gate_up, down, b_down):
  r = moe.route(logits, k, logits.shape[1])
  xg = moe.dispatch(inp, r)
  h = moe.add_expert_bias(moe.grouped_mx_gemm(xg, gate_up, r.off, routed_only=True, counts=r.counts), b_gate_up, r.off)
  y = moe.swiglu(h)
  z = moe.add_expert_bias(moe.grouped_mx_gemm(y, down, r.off, routed_only=True, counts=r.counts), b_down, r.off)
  return moe.combine(z, r, inp.shape[0], k).numpy()

@pytest.mark.parametrize("T,D,I,E,k,skew", [(1, 256, 256, 3, 1, 0), (5, 768, 256, 70, 8, 1), (33, 2048, 768, 5, 3, 1), (40, 1280, 512, 20, 4, 0), (130, 256, 768, 4, 4, 0), (600, 1024, 256, 9, 2, 2), (900, 512, 512, 12, 2, 0),
                                            (2600, 256, 768, 40, 2, 1), (4128, 4096, 256, 4, 4, 0), (6000, 256, 256, 80, 2, 0), (3100, 768, 512, 65, 4, 0), (700, 1536, 512, 512, 8, 1)])
def test_moe_feed_forward_at_every_tile_height(gpu, T, D, I, E, k, skew):
  """Tiles of 16, 32, 64, 128 and 256 rows (by the rows per expert; 256 where the counts, on the device, make them five ninths of the rounds or fewer: 9 / 5 rounds of the down product of 4 x 4128 rows), reductions of 2, 4, 6, 8, 10, 12 and 16 steps of 128 (scales
  are fetched four steps at a time, a last pair on its own), experts of no rows, of one, of several tiles and with a remainder, more experts than lanes: bits of the single steps, twice."""
  from tinygrad_amd import moe
  rng = np.random.default_rng(T + D + I + E)
  B = gpu.Buffer.from_numpy
  inp = moe.to_bf16_bits(rng.standard_normal((T, D)).astype(np.float32))
  logits = (rng.standard_normal((T, E)) + skew * np.linspace(0, 3, E)).astype(np.float32)
  def weight(n, kk): return moe.quantize_mxfp8(B(moe.to_bf16_bits((rng.standard_normal((E * n, kk), dtype=np.float32) * np.float32(kk ** -0.5)))))[:2]
  (gq, ge), (dq, de) = weight(2 * I, D), weight(D, I)
  args = (B(inp), B(logits), k, (gq.view(0, (E, 2 * I, D), np.uint8), ge.view(0, (E, 2 * I, D // 32), np.uint8)), B((rng.standard_normal((E, 2 * I)) * 0.1).astype(np.float32)),
          (dq.view(0, (E, D, I), np.uint8), de.view(0, (E, D, I // 32), np.uint8)), B((rng.standard_normal((E, D)) * 0.1).astype(np.float32)))
  ref = _single_steps(moe, *args)
  for _ in range(2): assert (moe.moe_feed_forward(*args).numpy() != ref).sum() == 0

@pytest.mark.parametrize("case", ["random", "masked", "fewer than k", "tiny"])
def test_moe_feed_forward_has_the_bits_of_the_single_steps(gpu, case):
  """Random rows; logits masked with -inf so that exactly k, or fewer than k, experts are left (the surplus picks weigh nothing); gate values whose sigmoid is a subnormal number."""
  from tinygrad_amd import moe
  T, D, I, E, k = 70, 512, 256, 16, 3
  rng = np.random.default_rng(len(case))
  B = gpu.Buffer.from_numpy
  inp, logits = moe.to_bf16_bits(rng.standard_normal((T, D)).astype(np.float32)), rng.standard_normal((T, E)).astype(np.float32)
  wgu, wdn = (rng.standard_normal((E, 2 * I, D)) * D ** -0.5).astype(np.float32), (rng.standard_normal((E, D, I)) * I ** -0.5).astype(np.float32)
  bgu, bdn = (rng.standard_normal((E, 2 * I)) * 0.1).astype(np.float32), (rng.standard_normal((E, D)) * 0.1).astype(np.float32)
  if case in ("masked", "fewer than k"):
    keep = np.argsort(rng.random((T, E)), axis=1)[:, :k if case == "masked" else k - 1]
    mask = np.full((T, E), -np.inf, np.float32); np.put_along_axis(mask, keep, 0, axis=1)
    logits += mask
  if case == "tiny":                                                   # gate = bias: 1.702 times it rounds to -87.5, -88 and -88.5, whose logistic function lies below the normal numbers
    wgu[:] = 0; bdn[:] = 0
    bgu[:, 0::2], bgu[:, 1::2] = np.array([-51.5, -51.75, -52.0], np.float32)[np.arange(E) % 3][:, None], 6.0
  args = (B(inp), B(logits), k, tuple(map(B, omx.quantize_mxfp8(wgu))), B(bgu), tuple(map(B, omx.quantize_mxfp8(wdn))), B(bdn))
  got, ref = moe.moe_feed_forward(*args).numpy(), _single_steps(moe, *args)
  assert case != "tiny" or (ref & 0x7FFF).any()
  np.testing.assert_array_equal(got, ref)

@pytest.mark.parametrize("T,E", [(70, 16), (900, 4)])
def test_moe_feed_forward_of_values_that_are_not_finite(gpu, T, E):
  """A row of infinities, one with a NaN and a NaN bias of one gate column (the largest magnitude of a block and its 32 results pass between lanes in registers): in low tiles and in full ones of
  128 rows, NaN where the single steps give NaN and their bits elsewhere."""
  from tinygrad_amd import moe
  D, I, k = 512, 256, 2
  rng = np.random.default_rng(T)
  B = gpu.Buffer.from_numpy
  x = rng.standard_normal((T, D)).astype(np.float32)
  x[3] = np.inf; x[17, 5] = np.nan
  wgu, wdn = (rng.standard_normal((E, 2 * I, D)) * D ** -0.5).astype(np.float32), (rng.standard_normal((E, D, I)) * I ** -0.5).astype(np.float32)
  bgu, bdn = (rng.standard_normal((E, 2 * I)) * 0.1).astype(np.float32), (rng.standard_normal((E, D)) * 0.1).astype(np.float32)
  bgu[1, 70] = np.nan
  args = (B(moe.to_bf16_bits(x)), B(rng.standard_normal((T, E)).astype(np.float32)), k, tuple(map(B, omx.quantize_mxfp8(wgu))), B(bgu), tuple(map(B, omx.quantize_mxfp8(wdn))), B(bdn))
  got, ref = moe.moe_feed_forward(*args).numpy(), _single_steps(moe, *args)
  nan = lambda b: (b & 0x7FFF) > 0x7F80
  np.testing.assert_array_equal(nan(got), nan(ref))
  np.testing.assert_array_equal(np.where(nan(got), 0, got), np.where(nan(ref), 0, ref))
