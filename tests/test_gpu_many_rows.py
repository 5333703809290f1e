"""Prefill steps of many rows on the GPU: tga_qlinear_many for every format at tile edges against a float64 product over the dequantized (fp16-rounded) weights, and whole steps - one
sequence and several, dense and MoE, one step and a prompt cut into several - against the same models prefilled position by position."""
import ctypes, dataclasses
import numpy as np, pytest
from decode_helpers import many_tile
from oracle import ggml as og, linear as ol, llm as ollm
from tinygrad_amd import synth

pytestmark = pytest.mark.gpu
FORMATS = ["Q4_0", "Q8_0", "F16", "MXFP4", "Q4_K", "Q5_K", "Q6_K", "IQ4_XS", "Q4_1", "Q5_0", "Q5_1"]

def _weight(rng, rt, t, n, k):
  if t == rt.F16:
    w = (rng.standard_normal((n, k)) * k ** -0.5).astype(np.float16)
    return w.view(np.uint8).reshape(-1), w.astype(np.float32)
  raw = synth.random_blocks(rng, t, n, k, sigma=0.0002 if t == rt.IQ4_XS else 0.003)
  return raw, og.ggml_data_to_tensor(raw, n * k, t).reshape(n, k).astype(np.float16).astype(np.float32)      # (the kernel multiplies fp16-rounded weights, model.py:376)

@pytest.mark.parametrize("fmt", FORMATS)
def test_many_rows_linear_at_tile_edges(gpu, fmt):
  """Rows 1 / 31 / 33 / 64 / 65 / 129 and outputs 16 / 127 / 129 / 300 around the tile heights, K of one and several steps; plain fp32 and fp16 results, + residual in place,
  silu(gate) * up, three matrices in one launch, with and without a workspace (split K).  Bar: float32 accumulation of exact products of fp16 values, K <= 768: each sum carries
  at most K 2^-24 relative to its absolute sum, 5e-5 of the largest result; fp16 results one more rounding, 2^-11.  Where a weight is a product and a difference of scales (K-quants,
  IQ4_XS, Q4_1, Q5_1) the kernel forms it with fused multiply-adds and the oracle with separate roundings: some weights then round to the neighbouring fp16 value, 2^-10 relative each,
  which bounds a sum by 2^-10 of its absolute sum; the linears' common bar of 1e-3 of the largest result holds them."""
  from tinygrad_amd import runtime as rt
  t = getattr(rt, fmt)
  rng = np.random.default_rng(t)
  ws = rt.Buffer((8 << 20,), np.uint8)
  def call(layers, x, outs, ydt, epi=0, resid=None, work=True):
    n = len(layers); VP = ctypes.c_void_p * n
    rt.check(rt.lib().tga_qlinear_many(t, n, VP(*[l[0].ptr for l in layers]), VP(*[(outs[i].ptr if i < len(outs) else None) for i in range(n)]), (ctypes.c_int64 * n)(*[l[1] for l in layers]),
                                       x.ptr, ydt, x.shape[0], x.shape[1], epi, resid.ptr if resid is not None else None, ws.ptr if work else None, ws.nbytes if work else 0, None))
  bar = 1e-3 if fmt in ("Q4_K", "Q5_K", "IQ4_XS", "Q4_1", "Q5_1") else 5e-5
  def close(got, ref, f16=False): assert ol.rel_err(got.astype(np.float32), ref) <= bar + (2.0 ** -11 if f16 else 0)
  for m, n, k in ((1, 16, 256), (31, 127, 768), (33, 300, 256), (64, 129, 512), (65, 16, 768), (129, 300, 512)):
    raw, w = _weight(rng, rt, t, n, k); raw2, w2 = _weight(rng, rt, t, n, k)
    wb, wb2 = rt.Buffer.from_numpy(raw), rt.Buffer.from_numpy(raw2)
    x = synth.activations(rng, m, k, np.float16); xb = rt.Buffer.from_numpy(x)
    ref, ref2 = ol.linear_f64(x.astype(np.float32), w), ol.linear_f64(x.astype(np.float32), w2)
    for work in (True, False):
      y = rt.Buffer((m, n), np.float32); call([(wb, n)], xb, [y], rt.F32, work=work); close(y.numpy(), ref)
      h = rt.Buffer((m, n), np.float16); call([(wb, n)], xb, [h], rt.F16, work=work); close(h.numpy(), ref, True)
      r = rng.standard_normal((m, n)).astype(np.float32); y = rt.Buffer.from_numpy(r); call([(wb, n)], xb, [y], rt.F32, 1, y, work=work); close(y.numpy(), ref + r)
    y = rt.Buffer((m, n), np.float32); call([(wb, n), (wb2, n)], xb, [y], rt.F32, 2)
    sw = ref / (1 + np.exp(-ref)) * ref2
    assert ol.rel_err(y.numpy(), sw) <= 4 * bar                                    # (two such sums and the exponential of one of them multiplied)
  ns, k, m = (128, 64, 80), 512, 70
  parts = [_weight(rng, rt, t, n, k) for n in ns]
  x = synth.activations(rng, m, k, np.float16); xb = rt.Buffer.from_numpy(x)
  bufs = [rt.Buffer.from_numpy(p[0]) for p in parts]
  for work in (True, False):
    outs = [rt.Buffer((m, n), np.float32) for n in ns]
    call(list(zip(bufs, ns)), xb, outs, rt.F32, work=work)
    for o, p in zip(outs, parts): close(o.numpy(), ol.linear_f64(x.astype(np.float32), p[1]))
  assert rt.lib().tga_qlinear_many(t, 1, (ctypes.c_void_p * 1)(bufs[0].ptr), (ctypes.c_void_p * 1)(outs[0].ptr), (ctypes.c_int64 * 1)(128), xb.ptr, rt.F32, m, 96, 0, None, None, 0, None) != 0

@pytest.mark.parametrize("m,n,k,epi", [(1283, (7500,), 3072, 0), (1281, (7501,), 3328, 0), (1408, (7440,), 3072, 1), (1345, (4096, 1616, 1808), 3072, 0), (1283, (3830,), 3072, 2), (1283, (2560,), 12544, 1)],
                         ids=["ragged", "odd", "resid", "three", "swiglu", "split"])
def test_wide_tiles_of_q4_0(gpu, m, n, k, epi):
  """The 256 x 128 tiles (twelve steps of 256 per workgroup and 320 workgroups or more): last tiles of 1, 3, 65 and 128 rows and of 12, 76, 96 and 118 outputs, thirteen steps, matrices that meet
  inside a tile, results that are no multiple of four, K split into parts of twelve and thirteen steps.  Weights are the same fp16 values as in the smaller tiles; float32 sums of K products in another order than the
  reference's (sgemm): each within K 2^-24 of its absolute sum at the very worst and about sqrt(K) 2^-24 in practice, 5e-5 of the largest result."""
  from tinygrad_amd import runtime as rt
  rng = np.random.default_rng(m)
  ws = rt.Buffer((64 << 20,), np.uint8)
  ns = n * 2 if epi == 2 else n
  parts = [_weight(rng, rt, rt.Q4_0, i, k) for i in ns]
  bufs = [rt.Buffer.from_numpy(p[0]) for p in parts]
  x = synth.activations(rng, m, k, np.float16); xb = rt.Buffer.from_numpy(x)
  refs = [x.astype(np.float32) @ p[1].T for p in parts]
  r = rng.standard_normal((m, n[0])).astype(np.float32)
  outs = [rt.Buffer.from_numpy(r) if epi == 1 else rt.Buffer((m, i), np.float32) for i in n]
  VP = ctypes.c_void_p * len(ns)
  rt.check(rt.lib().tga_qlinear_many(rt.Q4_0, len(ns), VP(*[b.ptr for b in bufs]), VP(*[(outs[i].ptr if i < len(outs) else None) for i in range(len(ns))]), (ctypes.c_int64 * len(ns))(*ns),
                                     xb.ptr, rt.F32, m, k, epi, outs[0].ptr if epi == 1 else None, ws.ptr, ws.nbytes, None))
  if epi == 2: refs = [refs[0] / (1 + np.exp(-refs[0])) * refs[1]]
  for o, ref in zip(outs, refs): assert ol.rel_err(o.numpy(), ref + r if epi == 1 else ref) <= (2e-4 if epi == 2 else 5e-5)

TALL = [("one-row", 385, (16400,), 1280, 0, 1, 1), ("ragged", 513, (14352,), 1536, 0, 1, 1), ("split", 1023, (4112,), 4096, 1, 3, 3), ("split-even", 1023, (4112,), 2816, 1, 2, None), ("three", 1025, (4096, 1040, 2064), 1280, 0, 1, 1),
        ("swiglu", 641, (7184,), 1280, 2, 1, 1), ("split-four", 1023, (4096,), 14336, 1, 4, 4), ("split-ten", 300, (4096,), 14336, 1, 10, None), ("rounds", 2047, (6160,), 3072, 0, 1, 1), ("four-steps", 1023, (14352, 14352), 1024, 0, 1, 1)]
@pytest.mark.parametrize("t,m,n,k,epi,parts", [pytest.param(t, *c[1:5], c[5 + i], id=f"{c[0]}-{name}") for i, (t, name) in enumerate([(2, "Q4_0"), (12, "Q4_K")]) for c in TALL if c[5 + i]])
def test_tall_tiles(gpu, t, m, n, k, epi, parts):
  """The 512 x 128 tiles, which the rule takes for each of these: last tiles of 1, 44 and 127 rows and of 16 outputs, four to fourteen steps a workgroup, odd and even, matrices that meet inside a tile, K split into two to ten
  parts, equal and not, for either type, float32 and fp16 results.
  Weights that begin four bytes behind a sixteen-byte line take the other tiles: the same fp16 weights in another order of sums, float32 sums of K products differ by about sqrt(K) 2^-24 of their absolute sum, 5e-5
  of the largest result at most.  So do those of the reference for Q4_0; for Q4_K, whose weights round differently now and then, the bar is that of test_many_rows_linear_at_tile_edges."""
  assert many_tile(t, n * 2 if epi == 2 else n, m, k, epi) == ((512, 128), parts)
  from tinygrad_amd import runtime as rt
  rng = np.random.default_rng(m + t)
  ws = rt.Buffer((64 << 20,), np.uint8)
  ns = n * 2 if epi == 2 else n
  parts = [_weight(rng, rt, t, i, k) for i in ns]
  x = synth.activations(rng, m, k, np.float16); xb = rt.Buffer.from_numpy(x)
  r = rng.standard_normal((m, n[0])).astype(np.float32)
  refs = [x.astype(np.float32) @ p[1].T for p in parts]
  if epi == 2: refs = [refs[0] / (1 + np.exp(-refs[0])) * refs[1]]
  VP = ctypes.c_void_p * len(ns)
  for dt, off in ((np.float32, 0), (np.float32, 4), (np.float16, 0)):
    if epi == 1 and dt == np.float16: continue
    bufs = [rt.Buffer.from_numpy(np.concatenate([np.zeros(off, np.uint8), p[0].reshape(-1).view(np.uint8)])) for p in parts]
    outs = [rt.Buffer.from_numpy(r) if epi == 1 else rt.Buffer((m, i), dt) for i in n]
    rt.check(rt.lib().tga_qlinear_many(t, len(ns), VP(*[b.ptr + off for b in bufs]), VP(*[(outs[i].ptr if i < len(outs) else None) for i in range(len(ns))]), (ctypes.c_int64 * len(ns))(*ns),
                                       xb.ptr, rt.F32 if dt == np.float32 else rt.F16, m, k, epi, outs[0].ptr if epi == 1 else None, ws.ptr, ws.nbytes, None))
    sums = 2e-4 if epi == 2 else 5e-5
    got = [o.numpy().astype(np.float32) for o in outs]
    if off == 0 and dt == np.float32: tall = got
    for o, o2, ref in zip(got, tall, refs):
      assert ol.rel_err(o, ref + r if epi == 1 else ref) <= ((4e-3 if epi == 2 else 1e-3) if t == 12 else sums) + (5e-4 if dt == np.float16 else 0)
      assert ol.rel_err(o, o2) <= sums + (5e-4 if dt == np.float16 else 0)

DENSE = dict(num_blocks=2, dim=512, hidden_dim=768, n_heads=8, n_kv_heads=2, norm_eps=1e-5, vocab_size=512, head_dim=64, rope_theta=500000.0)
DENSE128 = dict(num_blocks=2, dim=768, hidden_dim=512, n_heads=6, n_kv_heads=6, norm_eps=1e-5, vocab_size=512, head_dim=128, rope_theta=10000.0)
MOE = dict(num_blocks=2, dim=256, hidden_dim=256, n_heads=4, n_kv_heads=4, norm_eps=1e-5, vocab_size=512, head_dim=64, rope_theta=10000.0, qk_norm=256, num_experts=8, num_experts_per_tok=2)

def _model(cfg, seed, ctx=320, batch=0, **kw):
  from tinygrad_amd.llm import BatchedTransformer, Transformer, TransformerConfig, synth_state, synth_state_moe
  c = TransformerConfig(max_context=ctx, **cfg)
  sd = synth_state_moe(c, seed=seed) if c.num_experts else synth_state(c, seed=seed, **kw)
  return BatchedTransformer(c, sd, batch, max_new=8) if batch else Transformer(c, sd, max_new=8)

@pytest.mark.parametrize("cfg,kw", [(DENSE, {}), (DENSE, {"q4_k_m": True}), (DENSE128, {"linear_type": 8}), (DENSE128, {"linear_type": 1})], ids=["gqa4-hd64-q4_0", "gqa4-hd64-q4_k_m", "mha-hd128-q8_0", "mha-hd128-f16"])
@pytest.mark.parametrize("n,rows", [(18, 2048), (65, 2048), (130, 2048), (300, 2048), (300, 100)])
def test_prefill_of_many_rows_vs_position_by_position(gpu, monkeypatch, cfg, kw, n, rows):
  """Prompts around the row tiles of the attention (16 / 64) and of the linears, in one step and cut into steps of a hundred rows that attend to the cache of the ones before: caches within fp16
  rounding of the model prefilled token by token (2e-3, the bar of the chunked prefill), nothing written beyond the prompt, logits of the next step within 2e-3 (both sides
  are within 1e-3 of the reference's numerics)."""
  from tinygrad_amd import llm
  monkeypatch.setattr(llm, "MANY_ROWS", rows)
  a, b = _model(cfg, 5, **kw), _model(cfg, 5, **kw)
  b.prefill_chunk = 1
  prompt = [int(t) for t in np.random.default_rng(n).integers(0, cfg["vocab_size"], size=n)]
  for m in (a, b): m.prefill(prompt)
  assert (a._chunker or a._tail_chunkers[16]).x is None and a.prefill_steps == n - 1     # (no plain step was run)
  for ba, bb in zip(a.blk, b.blk):
    for ca, cb in ((ba.cache_k, bb.cache_k), (ba.cache_v, bb.cache_v)):
      ca, cb = ca.numpy().astype(np.float32), cb.numpy().astype(np.float32)
      assert ol.rel_err(ca[:, :n - 1], cb[:, :n - 1]) <= 2e-3 and not ca[:, n - 1:].any()
  for m in (a, b): m.decode_step()
  assert ol.rel_err(a.logits(), b.logits()) <= 2e-3
  longer = prompt[:n - 4] + [7] * 20                                               # a follow-up that keeps the cached prefix
  for m in (a, b): m.prefill(longer); m.decode_step(); m.check_state()
  assert ol.rel_err(a.logits(), b.logits()) <= 2e-3

@pytest.mark.parametrize("dim", [2048, 2304, 4352, 8192, 8448])
def test_prefill_rows_of_every_norm_width(gpu, dim):
  """The norm behind a linear keeps its row in one, two or four vectors per thread (up to 2048, 4096, 8192 values) and is a launch of its own beyond: the same bars as above."""
  cfg = dict(num_blocks=2, dim=dim, hidden_dim=512, n_heads=4, n_kv_heads=2, norm_eps=1e-5, vocab_size=256, head_dim=64, rope_theta=10000.0)
  a, b = _model(cfg, 7, 64), _model(cfg, 7, 64)
  b.prefill_chunk = 1
  prompt = np.random.default_rng(dim).integers(0, 256, size=40).tolist()
  for m in (a, b): m.prefill(prompt)
  assert (a._chunker or a._tail_chunkers[16]).x is None
  for ba, bb in zip(a.blk, b.blk):
    for ca, cb in ((ba.cache_k, bb.cache_k), (ba.cache_v, bb.cache_v)): assert ol.rel_err(ca.numpy().astype(np.float32), cb.numpy().astype(np.float32)) <= 2e-3
  for m in (a, b): m.decode_step()
  assert ol.rel_err(a.logits(), b.logits()) <= 2e-3

@pytest.mark.parametrize("cfg,B,n", [(DENSE, 3, 7), (DENSE, 9, 3), (DENSE, 5, 70), (DENSE128, 2, 33), (MOE, 4, 20), (MOE, 1, 40)], ids=["dense-3x7", "dense-9x3", "dense-5x70", "hd128-2x33", "moe-4x20", "moe-1x40"])
@pytest.mark.parametrize("rows", [2048, 24])
def test_batched_prefill_of_many_rows_vs_step_by_step(gpu, monkeypatch, cfg, B, n, rows):
  """The prompts of several sequences as steps of (sequences x positions) rows against the lockstep steps: every cache within 2e-3 except rows behind a router near-tie (MoE), whose share is
  bounded, and the logits of the first decoded token."""
  from tinygrad_amd import llm
  prompts = np.random.default_rng(B + n).integers(0, cfg["vocab_size"], size=(B, n)).tolist()
  a, b = _model(cfg, 9, 128, B), _model(cfg, 9, 128, B)
  monkeypatch.setattr(llm, "MANY_ROWS", rows)
  a.many_rows, b.many_rows = True, False
  a.prefill(prompts)
  assert a._rows_ws is not None
  b.prefill(prompts)
  assert b._rows_ws is None
  for ba, bb in zip(a.blk, b.blk):
    for nm in ("cache_k", "cache_v"):
      ca, cb = ba[nm].numpy().astype(np.float32), bb[nm].numpy().astype(np.float32)
      off = np.abs(ca - cb).max(axis=(1, 3)) / np.abs(cb).max()                    # per (sequence, position)
      assert not ca[:, :, n - 1:].any() and (off > 2e-3).mean() <= (0.05 if "num_experts" in cfg else 0)
  for m in (a, b): m.decode_step(); m.check_state()
  la, lb = a.logits(), b.logits()
  bad = np.abs(la - lb).max(axis=1) / np.abs(lb).max()
  assert (bad > 2e-3).sum() <= ((B + 3) // 4 if "num_experts" in cfg else 0), bad

@pytest.mark.parametrize("n", [18, 65, 130])
def test_rows_beyond_the_prompt_do_not_count(gpu, n):
  """What an earlier prompt left in the cache beyond this one's positions is never multiplied, finite or not: the caches have the bits of a fresh model's."""
  prompt = np.random.default_rng(n).integers(0, DENSE["vocab_size"], size=n).tolist()
  a, b = _model(DENSE, 11), _model(DENSE, 11)
  for blk in a.blk:
    for cache in (blk.cache_k, blk.cache_v): cache.copyin(np.full(cache.shape, np.nan, np.float16))
  for m in (a, b): m.prefill(prompt)
  for ba, bb in zip(a.blk, b.blk):
    for ca, cb in ((ba.cache_k, bb.cache_k), (ba.cache_v, bb.cache_v)): np.testing.assert_array_equal(ca.numpy()[:, :n - 1], cb.numpy()[:, :n - 1])

@pytest.mark.parametrize("cfg", [DENSE, DENSE128], ids=["hd64", "hd128"])
@pytest.mark.parametrize("n", [194, 257, 471])
def test_attention_of_rows_in_two_parts(gpu, cfg, n):
  """Chains of four tiles of keys and more, which two groups of waves share: rows that see no key of the second group's first tile beside rows that do (prefixes of 5 and 122 positions), an odd and an even number
  of tiles, caches that hold NaN behind the prompt; within 2e-3 of the model prefilled token by token, as above."""
  a, b = _model(cfg, 23, ctx=640), _model(cfg, 23, ctx=640)
  for blk in a.blk:
    for cache in (blk.cache_k, blk.cache_v): cache.copyin(np.full(cache.shape, np.nan, np.float16))
  b.prefill_chunk = 1
  rng = np.random.default_rng(n)
  prompt = rng.integers(0, cfg["vocab_size"], size=n).tolist()
  for keep in (0, 5, 122):
    p = prompt[:keep] + rng.integers(0, cfg["vocab_size"], size=n + keep % 7).tolist()
    for m in (a, b): m.prefill(p)
    for ba, bb in zip(a.blk, b.blk):
      for ca, cb in ((ba.cache_k, bb.cache_k), (ba.cache_v, bb.cache_v)): assert ol.rel_err(ca.numpy()[:, :len(p) - 1].astype(np.float32), cb.numpy()[:, :len(p) - 1].astype(np.float32)) <= 2e-3
    for m in (a, b): m.decode_step(); m.check_state()
    assert ol.rel_err(a.logits(), b.logits()) <= 2e-3
    prompt = p

@pytest.mark.parametrize("k,parts,kw", [(1024, 2, {}), (1536, 3, {}), (2048, 4, {"linear_type": 8}), (2560, 5, {"linear_type": 1}), (3072, 6, {}), (3584, 7, {"q4_k_m": True}), (4096, 8, {}), (5632, 11, {"linear_type": 8})],
                         ids=["2", "3", "4-q8_0", "5-f16", "6", "7-q4_k_m", "8", "11-q8_0"])
@pytest.mark.parametrize("norm", [0, 64])
def test_rotation_completes_the_sums_of_a_split(gpu, k, parts, kw, norm):
  """q / k / v whose K is split into 2 .. 11 parts, which the rotation sums (requested in fours, threes, twos and ones), heads with and without a norm, 24 heads for eight waves, a v of its own type and
  launch; 37 rows: within 2e-3 of the model prefilled token by token, as above."""
  cfg = dict(num_blocks=2, dim=k, hidden_dim=256, n_heads=20, n_kv_heads=4, norm_eps=1e-5, vocab_size=256, head_dim=64, rope_theta=10000.0, qk_norm=norm)
  t = 12 if "q4_k_m" in kw else kw.get("linear_type", 2)
  assert many_tile(t, (1280, 256) if "q4_k_m" in kw else (1280, 256, 256), 37, k)[1] == parts
  from tinygrad_amd.llm import Transformer, TransformerConfig, synth_state
  rng = np.random.default_rng(k)
  c = TransformerConfig(max_context=128, **cfg)
  sd = synth_state(c, seed=29, **kw)
  for blk in range(2):
    for name in ("q", "k"):
      if norm: sd[f"blk.{blk}.attn_{name}_norm.weight"] = (gpu.Buffer.from_numpy((1 + 0.1 * rng.standard_normal(norm)).astype(np.float32)), gpu.F32, (1, norm))
  a, b = Transformer(c, sd, max_new=8), Transformer(c, sd, max_new=8)
  b.prefill_chunk = 1
  p = rng.integers(0, 256, size=38).tolist()
  for m in (a, b): m.prefill(p)
  for ba, bb in zip(a.blk, b.blk):
    for ca, cb in ((ba.cache_k, bb.cache_k), (ba.cache_v, bb.cache_v)): assert ol.rel_err(ca.numpy()[:, :37].astype(np.float32), cb.numpy()[:, :37].astype(np.float32)) <= 2e-3

def _regions(model, cfg, n):
  """q, k, v and the attention's result of the last block in a step's workspace (x, xn, q, k, v, two halves of the query, result: pf_layout)."""
  nq, nk, at, out = cfg["n_heads"] * cfg["head_dim"], cfg["n_kv_heads"] * cfg["head_dim"], 0, {}
  for name, width, dtype in (("x", cfg["dim"], np.float32), ("xn", cfg["dim"], np.float16), ("q", nq, np.float32), ("k", nk, np.float32), ("v", nk, np.float32), ("qh", nq, np.float16), ("ql", nq, np.float16),
                             ("attn", nq, np.float16)):
    out[name] = (model._chunker or model._tail_chunkers[16])._rows_ws.view(at, (n, width), dtype)
    at += (out[name].nbytes + 255) // 256 * 256
  return out

@pytest.mark.parametrize("cfg", [DENSE, DENSE128], ids=["hd64", "hd128"])
def test_cache_rows_have_the_bits_of_the_other_appends(gpu, cfg):
  """A rotated key is the float32 result of one rounded product and one fused multiply-add, then rounded to fp16 (model.py:29-33 as every kernel that appends writes it): the bits of the cache rows,
  from the keys in the step's workspace.  (The exact sum in float64 carries the float32 rounding's ties right: products of two 24-bit numbers and a third one.)"""
  n, hd = 300, cfg["head_dim"]
  a = _model(dict(cfg, num_blocks=1), 17)
  a.prefill(np.random.default_rng(n).integers(0, cfg["vocab_size"], size=n + 1).tolist())
  k = _regions(a, cfg, n)["k"].numpy().reshape(n, -1, hd)
  rope = a.s.rope.numpy().reshape(-1, hd)[:n, None, :]
  x1, x2, c, s = k[..., :hd // 2], k[..., hd // 2:], rope[..., :hd // 2], rope[..., hd // 2:]
  f = np.float64
  ref = np.concatenate([(f(x1) * f(c) - f(x2 * s)).astype(np.float32), (f(x2) * f(c) + f(x1 * s)).astype(np.float32)], -1).astype(np.float16)
  np.testing.assert_array_equal(a.blk[0].cache_k.numpy()[:, :n].view(np.uint16), ref.transpose(1, 0, 2).view(np.uint16))

@pytest.mark.parametrize("cfg", [DENSE, DENSE128], ids=["hd64", "hd128"])
@pytest.mark.parametrize("scale", [0.5, 4.0])
def test_attention_of_rows_is_as_exact_as_the_float32_kernel(gpu, cfg, scale):
  """Attention in float64 over the cache rows and the queries of the workspace: the share of fp16 results that are not its rounded values is no larger than that of the float32 kernel that
  serves eight rows a call.  Bar: 1.15 times and three standard deviations of such a count (they differ by noise where the kernels are equally exact; sums over twice as many additions gave 1.4 times)."""
  from tinygrad_amd.llm import Transformer, TransformerConfig, synth_state
  n, hd, H, KV = 1024, cfg["head_dim"], cfg["n_heads"], cfg["n_kv_heads"]
  c = TransformerConfig(max_context=1088, **dict(cfg, num_blocks=1))
  sd = synth_state(c, seed=19, linear_type=gpu.F16)
  sd["blk.0.attn_norm.weight"][0].view(0, (c.dim,), np.float32).copyin(np.full(c.dim, scale, np.float32))      # scores of standard deviation 0.1 and 5
  a = Transformer(c, sd, max_new=8)
  a.prefill(np.random.default_rng(n).integers(0, cfg["vocab_size"], size=n + 1).tolist())
  reg = _regions(a, cfg, n)
  K, V = (x.numpy()[:, :n].astype(np.float64) for x in (a.blk[0].cache_k, a.blk[0].cache_v))
  q, rope = reg["q"].numpy().astype(np.float64).reshape(n, H, hd), a.s.rope.numpy().reshape(-1, hd)[:n, None, :].astype(np.float64)
  (x1, x2), (cs, sn) = (q[..., :hd // 2], q[..., hd // 2:]), (rope[..., :hd // 2], rope[..., hd // 2:])
  q = np.concatenate([x1 * cs - x2 * sn, x2 * cs + x1 * sn], -1)
  ref = np.empty((n, H, hd))
  for h in range(H):
    s = q[:, h] @ K[h // (H // KV)].T / np.sqrt(hd)
    s[np.triu_indices(n, 1)] = -np.inf
    p = np.exp(s - s.max(1, keepdims=True))
    ref[:, h] = p @ V[h // (H // KV)] / p.sum(1, keepdims=True)
  ref = ref.reshape(n, H * hd).astype(np.float16)
  B, state, part, out = 8, gpu.Buffer((16,), np.int32), gpu.Buffer((8 * H * 17 * (hd + 2),), np.float32).zero_(), gpu.Buffer((8, H * hd), np.float32)
  single = np.empty((n, H * hd), np.float16)
  for at in range(0, n, B):
    st = np.zeros(16, np.int32); st[0], st[3], st[5] = at, n, c.vocab_size
    state.copyin(st)
    gpu.check(gpu.lib().tga_attention_prefill_chunk(B, *[reg[nm].ptr + at * reg[nm].shape[1] * 4 for nm in "qkv"], None, None, c.norm_eps, 0, a.blk[0].cache_k.ptr, a.blk[0].cache_v.ptr, part.ptr, state.ptr,
                                                    H, KV, hd, c.max_context, a.s.rope.ptr, None, out.ptr, None))
    gpu.synchronize(); single[at:at + B] = out.numpy()
  off = [int((x.view(np.uint16) != ref.view(np.uint16)).sum()) for x in (reg["attn"].numpy(), single)]
  print(f"results that are not the rounded exact ones, of {ref.size}: rows {off[0]}, float32 kernel {off[1]}")
  assert off[0] <= 1.15 * off[1] + 3 * off[1] ** 0.5

def test_moe_prompts_keep_their_steps_unless_asked(gpu):
  """A MoE model's prefill computes the bits of steps of sixteen rows (and of lockstep steps): another order of sums turns expert choices at near-ties, so steps of many rows are the user's
  choice there (many_rows), not the default."""
  prompt = np.random.default_rng(3).integers(0, MOE["vocab_size"], size=90).tolist()
  a, b, rows = _model(MOE, 13), _model(MOE, 13), _model(MOE, 13)
  b.prefill_chunk, rows.many_rows = 16, True
  for m in (a, b, rows): m.prefill(prompt)
  for ba, bb in zip(a.blk, b.blk):
    for ca, cb in ((ba.cache_k, bb.cache_k), (ba.cache_v, bb.cache_v)): np.testing.assert_array_equal(ca.numpy(), cb.numpy())
  assert a._chunker.batch == 16 and a._chunker._rows_ws is None and rows._tail_chunkers[16]._rows_ws is not None
  batch = _model(MOE, 13, 128, 4)
  batch.prefill([prompt] * 4)
  assert batch._rows_ws is None

# ---- expert products: models whose embeddings decide the routing (no near-ties: the rows path and the steps agree at every position)
def _blocks_of_unit_gain(rng, rt, t, n, k):
  """(n, k) random blocks whose weights are about k ** -0.5."""
  if t == rt.F16: return (rng.standard_normal((n, k)) * k ** -0.5).astype(np.float16).view(np.uint8).reshape(-1)
  if t == rt.MXFP4: return synth.random_blocks(rng, t, n, k, mx_exp=(120, 124))
  seed, sigma = rng.integers(1 << 30), 0.003
  std = og.ggml_data_to_tensor(synth.random_blocks(np.random.default_rng(seed), t, n, k, sigma), n * k, t).std()
  return synth.random_blocks(np.random.default_rng(seed), t, n, k, sigma * k ** -0.5 / float(std))

def _routed(rt, seed=23, expert_type=None, gate=0.2, **over):
  """(config, state) of a MoE model in which token t goes to expert t % E first and to another one, given by t // E, second; experts add about as much to a row as its embedding has."""
  from tinygrad_amd.llm import TransformerConfig, synth_state_moe
  c = TransformerConfig(max_context=1152, **dict(MOE, **over))
  sd = synth_state_moe(c, seed=seed)
  rng, E, D, H = np.random.default_rng(seed), c.num_experts, c.dim, c.hidden_dim
  u = np.linalg.qr(rng.standard_normal((D, E)))[0].T * D ** 0.5                       # E directions, orthogonal, unit root mean square
  t = np.arange(c.vocab_size)
  first, second = t % E, (t % E + 1 + t // E % (E - 1)) % E
  put = lambda name, a, dt=np.float16: sd[name][0].view(0, a.shape, dt).copyin(a.astype(dt))
  put("token_embd.weight", 0.3 * (0.2 * rng.standard_normal((c.vocab_size, D)) + 0.8 * u[first] + 0.5 * u[second]))
  for i in range(c.num_blocks):
    p = f"blk.{i}."
    put(p + "attn_output.weight", 0.1 * rng.standard_normal((D, c.n_heads * c.head_dim)) * (c.n_heads * c.head_dim) ** -0.5)
    if i < c.leading_dense_blocks: continue
    put(p + "ffn_gate_inp.weight", gate * u * 10 / D)
    for nm, n, k in (("ffn_gate_exps", H, D), ("ffn_up_exps", H, D), ("ffn_down_exps", D, H)):
      if expert_type is None: continue
      sd[p + nm + ".weight"] = (rt.Buffer.from_numpy(np.concatenate([_blocks_of_unit_gain(rng, rt, expert_type, n, k) for _ in range(E)])), expert_type, (E, n, k))
  return c, sd

def _rows_and_steps_agree(rt, c, sd, prompt):
  """The prompt as steps of many rows and as the steps a MoE model takes by default: caches and logits within the bars of the dense models.  Returns the model of many rows."""
  from tinygrad_amd.llm import Transformer
  a, b = Transformer(c, sd, max_new=8), Transformer(c, sd, max_new=8)
  a.many_rows, b.many_rows = True, False
  for m in (a, b): m.prefill(prompt)
  chunker = a._chunker or a._tail_chunkers[16]
  assert chunker.x is None and chunker._rows_ws is not None
  for ba, bb in zip(a.blk, b.blk):
    for ca, cb in ((ba.cache_k, bb.cache_k), (ba.cache_v, bb.cache_v)):
      ca, cb = ca.numpy().astype(np.float32), cb.numpy().astype(np.float32)
      assert np.isfinite(ca).all() and ol.rel_err(ca, cb) <= 2e-3
  for m in (a, b): m.decode_step(); m.check_state()
  assert ol.rel_err(a.logits(), b.logits()) <= 2e-3
  return a

@pytest.mark.parametrize("counts", [(0, 1, 31, 32, 33, 65, 63, 31), (0, 1, 63, 64, 65, 129, 33, 32), (0, 1, 127, 128, 129, 257, 64, 100), (0, 0, 0, 700, 0, 0, 70, 10)], ids=["32", "64", "128", "skewed"])
def test_expert_tiles_of_every_height(gpu, counts):
  """Expert counts of no row, one, and one less and more than the tiles of 32, 64 and 128 rows that the average count asks for."""
  c, sd = _routed(gpu, num_experts_per_tok=1)
  E = c.num_experts
  rng = np.random.default_rng(sum(counts))
  cls = rng.permutation(np.repeat(np.arange(E), counts))
  prompt = [int(e + E * rng.integers(0, c.vocab_size // E)) for e in cls]
  _rows_and_steps_agree(gpu, c, sd, prompt + [3])                                   # (what block 0's experts add is in the keys and values of block 1)
  from tinygrad_amd.llm import Transformer
  a = Transformer(dataclasses.replace(c, num_blocks=1), sd, max_new=8)
  a.many_rows = True
  a.prefill(prompt + [3])
  n, up = len(prompt), lambda b: (b + 255) // 256 * 256
  r = _regions(a, MOE, n)
  at = sum(up(b.nbytes) for b in r.values()) + up(2 * n) + (64 << 20) + up(4 * n * E) + 3 * up(4 * n)        # (activations, partial sums, logits; selection, weights, places)
  assert (a._chunker or a._tail_chunkers[16])._rows_ws.view(at, (E,), np.int32).numpy().tolist() == list(counts)

@pytest.mark.parametrize("fmt", FORMATS)
def test_experts_of_every_format(gpu, fmt):
  """Expert matrices of every format the rows linears take, at tiles of 32 and of 64 rows."""
  c, sd = _routed(gpu, expert_type=getattr(gpu, fmt))
  rng = np.random.default_rng(1)
  for n in (70, 200): _rows_and_steps_agree(gpu, c, sd, rng.integers(0, c.vocab_size, size=n).tolist())

@pytest.mark.parametrize("over", [dict(expert_gating_func=2), dict(expert_gating_func=3), dict(expert_gating_func=4), dict(norm_topk_prob=True), dict(expert_gating_func=2, norm_topk_prob=True, routed_scaling_factor=2.5),
                                  dict(leading_dense_blocks=1, dense_hidden_dim=512, num_blocks=3), dict(head_dim=128, n_heads=2, n_kv_heads=2)],
                         ids=["sigmoid", "softmax of the picked", "sqrt softplus", "normed", "sigmoid, normed, scaled", "dense block first", "heads of 128"])
def test_routed_rows_of_other_kinds(gpu, over):
  c, sd = _routed(gpu, **over)
  _rows_and_steps_agree(gpu, c, sd, np.random.default_rng(2).integers(0, c.vocab_size, size=150).tolist())

@pytest.mark.parametrize("cfg", [DENSE, DENSE128], ids=["hd64", "hd128"])
def test_prefill_rows_with_norms_per_head(gpu, cfg):
  """q / k norms over each head (their weights differ from value to value) against the model prefilled token by token."""
  from tinygrad_amd.llm import Transformer, TransformerConfig, synth_state
  c = TransformerConfig(max_context=256, qk_norm=cfg["head_dim"], **cfg)
  sd, rng = synth_state(c, seed=29), np.random.default_rng(29)
  for i in range(c.num_blocks):
    for nm in ("q", "k"): sd[f"blk.{i}.attn_{nm}_norm.weight"] = (gpu.Buffer.from_numpy(rng.uniform(0.5, 2, c.head_dim).astype(np.float32)), gpu.F32, (1, c.head_dim))
  prompt = rng.integers(0, c.vocab_size, size=140).tolist()
  a, b = Transformer(c, sd, max_new=8), Transformer(c, sd, max_new=8)
  b.prefill_chunk = 1
  for m in (a, b): m.prefill(prompt)
  assert a._chunker._rows_ws is not None
  for ba, bb in zip(a.blk, b.blk):
    for ca, cb in ((ba.cache_k, bb.cache_k), (ba.cache_v, bb.cache_v)): assert ol.rel_err(ca.numpy().astype(np.float32), cb.numpy().astype(np.float32)) <= 2e-3
  for m in (a, b): m.decode_step(); m.check_state()
  assert ol.rel_err(a.logits(), b.logits()) <= 2e-3

def test_prompts_without_memory_for_their_rows_take_the_smaller_steps(gpu, monkeypatch):
  """No memory for the buffers of a step of many rows (277 MB at the 8B architecture's widths): the prompt is prefilled in the steps that need a few MB, for one sequence and for several."""
  from tinygrad_amd import llm
  prompt = np.random.default_rng(4).integers(0, DENSE["vocab_size"], size=150).tolist()
  a, b, several, several_b = _model(DENSE, 31), _model(DENSE, 31), _model(DENSE, 31, 160, 4), _model(DENSE, 31, 160, 4)
  b.many_rows = several_b.many_rows = False
  b.prefill(prompt); several_b.prefill([prompt[:40]] * 4)
  buffer = llm.Buffer
  def none_left(shape, dtype=np.uint8, **kw):
    if int(np.prod(shape)) * np.dtype(dtype).itemsize >= 60 << 20: raise RuntimeError("HIP Error 2, out of memory  [hipMalloc(ptr, cls) at pool.h:1]")
    return buffer(shape, dtype, **kw)
  none_left.from_numpy = buffer.from_numpy
  monkeypatch.setattr(llm, "Buffer", none_left)
  a.prefill(prompt); several.prefill([prompt[:40]] * 4)
  assert a._chunker._rows_ws is None and a._chunker.x is not None and several._rows_ws is None
  for ba, bb in zip(a.blk, b.blk): np.testing.assert_array_equal(ba.cache_k.numpy(), bb.cache_k.numpy())
  for ba, bb in zip(several.blk, several_b.blk): np.testing.assert_array_equal(ba["cache_k"].numpy(), bb["cache_k"].numpy())
