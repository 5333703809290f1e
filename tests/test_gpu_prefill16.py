"""Prompts of MoE models in steps of many rows whose sums run in the order of the steps of sixteen, eight and four rows (csrc/prefill16.hip): caches and logits have those steps' bits."""
import numpy as np, pytest

pytestmark = pytest.mark.gpu
BASE = dict(norm_eps=1e-5, vocab_size=512, rope_theta=10000.0)
# the rows of the dense linears dealt to eight waves (2048, 1024) and to four (1536: two rounds; 512: waves without a step), experts of 64, 48, 32, 24 and 8 units, heads of 64 and 128, query groups
CONFIGS = {
  "2048x1024": dict(num_blocks=3, dim=2048, hidden_dim=1024, n_heads=16, n_kv_heads=16, head_dim=128, qk_norm=2048, num_experts=64, num_experts_per_tok=8, **BASE),
  "1536x768": dict(num_blocks=2, dim=1536, hidden_dim=768, n_heads=12, n_kv_heads=12, head_dim=128, qk_norm=1536, num_experts=16, num_experts_per_tok=4, norm_topk_prob=True, **BASE),
  "1024x1536": dict(num_blocks=2, dim=1024, hidden_dim=1536, n_heads=16, n_kv_heads=4, head_dim=64, qk_norm=1024, num_experts=32, num_experts_per_tok=2, expert_gating_func=2, **BASE),
  "512x256": dict(num_blocks=3, dim=512, hidden_dim=256, n_heads=8, n_kv_heads=8, head_dim=64, qk_norm=512, num_experts=8, num_experts_per_tok=1, **BASE),
}

def _models(cfg, seed, ctx):
  from tinygrad_amd.llm import Transformer, TransformerConfig, synth_state_moe
  c = TransformerConfig(max_context=ctx, **cfg)
  sd = synth_state_moe(c, seed=seed)
  return Transformer(c, sd, max_new=8), Transformer(c, sd, max_new=8)

@pytest.mark.parametrize("name", list(CONFIGS))
@pytest.mark.parametrize("n,rows", [(17, 1024), (30, 1024), (78, 32), (134, 1024), (333, 128)])
def test_bits_of_the_steps_of_sixteen_rows(gpu, monkeypatch, name, n, rows):
  """Positions 16, 28 (16 + 8 + 4), 76, 132 and 332 in one step and in several: every key and value of every block, the logits behind them, and a follow-up prompt that keeps a prefix."""
  from tinygrad_amd import llm
  cfg = CONFIGS[name]
  a, b = _models(cfg, 11 + n, 384)
  prompt = np.random.default_rng(n).integers(0, cfg["vocab_size"], size=n).tolist()
  for p in (prompt, prompt[:n // 2] + [7] * 40):
    monkeypatch.setattr(llm, "ROWS16", rows); monkeypatch.setattr(llm, "ROWS16_MIN", 1)
    a.prefill(p)
    assert a._chunker._rows16_ws is not None and a._chunker.x is None        # (no step of sixteen was run)
    monkeypatch.setattr(llm, "ROWS16_MIN", 1 << 30)
    b.prefill(p)
    assert b._chunker is None or b._chunker._rows16_ws is None
    for i, (ba, bb) in enumerate(zip(a.blk, b.blk)):
      for ca, cb in ((ba.cache_k, bb.cache_k), (ba.cache_v, bb.cache_v)):
        diff = int((ca.numpy().view(np.uint16) != cb.numpy().view(np.uint16)).sum())
        assert diff == 0, f"block {i}"
    for m in (a, b): m.decode_step(); m.check_state()
    diff = int((a.logits().view(np.uint32) != b.logits().view(np.uint32)).sum())
    assert diff == 0

def _same_bits(a, b, n):
  for i, (ba, bb) in enumerate(zip(a.blk, b.blk)):
    for ca, cb in ((ba.cache_k, bb.cache_k), (ba.cache_v, bb.cache_v)): assert (ca.numpy().view(np.uint16)[:, :n - 1] == cb.numpy().view(np.uint16)[:, :n - 1]).all(), f"block {i}"
  for m in (a, b): m.decode_step(); m.check_state()
  assert (a.logits().view(np.uint32) == b.logits().view(np.uint32)).all()

# the rest of the range: attention rows of other widths than the residual's (attn_output over 9, 10, 12 and 16 steps of 256, dealt to four and to eight waves), and contexts of more than 24 splits
WIDE = {f"{h}x{hd}": dict(num_blocks=2, dim=512, hidden_dim=256, n_heads=h, n_kv_heads=kv, head_dim=hd, qk_norm=h * hd, num_experts=16, num_experts_per_tok=2, **BASE)
        for h, kv, hd in ((18, 6, 128), (40, 8, 64), (24, 24, 128), (32, 8, 128))}
LONG = {f"long-{h}x{hd}": dict(num_blocks=2, dim=512, hidden_dim=256, n_heads=h, n_kv_heads=h // 2, head_dim=hd, qk_norm=h * hd, num_experts=16, num_experts_per_tok=2, **BASE) for h, hd in ((8, 64), (4, 128))}

# gating by way of LDS: few experts of which many are taken, and more experts than a workgroup has lanes
MANY = {f"{e}-experts": dict(num_blocks=2, dim=512, hidden_dim=256, n_heads=8, n_kv_heads=8, head_dim=64, qk_norm=512, num_experts=e, num_experts_per_tok=k, **BASE) for e, k in ((24, 18), (80, 8), (300, 3))}

@pytest.mark.parametrize("name,n", [(name, 95) for name in {**WIDE, **MANY}] + [(name, 1667) for name in LONG])
def test_bits_over_the_rest_of_the_range(gpu, monkeypatch, name, n):
  """94 positions of wide attention rows, and of experts that are gated four or eight tokens a workgroup; 1666 positions (27 splits of 64, two steps: 1024 rows and 642 with the tail of eight)."""
  from tinygrad_amd import llm
  a, b = _models({**WIDE, **MANY, **LONG}[name], 5 + n, 128 if n < 128 else 2048)
  prompt = np.random.default_rng(n).integers(0, BASE["vocab_size"], size=n).tolist()
  a.prefill(prompt)
  assert a._chunker._rows16_ws is not None and a._chunker.x is None
  monkeypatch.setattr(llm, "ROWS16_MIN", 1 << 30)
  b.prefill(prompt)
  assert b._chunker._rows16_ws is None
  _same_bits(a, b, n)

def test_bits_of_steps_that_memory_cuts(gpu, monkeypatch):
  """Buffers bounded to less than a prompt's rows need (steps of fewer rows, a multiple of sixteen each), and no memory for them at all (the steps of sixteen)."""
  from tinygrad_amd import llm
  n = 300
  prompt = np.random.default_rng(n).integers(0, BASE["vocab_size"], size=n).tolist()
  a, b = _models(CONFIGS["512x256"], n, 384)
  c, d = _models(CONFIGS["512x256"], n, 384)
  real, sizes = llm.Buffer, []
  class Counted(real):
    def __init__(self, shape, *args, **kw):
      sizes.append(int(np.prod(shape))); super().__init__(shape, *args, **kw)
  monkeypatch.setattr(llm, "ROWS16_BYTES", 1 << 20); monkeypatch.setattr(llm, "Buffer", Counted)
  a.prefill(prompt)
  monkeypatch.setattr(llm, "Buffer", real)
  ws = a._chunker._rows16_ws
  assert ws is not None and a._chunker.x is None and ws.nbytes in sizes
  monkeypatch.setattr(llm, "ROWS16_BYTES", 1 << 29)
  c.prefill(prompt)
  assert ws.nbytes < c._chunker._rows16_ws.nbytes // 2
  def none(shape, *args, **kw):
    if int(np.prod(shape)) == c._chunker._rows16_ws.nbytes: raise RuntimeError("HIP Error 2, out of memory")
    return real(shape, *args, **kw)
  monkeypatch.setattr(llm, "Buffer", none)
  d.prefill(prompt)
  monkeypatch.setattr(llm, "Buffer", real)
  assert d._chunker._rows16_ws is None and d._chunker.x is not None
  monkeypatch.setattr(llm, "ROWS16_MIN", 1 << 30)
  for m in (a, c, d):
    b.prefill(prompt)
    _same_bits(m, b, n)

@pytest.mark.parametrize("over", [dict(expert_gating_func=f, norm_topk_prob=n, routed_scaling_factor=r) for f in (1, 2, 3, 4) for n, r in ((False, 2.5), (True, 1.0), (True, 2.5))],
                         ids=lambda o: "-".join(str(v) for v in o.values()))
def test_bits_of_every_gating(gpu, monkeypatch, over):
  """Softmax, sigmoid, softmax of the picked and sqrt softplus, weights normed and scaled or not; every expert's router row is there twice, so picks are ties."""
  from tinygrad_amd import llm
  from tinygrad_amd.llm import Transformer, TransformerConfig, synth_state_moe
  c = TransformerConfig(max_context=192, **dict(CONFIGS["512x256"], num_experts=24, num_experts_per_tok=5, **over))
  sd = synth_state_moe(c, seed=41)
  for i in range(c.num_blocks):
    r = sd[f"blk.{i}.ffn_gate_inp.weight"][0].view(0, (24, c.dim), np.float16)
    w = r.numpy(); w[1::2] = w[::2]; r.copyin(w)
  a, b = Transformer(c, sd, max_new=8), Transformer(c, sd, max_new=8)
  prompt = np.random.default_rng(41).integers(0, BASE["vocab_size"], size=150).tolist()
  a.prefill(prompt)
  assert a._chunker._rows16_ws is not None and a._chunker.x is None
  monkeypatch.setattr(llm, "ROWS16_MIN", 1 << 30)
  b.prefill(prompt)
  _same_bits(a, b, 150)

@pytest.mark.parametrize("name", list(CONFIGS))
def test_bits_with_norm_weights_of_any_value(gpu, monkeypatch, name):
  """Norm weights that are no powers of two (the synthetic models' are 1): a normalised value is rounded where the steps of sixteen, eight and four rows round it."""
  from tinygrad_amd import llm
  from tinygrad_amd.llm import Transformer, TransformerConfig, synth_state_moe
  cfg, rng, n = CONFIGS[name], np.random.default_rng(37), 350
  c = TransformerConfig(max_context=384, **cfg)
  sd = synth_state_moe(c, seed=37)
  for key, (b, _, shape) in sd.items():
    if key.endswith("norm.weight"): b.view(0, shape, np.float32).copyin((rng.uniform(0.3, 3, shape) * rng.choice([-1, 1], shape)).astype(np.float32))
  for m in (n, n - 26, 140):                                                        # (349, 323 and 139 positions: behind the steps of sixteen 8 + 4 + 1, 3 and 8 + 3)
    prompt = rng.integers(0, cfg["vocab_size"], size=m).tolist()
    a, b = Transformer(c, sd, max_new=8), Transformer(c, sd, max_new=8)
    monkeypatch.setattr(llm, "ROWS16_MIN", 16)
    a.prefill(prompt)
    monkeypatch.setattr(llm, "ROWS16_MIN", 1 << 30)
    b.prefill(prompt)
    assert a._chunker._rows16_ws is not None and b._chunker._rows16_ws is None
    _same_bits(a, b, m)

@pytest.mark.parametrize("name", list(CONFIGS))
def test_expert_products_of_values_of_every_size(gpu, monkeypatch, name):
  """The experts' products are matrix-core products of two values with zeros beside them, in place of v_dot2_f32_f16: the bits over activations from subnormal fp16 numbers to 2^13 in one sum (norm
  weights of 2^-24 .. 2^12, both signs) and over hidden values as far apart (block scales of 2^-26 .. 2^-14)."""
  from tinygrad_amd import llm
  from tinygrad_amd.llm import Transformer, TransformerConfig, synth_state_moe
  cfg, rng = CONFIGS[name], np.random.default_rng(31)
  c = TransformerConfig(max_context=192, **cfg)
  sd = synth_state_moe(c, seed=31)
  for i in range(c.num_blocks):
    w = (2.0 ** rng.uniform(-24, 12, c.dim) * rng.choice([-1, 1], c.dim)).astype(np.float32)
    sd[f"blk.{i}.ffn_norm.weight"][0].view(0, (c.dim,), np.float32).copyin(w)
    for nm in ("gate", "up"):
      b = sd[f"blk.{i}.ffn_{nm}_exps.weight"][0]
      raw = b.numpy().view(np.uint8).reshape(-1, 17)
      raw[:, 0] = 127 - rng.integers(14, 27, len(raw) // (c.dim // 32)).repeat(c.dim // 32)      # (a scale for each row: rows of the hidden layer lie apart)
      b.copyin(raw.reshape(b.shape))
  prompt = rng.integers(0, cfg["vocab_size"], size=125).tolist()
  a, b = Transformer(c, sd, max_new=8), Transformer(c, sd, max_new=8)
  a.prefill(prompt)
  monkeypatch.setattr(llm, "ROWS16_MIN", 1 << 30)
  b.prefill(prompt)
  assert a._chunker._rows16_ws is not None and b._chunker._rows16_ws is None and np.isfinite(b.blk[-1].cache_v.numpy()).all()
  _same_bits(a, b, 125)

def test_one_step_of_sixteen_stays_one(gpu):
  """Sixteen to nineteen positions are one step of sixteen rows (a graph) and single ones; from twenty on, or where a row's experts have many hidden values, all rows go together."""
  wide = dict(CONFIGS["512x256"], hidden_dim=1536, num_experts_per_tok=8, num_blocks=1)
  for cfg, n, together in ((CONFIGS["512x256"], 17, False), (CONFIGS["512x256"], 20, False), (CONFIGS["512x256"], 21, True), (wide, 16, False), (wide, 17, True), (wide, 20, True)):
    m = _models(cfg, n, 64)[0]
    m.prefill(list(range(n)))
    assert (m._chunker is not None and m._chunker._rows16_ws is not None) == together, (n, together)

@pytest.mark.parametrize("name", ["1536x768", "512x256"])
@pytest.mark.parametrize("n,at", [(40, 21), (100, 70), (333, 200)])
def test_values_that_are_not_finite_stay_with_later_positions(gpu, name, n, at):
  """A token whose value in one column leaves the fp16 range: the keys and values of the positions in front of it are those of a prompt that has another token there, in every block."""
  from tinygrad_amd.llm import Transformer, TransformerConfig, synth_state_moe
  cfg = dict(CONFIGS[name], num_blocks=3)
  c = TransformerConfig(max_context=384, **cfg)
  sd = synth_state_moe(c, seed=n)
  def edit(key, f):
    b, _, shape = sd[key]
    w = b.numpy().view(np.float16).reshape(shape); f(w); b.copyin(w.view(np.uint8).reshape(b.shape).view(b.dtype))
  def column(w): w[:, 0] = 0; w[5, 0] = 100
  def row(w): w[0, 0] = 60000
  edit("token_embd.weight", column); edit("blk.0.attn_v.weight", row)            # (only token 5 has anything in column 0, and 60000 times that is infinite)
  prompt = np.random.default_rng(n).integers(6, cfg["vocab_size"], size=n).tolist()
  other = prompt[:at] + [5] + prompt[at + 1:]
  a, b = Transformer(c, sd, max_new=8), Transformer(c, sd, max_new=8)
  a.prefill(other); b.prefill(prompt)
  assert a._chunker._rows16_ws is not None and np.isinf(a.blk[0].cache_v.numpy()[0, at, 0])
  for ba, bb in zip(a.blk, b.blk):
    for ca, cb in ((ba.cache_k, bb.cache_k), (ba.cache_v, bb.cache_v)):
      ca, cb = ca.numpy()[:, :at], cb.numpy()[:, :at]
      assert np.isfinite(cb).all(); np.testing.assert_array_equal(ca.view(np.uint16), cb.view(np.uint16))

@pytest.mark.parametrize("name,n,ctx", [("2048x1024", 22, 576), ("2048x1024", 40, 1024), ("1536x768", 23, 128), ("1024x1536", 136, 256), ("1024x1536", 1399, 2048), ("512x256", 206, 768), ("512x256", 259, 1600), ("512x256", 132, 136)])
def test_bits_of_the_last_positions(gpu, monkeypatch, name, n, ctx):
  """The one to three positions behind a prompt's last step of four together (tga_prefill16_tail) against single steps: one, two and three tiles of attention per split, rows on either side of a split's
  edge (the second prompt of 206: 127, 128, 129), a cache that ends soon behind the prompt, and prompts that keep a prefix and leave another number of them."""
  from tinygrad_amd import llm
  a, b = _models(CONFIGS[name], 3 + n, ctx)
  prompt = np.random.default_rng(n).integers(0, BASE["vocab_size"], size=n).tolist()
  for p in (prompt, prompt[:n // 2] + [9] * 28, prompt[:n - 1]):
    if len(p) >= ctx: continue
    for m, least in ((a, 1), (b, 1 << 30)):
      monkeypatch.setattr(llm, "ROWS16_TAIL", least)
      m.prefill(p, reuse_cache=p is not prompt[:n - 1])
      m.check_state()
    assert a._chunker._rows16_ws is not None and b._chunker._rows16_ws is not None
    for i, (ba, bb) in enumerate(zip(a.blk, b.blk)):
      for ca, cb in ((ba.cache_k, bb.cache_k), (ba.cache_v, bb.cache_v)): assert (ca.numpy().view(np.uint16) == cb.numpy().view(np.uint16)).all(), f"block {i}"
    _same_bits(a, b, len(p))
