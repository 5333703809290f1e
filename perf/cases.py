"""The work a program has this framework do, as measurable cases: stand-alone linears over GGUF blocks, block dequantisation, MXFP8 quantisation, the grouped
MXFP8 MoE feed-forward, and whole models (a prompt to its first logits, the next token of a context that is in the cache, several sequences in lockstep).

A case is a dict of plain values; `kind` picks the path, the other fields are its sizes.  listed() holds the sizes the repository's own configurations, tests
and benchmark name (the 8B llama architecture, the 64-expert MoE architecture, the grouped feed-forward); draw() gives other sizes of the same ranges.
Every call goes through the public entry points with the buffers a program would keep: weights, models and result buffers are made in prepare(), results that
the entry point allocates are allocated in run()."""
import math
import numpy as np
import torch
from tinygrad_amd import moe, runtime as rt
from tinygrad_amd.gguf import ggml_data_to_tensor
from tinygrad_amd.llm import BatchedTransformer, LLAMA3_8B, OLMOE, Transformer, TransformerConfig, synth_state, synth_state_moe
from tinygrad_amd.nn import QuantLinear
from tinygrad_amd.runtime import Buffer, GGML_QUANT

TYPES = {"q4_0": rt.Q4_0, "q4_1": rt.Q4_1, "q5_0": rt.Q5_0, "q5_1": rt.Q5_1, "q8_0": rt.Q8_0, "q4_k": rt.Q4_K, "q5_k": rt.Q5_K, "q6_k": rt.Q6_K, "iq4_xs": rt.IQ4_XS,
         "iq3_xxs": rt.IQ3_XXS, "iq3_s": rt.IQ3_S, "iq2_s": rt.IQ2_S, "q1_0": rt.Q1_0, "mxfp4": rt.MXFP4, "f16": rt.F16}
# The types that model files hold most: drawn three times as often as the rest
COMMON = ["q4_0", "q8_0", "q4_k", "q5_k", "q6_k", "f16"]
FLOATS = {"f16": (torch.float16, np.float16), "f32": (torch.float32, np.float32)}


def listed():
  llama = dict(arch="llama", blocks=32, dim=4096, hidden=14336, heads=32, kv_heads=8, head_dim=128, vocab=128256)
  olmoe = dict(arch="moe", blocks=16, dim=2048, hidden=1024, heads=16, kv_heads=16, head_dim=128, vocab=50304, experts=64, topk=8)
  return [
    # the smallest call: one attention projection of the 8B architecture on one row
    dict(name="linear_q4_0_row", kind="linear", type="q4_0", n=4096, k=4096, m=1, x="f16", y="f16"),
    # the 8B architecture's lm-head on the rows of a small batch
    dict(name="linear_q6_k_head_rows", kind="linear", type="q6_k", n=128256, k=4096, m=4, x="f16", y="f16"),
    # one ffn matrix expanded while a model is loaded into a program that wants plain values
    dict(name="dequant_q4_k", kind="dequant", type="q4_k", n=14336, k=4096, y="f16"),
    # activations of a long sequence on their way into an MXFP8 product
    dict(name="mxfp8_quantize_rows", kind="quantize", op="rows", rows=16384, k=4096),
    # the MoE feed-forward of a prefill: 2000 tokens, top-8 of 64 experts, skewed popularity
    dict(name="moe_ffn_prefill", kind="moe_ffn", tokens=2000, dim=2048, inter=512, experts=64, topk=8, zipf=1.1),
    # such a layer on the tokens of a decode batch
    dict(name="moe_ffn_decode", kind="moe_ffn", tokens=32, dim=2048, inter=768, experts=64, topk=8, zipf=1.1),
    # the next token of a single 8B sequence (the headline benchmark's shape)
    dict(name="decode_8b_q4_0", kind="decode", weights="q4_0", prompt=1024, **llama),
    # the next token of a single sequence of the MoE architecture
    dict(name="decode_olmoe", kind="decode", weights="mxfp4", prompt=512, **olmoe),
    # a new 1024-token prompt up to its first logits
    dict(name="prefill_8b_q4_0", kind="prefill", weights="q4_0", prompt=1024, **llama),
    dict(name="prefill_olmoe", kind="prefill", weights="mxfp4", prompt=512, **olmoe),
    # four new prompts in lockstep up to their first logits, the tensor types of a Q4_K_M file
    dict(name="batch_prompts_8b_q4_k_m", kind="batch", weights="q4_k_m", batch=4, prompt=128, **llama),
    # one lockstep step: eight sequences from their first token
    dict(name="batch_step_8b_q8_0", kind="batch", weights="q8_0", batch=8, prompt=1, **llama),
  ]


def _log(rng, lo, hi): return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

def _draw_model(rng, kind):
  head_dim = rng.choice([64, 128, 128])
  if kind != "moe":
    kv = rng.choice([2, 4, 4, 8])
    heads = kv * rng.choice([1, 2, 4, 4])
    while heads * head_dim % 256 or heads * head_dim < 512: heads += kv
    dim = heads * head_dim
    return dict(arch="llama", weights=rng.choice(["q4_0", "q4_0", "q8_0", "q4_k_m", "q4_k_m", "f16"]), blocks=rng.randint(2, 16), dim=dim, hidden=256 * rng.randint(dim * 5 // 512, dim * 7 // 512),
                heads=heads, kv_heads=kv, head_dim=head_dim, vocab=_log(rng, 8000, 128256))
  heads = rng.choice([8, 12, 16]) * (128 // head_dim)
  return dict(arch="moe", weights="mxfp4", blocks=rng.randint(2, 10), dim=heads * head_dim, hidden=256 * rng.randint(2, 6), heads=heads, kv_heads=heads, head_dim=head_dim,
              vocab=_log(rng, 8000, 65536), experts=rng.choice([16, 32, 64]), topk=rng.choice([2, 4, 8]))

def draw(rng):
  kind = rng.choice(["linear", "linear", "dequant", "quantize", "moe_ffn", "moe_ffn", "decode", "prefill", "prefill", "batch"])
  if kind == "linear":
    return dict(kind=kind, type=rng.choice(3 * COMMON + sorted(TYPES)), n=_log(rng, 33, 32768), k=256 * _log(rng, 1, 56), m=_log(rng, 1, 128), x=rng.choice(["f16", "f16", "f32"]), y=rng.choice(["f16", "f32"]))
  if kind == "dequant": return dict(kind=kind, type=rng.choice(COMMON[:-1] + sorted(set(TYPES) - {"f16"})), n=_log(rng, 1, 32768), k=256 * _log(rng, 1, 28), y=rng.choice(["f16", "f32"]))
  if kind == "quantize":
    op = rng.choice(["rows", "rows_f32", "swiglu", "transpose"])
    if op == "transpose": return dict(kind=kind, op=op, rows=32 * _log(rng, 1, 256), k=64 * _log(rng, 2, 100))
    return dict(kind=kind, op=op, rows=_log(rng, 1, 8192), k=32 * _log(rng, 8, 200))
  if kind == "moe_ffn":
    # rows padded to 256 per expert x inter stays within 2^24, where every result is right: swiglu() returns wrong values beyond (of the 128 x 768 layer of the grouped
    # GEMM benchmark, for one), so a larger layer has nothing to be compared with
    tokens, dim, inter = _log(rng, 1, 4096), 256 * rng.randint(2, 8), 256 * rng.randint(1, 3)
    experts, topk = rng.choice([8, 16, 32, 64, 80]), rng.choice([1, 2, 4, 6, 8])
    while moe.m_max_for(tokens, topk, experts) * inter > 1 << 24:
      if inter > 256: inter -= 256
      else: tokens = tokens * 3 // 4
    return dict(kind=kind, tokens=tokens, dim=dim, inter=inter, experts=experts, topk=topk, zipf=rng.choice([0.0, 0.6, 1.1]))
  model = _draw_model(rng, rng.choice(["llama", "llama", "moe"]))
  if kind == "batch": return dict(kind=kind, batch=rng.randint(2, 16), prompt=_log(rng, 1, 96), **model)
  return dict(kind=kind, prompt=_log(rng, 9, 1024 if model["arch"] == "llama" else 512), **model)


# ---- inputs
def _gen(seed): return torch.Generator(device="cuda").manual_seed(int(seed))

def _buffer(t: torch.Tensor, dtype) -> Buffer:
  """A window of the framework on a tensor's memory."""
  return Buffer(tuple(t.shape), dtype, ptr=t.data_ptr(), owner=t)

class _Exported:
  """A result buffer under the array-interface protocol (the tensor made from it keeps it alive)."""
  def __init__(self, b: Buffer, typestr: str):
    self.buffer, self.__cuda_array_interface__ = b, dict(shape=b.shape, typestr=typestr, data=(b.ptr, False), strides=None, version=3)

def _tensor(b: Buffer, dtype=None) -> torch.Tensor:
  t = torch.as_tensor(_Exported(b, "<i2" if dtype == torch.bfloat16 else np.dtype(b.dtype).str), device="cuda")
  return t.view(dtype) if dtype is not None else t

def _blocks(gen, ggml_type: int, n: int, k: int) -> torch.Tensor:
  """(n, k) weights as GGUF block bytes: uniform payload bytes and scales that make a weight about k ** -0.5 (what tinygrad_amd.synth writes on the host)."""
  if ggml_type == rt.F16: return (torch.randn((n, k), generator=gen, device="cuda") * k ** -0.5).half().view(torch.uint8).reshape(-1)
  nel, nby = GGML_QUANT[ggml_type]
  nb = n * (k // nel)
  b = torch.randint(0, 256, (nb, nby), generator=gen, device="cuda", dtype=torch.uint8)
  def scale(s): return (torch.randn(nb, generator=gen, device="cuda").abs() * s + s / 4).half().view(torch.uint8).reshape(nb, 2)
  s = k ** -0.5
  per = {rt.Q4_0: 1 / 5, rt.Q4_1: 1 / 5, rt.Q5_0: 1 / 9, rt.Q5_1: 1 / 9, rt.Q8_0: 1 / 74, rt.Q4_K: 1 / 250, rt.Q5_K: 1 / 500, rt.Q6_K: 1 / 1400, rt.IQ4_XS: 1 / 1200, rt.IQ3_XXS: 1 / 180, rt.IQ3_S: 1 / 120,
         rt.IQ2_S: 1 / 60, rt.Q1_0: 1.0}
  if ggml_type == rt.MXFP4: b[:, 0] = torch.randint(118, 122, (nb,), generator=gen, device="cuda", dtype=torch.uint8)
  elif ggml_type == rt.Q6_K: b[:, 208:210] = scale(s * per[ggml_type])
  else:
    b[:, 0:2] = scale(s * per[ggml_type])
    if ggml_type in (rt.Q4_1, rt.Q5_1): b[:, 2:4] = (torch.randn(nb, generator=gen, device="cuda") * s).half().view(torch.uint8).reshape(nb, 2)
    if ggml_type in (rt.Q4_K, rt.Q5_K): b[:, 2:4] = scale(s / 30)
  return b.reshape(-1)

def _config(case, max_context):
  c = dict(num_blocks=case["blocks"], dim=case["dim"], hidden_dim=case["hidden"], n_heads=case["heads"], n_kv_heads=case["kv_heads"], norm_eps=1e-5, vocab_size=case["vocab"], head_dim=case["head_dim"])
  if case["arch"] == "moe":
    c.update(rope_theta=OLMOE["rope_theta"], qk_norm=case["heads"] * case["head_dim"], num_experts=case["experts"], num_experts_per_tok=case["topk"])
  else: c.update(rope_theta=LLAMA3_8B["rope_theta"])
  return TransformerConfig(max_context=max_context, **c)

def _weights(case, config, seed):
  if case["arch"] == "moe":
    sd = synth_state_moe(config, seed=seed)
    rt.synchronize()
    for name, (b, t, _) in sd.items():                                      # expert weights about k ** -0.5 like the dense ones: two exponent steps below the synthetic writer's
      if t == rt.MXFP4: _tensor(b).view(-1, GGML_QUANT[t][1])[:, 0] -= 2
    torch.cuda.synchronize()
    return sd
  if case["weights"] == "q4_k_m": return synth_state(config, seed=seed, q4_k_m=True)
  return synth_state(config, seed=seed, linear_type=TYPES[case["weights"]])

def _prompt(gen, case, rows=1):
  return torch.randint(0, case["vocab"], (rows, case["prompt"]), generator=gen, device="cuda").tolist()


def prepare(case, seed):
  kind, gen = case["kind"], _gen(seed)
  rt.init(0)
  if kind == "linear":
    (xt, xn), (yt, yn) = FLOATS[case["x"]], FLOATS[case["y"]]
    w = _blocks(gen, TYPES[case["type"]], case["n"], case["k"])
    x = torch.randn((case["m"], case["k"]), generator=gen, device="cuda").to(xt)
    y = torch.empty((case["m"], case["n"]), device="cuda", dtype=yt)
    s = dict(layer=QuantLinear(_buffer(w, np.uint8), TYPES[case["type"]], case["n"], case["k"]), x=_buffer(x, xn), out=_buffer(y, yn), y=y)
  elif kind == "dequant":
    t = TYPES[case["type"]]
    s = dict(blocks=_buffer(_blocks(gen, t, case["n"], case["k"]), np.uint8), n=case["n"] * case["k"], type=t, dtype=FLOATS[case["y"]][1])
  elif kind == "quantize":
    def rows(): return torch.randn((case["rows"], case["k"]), generator=gen, device="cuda") * torch.exp(torch.randn((case["rows"], 1), generator=gen, device="cuda"))
    if case["op"] == "rows_f32": s = dict(op=case["op"], x=[_buffer(rows(), np.float32)])
    else: s = dict(op=case["op"], x=[_buffer(rows().bfloat16(), np.uint16) for _ in range(2 if case["op"] == "swiglu" else 1)])
  elif kind == "moe_ffn":
    T, D, I, E = case["tokens"], case["dim"], case["inter"], case["experts"]
    def weight(n, k):                                                       # quantized once, as a program loads them
      w = torch.empty((E * n, k), device="cuda", dtype=torch.bfloat16).normal_(0, k ** -0.5, generator=gen)
      q, e8, _ = moe.quantize_mxfp8(_buffer(w, np.uint16))
      rt.synchronize()
      return q.view(0, (E, n, k), np.uint8), e8.view(0, (E, n, k // 32), np.uint8)
    pop = torch.arange(1, E + 1, device="cuda").float().pow(-case["zipf"]).log()[torch.randperm(E, generator=gen, device="cuda")]
    gumbel = -torch.empty((T, E), device="cuda").exponential_(generator=gen).log()
    s = dict(inp=_buffer(torch.randn((T, D), generator=gen, device="cuda").bfloat16(), np.uint16), logits=_buffer((pop + gumbel).contiguous(), np.float32), topk=case["topk"],
             gate_up=weight(2 * I, D), b_gate_up=_buffer(torch.randn((E, 2 * I), generator=gen, device="cuda") * 0.1, np.float32),
             down=weight(D, I), b_down=_buffer(torch.randn((E, D), generator=gen, device="cuda") * 0.1, np.float32))
  elif kind == "batch":
    c = _config(case, (case["prompt"] + 65 + 63) // 64 * 64)
    s = dict(model=BatchedTransformer(c, _weights(case, c, seed), case["batch"], max_new=64), prompts=_prompt(gen, case, case["batch"]))
    s["logits"] = _tensor(s["model"].logits_buf)
  else:
    c = _config(case, (case["prompt"] + 65 + 63) // 64 * 64)
    m = Transformer(c, _weights(case, c, seed), max_new=64)
    s = dict(model=m, prompt=_prompt(gen, case)[0], logits=_tensor(m.s.logits))
    if kind == "decode": m.prefill(s["prompt"])                             # the conversation so far is in the cache
    # the keys and values of the prompt, of the last block (each depends on all the blocks before); not of the MoE architecture, where single positions whose
    # routing crosses a near-tie differ between any two orders of summation
    s["cache"] = [_tensor(m.blk[-1].cache_k), _tensor(m.blk[-1].cache_v)] if kind == "prefill" and case["arch"] == "llama" else []
  torch.cuda.synchronize()
  return dict(kind=kind, **s)


def run(state):
  kind = state["kind"]
  if kind == "linear":
    state["layer"](state["x"], out=state["out"])
    return state["y"]
  if kind == "dequant": return _tensor(ggml_data_to_tensor(state["blocks"], state["n"], state["type"], out_dtype=state["dtype"]))
  if kind == "quantize":
    op, x = state["op"], state["x"]
    out = moe.fused_silu_mul_quantize_mxfp8(*x) if op == "swiglu" else moe.transpose_quantize_mxfp8(*x) if op == "transpose" else moe.quantize_mxfp8(*x)
    return [_tensor(b) for b in out[:2]] + ([_tensor(out[2].view(0, (out[2].nbytes,), np.uint8))] if out[2] is not None else [])
  if kind == "moe_ffn":
    return _tensor(moe.moe_feed_forward(state["inp"], state["logits"], state["topk"], state["gate_up"], state["b_gate_up"], state["down"], state["b_down"]), torch.bfloat16)
  m = state["model"]
  if kind == "batch":
    m.prefill(state["prompts"])
    m.decode_step()
    return state["logits"]
  if kind == "decode":
    for _ in m.generate(state["prompt"], 1): pass
    return state["logits"]
  m.prefill(state["prompt"], reuse_cache=False)
  m.decode_step()
  return [state["logits"], *state["cache"]]


# ---- what a pass cannot do without
def _nbytes(t: str, n: int) -> int:
  if t == "f16": return 2 * n
  nel, nby = GGML_QUANT[TYPES[t]]
  return n // nel * nby

def work(case):
  kind = case["kind"]
  size = {"f16": 2, "f32": 4}
  if kind == "linear":
    n, k, m = case["n"], case["k"], case["m"]
    return dict(bytes=_nbytes(case["type"], n * k) + m * k * size[case["x"]] + m * n * size[case["y"]], flops=2 * m * n * k)
  if kind == "dequant":
    n = case["n"] * case["k"]
    return dict(bytes=_nbytes(case["type"], n) + n * size[case["y"]], flops=2 * n)
  if kind == "quantize":
    n = case["rows"] * case["k"]
    reads = {"rows": 2, "rows_f32": 4, "swiglu": 4, "transpose": 2}[case["op"]]
    return dict(bytes=n * (reads + 1) + n // 32 + n // 32, flops=2 * n)
  if kind == "moe_ffn":
    T, D, I, E, k = (case[f] for f in ("tokens", "dim", "inter", "experts", "topk"))
    p = np.arange(1, E + 1) ** -float(case["zipf"])
    hit = float(np.sum(1 - (1 - p / p.sum()) ** (T * k)))                    # experts that some token picks, about
    return dict(bytes=hit * 3 * D * I * (1 + 1 / 32) + T * D * 4 + T * E * 4, flops=2 * T * k * 3 * D * I)
  c, rows = case, case.get("batch", 1)
  qkv, attn = (c["heads"] + 2 * c["kv_heads"]) * c["head_dim"] * c["dim"], c["heads"] * c["head_dim"] * c["dim"]
  tokens = rows * (1 if kind == "decode" else c["prompt"])
  head = c["vocab"] * c["dim"]
  kv_row = c["kv_heads"] * c["head_dim"] * 2 * 2
  if c["arch"] == "moe":
    hit = c["experts"] * (1 - (1 - c["topk"] / c["experts"]) ** tokens)
    dense, ffn, used = qkv + attn + c["experts"] * c["dim"], 3 * c["dim"] * c["hidden"] * hit, 3 * c["dim"] * c["hidden"] * c["topk"]
    wbytes = c["blocks"] * (2 * dense + _nbytes("mxfp4", int(ffn) // 32 * 32)) + 2 * head
  else:
    dense, used = qkv + attn, 3 * c["dim"] * c["hidden"]
    t = "q4_k" if c["weights"] == "q4_k_m" else c["weights"]
    wbytes = c["blocks"] * _nbytes(t, dense + used) + _nbytes("q6_k", head)
  ctx = c["prompt"]
  kv = c["blocks"] * kv_row * (ctx if kind == "decode" else tokens)
  seen = ctx if kind == "decode" else tokens * (ctx + 1) / 2                  # (position, cached position) pairs
  return dict(bytes=wbytes + kv + rows * c["vocab"] * 4, flops=2 * (c["blocks"] * (dense + used) * tokens + rows * head) + c["blocks"] * 4 * c["heads"] * c["head_dim"] * seen)


def tolerance(case):
  """Relative errors (2-norm; largest value in units of the result's root mean square) about four times what the paths show against sums in 64 bits or, for whole
  models, against the same prompt taken in chunks of other sizes, which run other kernels (measured on MI355X)."""
  kind = case["kind"]
  if kind in ("dequant", "quantize"): return "exact"                      # one rounding of an exact product; block maxima and round-to-nearest codes
  if kind == "linear": return {"rel": 1.2e-3, "max": 5e-3}                # fp16-rounded weights and results: 3.0e-4, 1.2e-3
  if kind == "moe_ffn": return {"rel": 1e-2, "max": 0.2}                  # bf16 roundings between MXFP8 products: 2.4e-3, 4.4e-2
  if case["arch"] == "llama": return {"rel": 4e-3, "max": 2.5e-2}         # fp16 activations through 32 blocks: 8.8e-4, 4.5e-3
  return {"rel": 2e-2, "max": 0.3}                                        # ... and expert choices across near-ties: 1.3e-2 over the rows of a prompt, logits 2.6e-3 .. 6e-3
