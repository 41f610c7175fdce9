"""Workloads of the package as its users run them, for measuring speed and comparing results between versions.

A case is a plain dict; ``kind`` names the part of the package that it drives, always through public entry points:

* ``path``       the hot path of an attention layer without its projections: RMSNorm, rotary table, rotary, attention
* ``model``      one training step's forward and backward of a small ``LlamaForCausalLM``
* ``attention``  attention alone: ``AttentionModule`` (causal, or with an additive mask) or the splash-attention wrapper
                 (packed documents, sliding window)
* ``norm``       residual add + RMSNorm, or RMSNorm alone
* ``rope``       rotary embedding of q and k with tables in hand, rotate-half or interleaved
* ``swiglu``     the gate product of the MLP
* ``loss``       next-token cross entropy over a large vocabulary

``train`` cases run forward and backward and return the outputs and every gradient; the others run the forward as an
evaluation loop does, under ``torch.no_grad``.
"""

from __future__ import annotations

import math
import random

import torch

import torchprime_amd as tpa
from torchprime_amd import ops

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
ESIZE = {"bf16": 2, "f16": 2, "f32": 4}
# relative rounding error (2-norm) of results that are kept in the data type; sums are taken in fp32
REL = {"bf16": 1e-2, "f16": 2e-3, "f32": 2e-5}


# ------------------------------------------------------------------------------------------------
# the cases
# ------------------------------------------------------------------------------------------------
def _attention(name, B, Hq, Hkv, S, Dqk, Dv, mask, dtype, train, window=0):
  c = dict(kind="attention", B=B, Hq=Hq, Hkv=Hkv, S=S, Dqk=Dqk, Dv=Dv, mask=mask, window=window, dtype=dtype, train=train)
  return dict(c, name=name) if name else c


def listed():
  return [
    # The reference's CPU-runnable configuration: one attention layer of hidden 512, 8 heads of 64, fp32.  Unit tests,
    # debugging and parity runs live at this size; nine short kernels, bound by launches and latency.
    dict(name="tiny_fp32_path", kind="path", B=2, S=128, Hq=8, Hkv=8, D=64, dtype="f32", train=True),
    # A whole small model (hidden 512, 8 heads of 64, two layers, the reference's test fixture cut from Llama 3.1) in
    # bf16: what a first try-out and every CI job runs, host-bound from end to end.
    dict(name="small_model_step", kind="model", B=2, S=256, layers=2, vocab=256, splash=True, dtype="bf16", train=True),
    # The headline: one Llama-3-8B attention layer in training.
    _attention("llama3_8b_train", 4, 32, 8, 8192, 128, 128, "causal", "bf16", True),
    # The same layer fed packed documents of 64..4096 tokens, as pre-training feeds it.
    _attention("llama3_8b_packed_train", 4, 32, 8, 8192, 128, 128, "packed", "bf16", True),
    # Scoring one prompt of ordinary, odd length with the 70B model's heads: forward only.
    _attention("llama3_70b_eval_odd", 1, 64, 8, 3001, 128, 128, "causal", "bf16", False),
    # DeepSeek-V3's asymmetric heads (192 for q/k, 128 for v) in training.
    _attention("deepseek_v3_train", 1, 128, 128, 4096, 192, 128, "causal", "bf16", True),
    # Fine-tuning on one medium sequence of odd length with a local window of 1024 keys.
    _attention("window_train_odd", 1, 32, 8, 2047, 128, 128, "window", "bf16", True, 1024),
    # Fine-tuning on right-padded batches through the eager branch: causal + padding as an additive mask.
    _attention("padded_batch_train", 4, 32, 8, 1000, 128, 128, "padding", "bf16", True),
    # The residual stream of a Llama-3-8B layer: residual add + RMSNorm at 4 x 8192 tokens, the largest streaming case.
    dict(name="add_norm_8b", kind="norm", rows=32768, hidden=4096, residual=True, dtype="bf16", train=True),
    # DeepSeek-V3's rotary at that model's own size: 64 rotated dims of 128 q heads and of one shared key, interleaved.
    dict(name="rope_deepseek_v3", kind="rope", B=1, Hq=128, Hkv=1, S=4096, D=64, interleaved=True, dtype="bf16", train=True),
    # The MLP's gate product at the Llama-3-8B width for a batch of odd length.
    dict(name="swiglu_8b_odd", kind="swiglu", rows=3001, cols=14336, dtype="bf16", train=True),
    # The loss of one 4096-token sequence over Llama 3's vocabulary; the models hand it fp32 logits.
    dict(name="loss_llama3", kind="loss", B=1, S=4096, V=128256, dtype="f32", train=True),
  ]


def _log_int(rng, lo, hi):
  return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _length(rng, lo, hi):
  """A length between lo and hi, spread over its logarithm; half of them as they come, half rounded to a multiple of 64."""
  n = _log_int(rng, lo, hi)
  return n if rng.random() < 0.5 else max(lo, min(hi, (n + 32) // 64 * 64))


def draw(rng):
  kind = rng.choices(["attention", "path", "model", "norm", "rope", "swiglu", "loss"], [9, 3, 2, 2, 1, 1, 2])[0]
  train = rng.random() < 0.75
  half = "bf16" if rng.random() < 0.8 else "f16"
  if kind == "attention":
    Hq, Hkv, Dqk, Dv = rng.choice([(32, 8, 128, 128), (64, 8, 128, 128), (8, 8, 64, 64), (32, 8, 64, 64), (128, 128, 192, 128),
                                   (16, 16, 192, 128)])  # fmt: skip
    mask = rng.choice(["causal", "causal", "packed", "window", "padding"])
    S = _length(rng, 128, 2048 if mask == "padding" else 8192)
    # no more (head, query, key) pairs than the largest listed case has; padded batches stay at the sizes they have
    most = (4 * 32 * 8192 * 8192 // (4 if Dqk > 128 else 2)) // (Hq * S * S)
    B = min(rng.choice([1, 1, 2, 4, 8]), max(1, most))
    window = _log_int(rng, 64, max(65, S // 2)) if mask == "window" else 0
    return _attention(None, B, Hq, Hkv, S, Dqk, Dv, mask, half, train, window)
  if kind == "path":
    Hq, Hkv, D = rng.choice([(8, 8, 64), (32, 8, 64), (32, 8, 128), (16, 4, 128)])
    f32 = rng.random() < 0.35
    B, S = rng.choice([1, 2, 4]), _length(rng, 16, 512 if f32 else 2048)
    return dict(kind=kind, B=B, S=S, Hq=Hq, Hkv=Hkv, D=D, dtype="f32" if f32 else half, train=train)
  if kind == "model":
    return dict(kind=kind, B=rng.choice([1, 2, 4]), S=_length(rng, 8, 512), layers=rng.choice([1, 2]), vocab=rng.choice([128, 256]),
                splash=rng.random() < 0.7, dtype=rng.choice(["bf16", "f32"]), train=train)  # fmt: skip
  if kind == "norm":
    hidden = rng.choice([512, 1000, 1536, 2048, 4096, 5120, 7168, 8192])
    rows = _log_int(rng, 16, 32768 * 4096 // max(hidden, 4096))
    return dict(kind=kind, rows=rows, hidden=hidden, residual=rng.random() < 0.6, dtype=rng.choice([half, half, half, "f32"]) if rows <= 8192 else half,
                train=train)  # fmt: skip
  if kind == "rope":
    Hq, Hkv, D, inter = rng.choice([(32, 8, 128, False), (64, 8, 128, False), (8, 8, 64, False), (128, 1, 64, True)])
    S = _length(rng, 16, 8192)
    B = min(rng.choice([1, 2, 4]), max(1, 4 * 32 * 8192 // (Hq * S)))
    return dict(kind=kind, B=B, Hq=Hq, Hkv=Hkv, S=S, D=D, interleaved=inter, dtype=half, train=train)
  if kind == "swiglu":
    return dict(kind=kind, rows=_log_int(rng, 16, 16384), cols=rng.choice([1408, 8192, 14336, 14344]), dtype=half, train=train)
  V = rng.choice([256, 32000, 128256, 50257])
  return dict(kind="loss", B=rng.choice([1, 2]), S=_length(rng, 16, 2048), V=V, dtype=rng.choice(["f32", "f32", "bf16"]), train=train)


# ------------------------------------------------------------------------------------------------
# inputs
# ------------------------------------------------------------------------------------------------
class _Source:
  """Normal-distributed tensors on the GPU from one seed."""

  def __init__(self, seed, dtype):
    self.gen = torch.Generator(device="cuda").manual_seed(seed)
    self.dtype = dtype

  def normal(self, *shape, dtype=None, grad=False):
    t = torch.randn(shape, generator=self.gen, device="cuda", dtype=torch.float32).to(dtype or self.dtype)
    return t.requires_grad_(grad)

  def heads(self, B, H, S, D, grad=False):
    """(B, H, S, D) as the projections leave it: a view of (B, S, H, D) memory."""
    return self.normal(B, S, H, D).transpose(1, 2).requires_grad_(grad)

  def ids(self, high, *shape):
    return torch.randint(high, shape, generator=self.gen, device="cuda")


def _documents(rng, B, S):
  """Segment ids of B rows, each packed with documents of 64..4096 tokens (no longer than half a short row)."""
  rows = []
  for _ in range(B):
    ids, doc = [], 0
    while len(ids) < S:
      ids += [doc] * min(rng.randint(min(64, S), max(64, min(4096, S // 2))), S - len(ids))
      doc += 1
    rows.append(ids)
  return rows


def _pad_lengths(rng, B, S):
  """Real lengths of B right-padded rows: the longest row fills the batch."""
  return [S] + [rng.randint(S // 3, S) for _ in range(B - 1)]


def prepare(case, seed):
  kind, dt, train = case["kind"], DTYPES[case["dtype"]], case["train"]
  src, rng = _Source(seed, dt), random.Random(seed)
  st = {"case": case, "train": train}
  if kind == "attention":
    B, Hq, Hkv, S = case["B"], case["Hq"], case["Hkv"], case["S"]
    st["q"] = src.heads(B, Hq, S, case["Dqk"], train)
    st["k"] = src.heads(B, Hkv, S, case["Dqk"], train)
    st["v"] = src.heads(B, Hkv, S, case["Dv"], train)
    st["do"] = src.heads(B, Hq, S, case["Dv"]) if train else None
    kernel = None if case["mask"] == "padding" else "splash_attention"
    st["module"] = tpa.AttentionModule(tpa.Config(attention_kernel=kernel, num_attention_heads=Hq, num_key_value_heads=Hkv,
                                                  attention_dropout=False))  # fmt: skip
    st["attention_mask"], st["segment_ids"], st["config"] = None, None, None
    if case["mask"] == "packed":
      st["segment_ids"] = torch.tensor(_documents(rng, B, S), dtype=torch.int32, device="cuda")
      st["config"] = tpa.SplashAttentionConfig().to_json()
    elif case["mask"] == "window":
      st["config"] = tpa.SplashAttentionConfig(attentiontype_local_sliding=True, slide_window_size=case["window"]).to_json()
    elif case["mask"] == "padding":
      low = torch.finfo(dt).min
      keys = torch.arange(S, device="cuda")
      real = keys[None] < torch.tensor(_pad_lengths(rng, B, S), device="cuda")[:, None]
      seen = (keys[None, :] <= keys[:, None])[None] & real[:, None, :]
      st["attention_mask"] = torch.zeros((B, 1, S, S), dtype=dt, device="cuda").masked_fill_(~seen[:, None], low)
  elif kind == "path":
    B, S, Hq, Hkv, D = case["B"], case["S"], case["Hq"], case["Hkv"], case["D"]
    st["x"] = src.normal(B, S, Hq * D, grad=train)
    st["k"], st["v"] = src.heads(B, Hkv, S, D, train), src.heads(B, Hkv, S, D, train)
    st["do"] = src.heads(B, Hq, S, D) if train else None
    st["norm"] = _norm_module(src, Hq * D, train)
    st["rotary"] = tpa.LlamaRotaryEmbedding(D, 500000.0).to("cuda")
    st["positions"] = torch.arange(S, device="cuda")[None].float()
    st["module"] = tpa.AttentionModule(tpa.Config(attention_kernel="splash_attention", num_attention_heads=Hq,
                                                  num_key_value_heads=Hkv, attention_dropout=False))  # fmt: skip
  elif kind == "model":
    cfg = tpa.Config(vocab_size=case["vocab"], num_hidden_layers=case["layers"], max_position_embeddings=131072, hidden_size=512,
                     intermediate_size=64, num_attention_heads=8, num_key_value_heads=8, hidden_act="silu", initializer_range=0.02,
                     rms_norm_eps=1e-5, attention_dropout=False, attention_bias=False, rope_theta=500000.0,
                     attention_kernel="splash_attention" if case["splash"] else None)  # fmt: skip
    model = tpa.LlamaForCausalLM(cfg).to("cuda").to(dt)
    with torch.no_grad():
      for p in model.parameters():
        p.copy_(1 + 0.1 * src.normal(*p.shape) if p.dim() == 1 else 0.02 * src.normal(*p.shape))
    st["model"] = model.requires_grad_(train)
    st["params"] = list(model.parameters())
    st["ids"] = src.ids(case["vocab"], case["B"], case["S"])
    st["ones"] = torch.ones_like(st["ids"])
  elif kind == "norm":
    st["x"], st["dy"] = src.normal(case["rows"], case["hidden"], grad=train), src.normal(case["rows"], case["hidden"])
    st["norm"] = _norm_module(src, case["hidden"], train)
    if case["residual"]:
      st["res"], st["dh"] = src.normal(case["rows"], case["hidden"], grad=train), src.normal(case["rows"], case["hidden"])
  elif kind == "rope":
    B, S, D = case["B"], case["S"], case["D"]
    st["q"], st["k"] = src.heads(B, case["Hq"], S, D, train), src.heads(B, case["Hkv"], S, D, train)
    st["dq"], st["dk"] = src.heads(B, case["Hq"], S, D), src.heads(B, case["Hkv"], S, D)
    rotary = tpa.LlamaRotaryEmbedding(D, 10000.0 if case["interleaved"] else 500000.0).to("cuda")
    st["cos"], st["sin"] = rotary(st["q"], torch.arange(S, device="cuda")[None].float())
  elif kind == "swiglu":
    st["gate"], st["up"] = (src.normal(case["rows"], case["cols"], grad=train) for _ in range(2))
    st["do"] = src.normal(case["rows"], case["cols"])
  else:
    st["logits"] = src.normal(case["B"], case["S"], case["V"], grad=train)
    labels = src.ids(case["V"], case["B"], case["S"])
    labels[:, : case["S"] // 8] = -100  # a prompt that is not trained on
    st["labels"] = labels
  return st


def _norm_module(src, hidden, train):
  norm = tpa.LlamaRMSNorm(hidden, eps=1e-5).to("cuda").to(src.dtype)
  with torch.no_grad():
    norm.weight.copy_(1 + 0.1 * src.normal(hidden))
  return norm.requires_grad_(train)


# ------------------------------------------------------------------------------------------------
# one pass
# ------------------------------------------------------------------------------------------------
def _attend(st):
  case = st["case"]
  if case["mask"] in ("packed", "window"):
    return tpa.tpu_splash_attention_jax_call_wrapper(
      mask=None, query=st["q"], key=st["k"], value=st["v"], config=st["config"], decoder_segment_ids=st["segment_ids"],
      causal=True, sm_scale=1.0 / math.sqrt(case["Dv"]),
    )[0]  # fmt: skip
  return st["module"](st["q"], st["k"], st["v"], st["attention_mask"])


def _forward(st):
  """(outputs, the tensors that gradients are taken of, the gradients that come in)."""
  case, kind = st["case"], st["case"]["kind"]
  if kind == "attention":
    return [_attend(st)], [st["q"], st["k"], st["v"]], [st["do"]]
  if kind == "path":
    q = st["norm"](st["x"]).view(case["B"], case["S"], case["Hq"], case["D"]).transpose(1, 2)
    cos, sin = st["rotary"](q, st["positions"])
    q, k = tpa.apply_rotary_pos_emb(q, st["k"], cos, sin)
    return [st["module"](q, k, st["v"])], [st["x"], st["norm"].weight, st["k"], st["v"]], [st["do"]]
  if kind == "model":
    logits, loss = st["model"](input_ids=st["ids"], labels=st["ids"], attention_mask=st["ones"])
    return [loss, logits], st["params"], None
  if kind == "norm":
    if case["residual"]:
      return list(tpa.add_rms_norm(st["x"], st["res"], st["norm"])), [st["x"], st["res"], st["norm"].weight], [st["dy"], st["dh"]]
    return [st["norm"](st["x"])], [st["x"], st["norm"].weight], [st["dy"]]
  if kind == "rope":
    apply = tpa.apply_rotary_pos_emb_interleave if case["interleaved"] else tpa.apply_rotary_pos_emb
    return list(apply(st["q"], st["k"], st["cos"], st["sin"])), [st["q"], st["k"]], [st["dq"], st["dk"]]
  if kind == "swiglu":
    return [ops.swiglu(st["gate"], st["up"])], [st["gate"], st["up"]], [st["do"]]
  return [tpa.cross_entropy_loss(st["logits"], st["labels"], case["V"])], [st["logits"]], None


def run(st):
  if not st["train"]:
    with torch.no_grad():
      return [o.detach() for o in _forward(st)[0]]
  outs, leaves, grads = _forward(st)
  got = torch.autograd.grad(outs[:1] if grads is None else outs, leaves, grads)
  return [o.detach() for o in outs] + list(got)


# ------------------------------------------------------------------------------------------------
# what a pass cannot do without, and how exact its results are
# ------------------------------------------------------------------------------------------------
def _pairs(case):
  """(query, key) pairs that take part, over the whole batch; for packed and padded rows those of a typical batch."""
  B, S = case["B"], case["S"]
  causal = S * (S + 1) // 2
  mask = case.get("mask", "causal")
  rng = random.Random(1)
  if mask == "window":
    w = min(case["window"], S - 1)
    return B * (causal - (S - w) * (S - w - 1) // 2)
  if mask == "packed":
    total = 0
    for ids in _documents(rng, B, S):
      n = [ids.count(d) for d in set(ids)]
      total += sum(x * (x + 1) // 2 for x in n)
    return total
  if mask == "padding":
    return sum(n * (n + 1) // 2 + (S - n) * n for n in _pad_lengths(rng, B, S))
  return B * causal


def _attention_work(case, Hq, Hkv, Dqk, Dv, esize):
  """Two products forward, four more backward; q, k, v (and dO) read, the output (and three gradients) written."""
  times = 3 if case["train"] else 1
  tokens = case["B"] * case["S"]
  q, kv, o = tokens * Hq * Dqk, tokens * Hkv * (Dqk + Dv), tokens * Hq * Dv
  return {"flops": times * 2.0 * Hq * (Dqk + Dv) * _pairs(case), "bytes": float(esize * (q + kv + o) * (2 if case["train"] else 1))}


def work(case):
  kind, e, train = case["kind"], ESIZE[case["dtype"]], case["train"]
  if kind == "attention":
    w = _attention_work(case, case["Hq"], case["Hkv"], case["Dqk"], case["Dv"], e)
    if case["mask"] == "padding":
      w["bytes"] += e * case["B"] * case["S"] ** 2
    return w
  if kind == "path":
    return _attention_work(case, case["Hq"], case["Hkv"], case["D"], case["D"], e)
  if kind == "model":
    tokens, H, V = case["B"] * case["S"], 512, case["vocab"]
    weights = case["layers"] * (4 * H * H + 3 * H * 64) + V * H
    attn = _attention_work(case, 8, 8, 64, 64, e)
    return {"flops": (6.0 if train else 2.0) * tokens * weights + case["layers"] * attn["flops"],
            "bytes": float(e * (weights + V * H) * (2 if train else 1) + 4 * tokens * V)}  # fmt: skip
  if kind == "norm":
    n = case["rows"] * case["hidden"]
    # forward: x (residual) in, y (sum) out; backward: the outputs' gradients in, one gradient out for x and residual alike
    moved = (2 if case["residual"] else 1) * 2 + ((3 if case["residual"] else 2) if train else 0)
    return {"flops": 10.0 * n, "bytes": float(e * n * moved)}
  if kind == "rope":
    n = case["B"] * case["S"] * (case["Hq"] + case["Hkv"]) * case["D"]
    return {"flops": 3.0 * n * (2 if train else 1), "bytes": float(e * n * (4 if train else 2))}
  if kind == "swiglu":
    n = case["rows"] * case["cols"]
    return {"flops": 8.0 * n, "bytes": float(e * n * (6 if train else 3))}
  n = case["B"] * case["S"] * case["V"]
  return {"flops": 6.0 * n, "bytes": float(e * n * (2 if train else 1))}


def tolerance(case):
  rel = REL[case["dtype"]]
  if case["kind"] == "model":
    # gradients that came through two layers, a dozen roundings deep
    return {"rel": 3e-2 if case["dtype"] == "bf16" else 1e-4}
  if case["kind"] == "loss" and not case["train"]:
    return {"rel": 1e-5}
  return {"rel": rel}
