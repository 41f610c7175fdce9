"""``torch.library`` custom ops (namespace ``tprime``) over the HIP kernels in ``libtprime_hip.so``.

The operators live in ``_tprime_ops.so`` (``csrc/torch_ops.cpp``): their registration with the dispatcher, their
autograd nodes and the Python entry points used here.  This module holds their fake (shape) functions and the Python
functions users call.  As in the reference's own custom-op precedent, ``xla::offload_name`` in
torchprime/torch_xla_models/offloading.py:14-38, every op has a fake and an autograd registration, so the ops stay
traceable by functorch/AOT autograd as torchprime's remat tooling expects
(torchprime/torch_xla_models/tests/test_remat_all.py:143-202).

Every op is GPU-only: CPU tensors raise, nothing falls back to torch math.
"""

from __future__ import annotations

import math

import torch
from torch import Tensor
from torch.compiler import is_compiling
from torch.overrides import has_torch_function_variadic as overridden

try:
  from . import _tprime_ops as _native
except ImportError as e:
  raise ImportError(
    f"torchprime_amd/_tprime_ops.so is not built or does not load ({e}). Run `python -c 'import __graft_entry__ as g; "
    "g.build()'` (or `make -C torchprime_amd/csrc`) first; there is no fallback path."
  ) from e

__all__ = [
  "rmsnorm",
  "rope_table",
  "rope_apply",
  "attention",
  "add_rmsnorm",
  "l2norm",
  "scale_rows",
  "swiglu",
  "cross_entropy",
  "cross_entropy_fwd",
]

# the operators themselves (with all their outputs), for callers below autograd and for traces
_ops = torch.ops.tprime
rmsnorm_fwd, rmsnorm_bwd = _ops.rmsnorm_fwd.default, _ops.rmsnorm_bwd.default
add_rmsnorm_fwd, add_rmsnorm_bwd = _ops.add_rmsnorm_fwd.default, _ops.add_rmsnorm_bwd.default
rope_table, rope_apply_op = _ops.rope_table.default, _ops.rope_apply.default
attn_fwd, attn_bwd = _ops.attn_fwd.default, _ops.attn_bwd.default
attn_fwd_masked, attn_bwd_masked = _ops.attn_fwd_masked.default, _ops.attn_bwd_masked.default
attn_fwd_pairs, attn_bwd_pairs = _ops.attn_fwd_pairs.default, _ops.attn_bwd_pairs.default
l2norm_fwd, l2norm_bwd = _ops.l2norm_fwd.default, _ops.l2norm_bwd.default
scale_rows = _ops.scale_rows.default
swiglu_fwd, swiglu_bwd = _ops.swiglu_fwd.default, _ops.swiglu_bwd.default
cross_entropy_fwd, cross_entropy_bwd = _ops.cross_entropy_fwd.default, _ops.cross_entropy_bwd.default


# ------------------------------------------------------------------------------------------------
# shapes, dtypes and layouts of the outputs (fake tensors)
# ------------------------------------------------------------------------------------------------
def _empty_like_heads(x: Tensor, last: int | None = None) -> Tensor:
  """New (B,H,S,D') tensor.  Head-minor inputs (the (B,S,H,D)-memory views the attention modules
  build with ``.view(B,S,H,D).transpose(1,2)``) get the same head-minor memory order so the caller's
  ``transpose(1,2).contiguous()`` afterwards is free; anything else gets plain contiguous memory."""
  B, H, S, D = x.shape
  D = D if last is None else last
  if x.stride(1) < x.stride(2):
    return torch.empty((B, S, H, D), dtype=x.dtype, device=x.device).transpose(1, 2)
  return torch.empty((B, H, S, D), dtype=x.dtype, device=x.device)


@torch.library.register_fake("tprime::rmsnorm_fwd")
def _(x, weight, eps):
  out_dtype = torch.result_type(weight, x)
  rows = x.numel() // max(x.shape[-1], 1)
  return x.new_empty(x.shape, dtype=out_dtype), x.new_empty((rows,), dtype=torch.float32)


@torch.library.register_fake("tprime::rmsnorm_bwd")
def _(dy, x, weight, rstd):
  return torch.empty_like(x, memory_format=torch.contiguous_format), torch.empty_like(weight)


@torch.library.register_fake("tprime::add_rmsnorm_fwd")
def _(x, residual, weight, eps):
  rows = x.numel() // max(x.shape[-1], 1)
  return (x.new_empty(x.shape, dtype=torch.result_type(weight, x)), torch.empty_like(x, memory_format=torch.contiguous_format),
          x.new_empty((rows,), dtype=torch.float32))


@torch.library.register_fake("tprime::add_rmsnorm_bwd")
def _(dy, dh, h, weight, rstd):
  return torch.empty_like(h, memory_format=torch.contiguous_format), torch.empty_like(weight)


@torch.library.register_fake("tprime::rope_table")
def _(inv_freq, position_ids, attention_scaling, dtype):
  Bp, S = position_ids.shape
  c = inv_freq.new_empty((Bp, S, 2 * inv_freq.shape[0]), dtype=dtype)
  return c, torch.empty_like(c)


@torch.library.register_fake("tprime::rope_apply")
def _(q, k, cos, sin, pos, interleaved, backward):
  return _empty_like_heads(q), _empty_like_heads(k)


@torch.library.register_fake("tprime::attn_fwd")
def _(q, k, v, seg, sm_scale, causal):
  B, Hq, Sq, _ = q.shape
  return _empty_like_heads(q, v.shape[-1]), q.new_empty((B, Hq, Sq), dtype=torch.float32)


@torch.library.register_fake("tprime::attn_bwd")
def _(dout, q, k, v, out, lse, seg, sm_scale, causal):
  return _empty_like_heads(q), _empty_like_heads(k), _empty_like_heads(v)


@torch.library.register_fake("tprime::attn_fwd_masked")
def _(q, k, v, seg, qpos, sm_scale, causal, causal_offset, window_left, window_right, soft_cap, bias=None):
  B, Hq, Sq, _ = q.shape
  return _empty_like_heads(q, v.shape[-1]), q.new_empty((B, Hq, Sq), dtype=torch.float32)


@torch.library.register_fake("tprime::attn_bwd_masked")
def _(dout, q, k, v, out, lse, seg, qpos, sm_scale, causal, causal_offset, window_left, window_right, soft_cap, bias=None):
  return _empty_like_heads(q), _empty_like_heads(k), _empty_like_heads(v)


@torch.library.register_fake("tprime::attn_fwd_pairs")
def _(q, k, v, mask, sm_scale, causal_padded=False):
  B, Hq, Sq, _ = q.shape
  words = _native.mask_pairs_words(mask.shape[0], Sq, k.shape[2])
  return _empty_like_heads(q, v.shape[-1]), q.new_empty((B, Hq, Sq), dtype=torch.float32), q.new_empty((words,), dtype=torch.int32)


@torch.library.register_fake("tprime::attn_bwd_pairs")
def _(dout, q, k, v, out, lse, pairs, mask_batches, sm_scale, causal_padded=False):
  return _empty_like_heads(q), _empty_like_heads(k), _empty_like_heads(v)


@torch.library.register_fake("tprime::l2norm_fwd")
def _(x, eps):
  return torch.empty_like(x, memory_format=torch.contiguous_format), x.new_empty((x.numel() // max(x.shape[-1], 1),), dtype=torch.float32)


@torch.library.register_fake("tprime::l2norm_bwd")
def _(dy, x, rstd):
  return torch.empty_like(x, memory_format=torch.contiguous_format)


@torch.library.register_fake("tprime::scale_rows")
def _(x, scale):
  return torch.empty_like(x, memory_format=torch.contiguous_format)


@torch.library.register_fake("tprime::swiglu_fwd")
def _(gate, up):
  return torch.empty_like(gate, memory_format=torch.contiguous_format)


@torch.library.register_fake("tprime::swiglu_bwd")
def _(dout, gate, up):
  return torch.empty_like(gate, memory_format=torch.contiguous_format), torch.empty_like(up, memory_format=torch.contiguous_format)


@torch.library.register_fake("tprime::cross_entropy_fwd")
def _(logits, labels, ignore_index, scored_only=False):
  B, S, _ = logits.shape
  return logits.new_empty((), dtype=torch.float32), logits.new_empty((B * S,), dtype=torch.float32), logits.new_empty((2,), dtype=torch.float32)


@torch.library.register_fake("tprime::cross_entropy_bwd")
def _(dloss, logits, labels, lse, loss_and_count, ignore_index):
  return torch.empty_like(logits, memory_format=torch.contiguous_format)


# ------------------------------------------------------------------------------------------------
# what users call
# ------------------------------------------------------------------------------------------------
# (A compiler that traces does not see into _native, nor does what overrides calls on these tensors, __torch_function__: fx
# proxies, tensor subclasses, an active function mode.  For them the operators are called by name, as torch.ops functions.)
def rmsnorm(x: Tensor, weight: Tensor, eps: float) -> Tensor:
  """``weight * (x.float() * rsqrt(mean(x.float()**2, -1) + eps)).to(x.dtype)`` in one pass."""
  return rmsnorm_fwd(x, weight, eps)[0] if is_compiling() or overridden(x, weight) else _native.rmsnorm(x, weight, eps)


def add_rmsnorm(x: Tensor, residual: Tensor, weight: Tensor, eps: float) -> tuple[Tensor, Tensor]:
  """``h = residual + x; y = rms_norm(h, weight, eps)`` in one pass; returns ``(y, h)``."""
  if is_compiling() or overridden(x, residual, weight):
    return add_rmsnorm_fwd(x, residual, weight, eps)[:2]
  return _native.add_rmsnorm(x, residual, weight, eps)


def rope_table_like(inv_freq: Tensor, position_ids: Tensor, attention_scaling: float, x: Tensor) -> tuple[Tensor, Tensor]:
  """cos/sin tables ``(Bp, S, 2*half)`` in ``x``'s dtype from ``inv_freq (half)`` and float ``position_ids (Bp, S)``."""
  if is_compiling() or overridden(inv_freq, position_ids, x):
    return rope_table(inv_freq, position_ids, attention_scaling, x.dtype)
  return _native.rope_table(inv_freq, position_ids, attention_scaling, x)


def rope_apply(q: Tensor, k: Tensor, cos: Tensor, sin: Tensor, pos: Tensor | None = None, interleaved: int = 0):
  """``(q*cos + rotate_half(q)*sin, k*cos + rotate_half(k)*sin)`` for (B,H,S,D) q and k in one launch.

  ``interleaved``: 0 rotate-half, 1 DeepSeek ([evens | odds] output), 2 adjacent pairs in place (Llama-4)."""
  if is_compiling() or overridden(q, k, cos, sin, pos):
    return rope_apply_op(q, k, cos, sin, pos, int(interleaved), False)
  return _native.rope_apply(q, k, cos, sin, pos, int(interleaved))


def attention(
  q: Tensor, k: Tensor, v: Tensor, segment_ids: Tensor | None = None, sm_scale: float | None = None, causal: bool = True,
  *, window: tuple[int | None, int | None] | None = None, soft_cap: float | None = None,
  q_positions: Tensor | None = None, causal_offset: int = 0, bias: Tensor | None = None,
) -> Tensor:  # fmt: skip
  """Causal / segment-masked GQA attention: q (B,Hq,S,Dqk), k (B,Hkv,S,Dqk), v (B,Hkv,S,Dv) -> (B,Hq,S,Dv).

  ``sm_scale=None`` means ``1/sqrt(v.shape[-1])``, the scale AttentionModule uses
  (torchprime/torch_xla_models/attention.py:54-58, 107, 143, 154).

  ``window=(left, right)``: key j only if ``pos - left <= j <= pos + right`` (None: unbounded; LocalMask,
  kernel_utils.py:266-275).  ``soft_cap``: logits become ``cap * tanh(logits / cap)`` (kernel_utils.py:292).
  ``q_positions`` (Sq) int: query row i stands for position ``q_positions[i]`` of the key order
  (LoadBalancedCausalMask.q_sequence, parallelism_utils.py:109-132); ``causal_offset``: that mask's ``offset``.
  ``bias`` (1|B, 1|Hq, Sq, Skv): added to the scaled logits before the softmax, the eager branch's additive mask
  (torchprime/torch_xla_models/attention.py:151-158); it is a constant (no gradient), -inf forbids a pair, and a
  query row whose every key is forbidden gives zeros where the reference's softmax gives NaN."""
  if soft_cap is not None and soft_cap <= 0:
    raise ValueError(f"soft_cap must be positive, got {soft_cap}")
  if sm_scale is None:
    sm_scale = 1.0 / math.sqrt(v.shape[-1])
  wl, wr = (-1, -1) if window is None else tuple(-1 if w is None else int(w) for w in window)
  if bias is None and q_positions is None and wl < 0 and wr < 0 and soft_cap is None and (causal_offset == 0 or not causal):
    if is_compiling() or overridden(q, k, v, segment_ids):
      return attn_fwd(q, k, v, segment_ids, sm_scale, causal)[0]
    return _native.attention(q, k, v, segment_ids, sm_scale, causal)
  if bias is not None:
    bias = bias.detach()
  args = (q, k, v, segment_ids, q_positions, sm_scale, causal, causal_offset, wl, wr, float(soft_cap or 0.0), bias)
  return attn_fwd_masked(*args)[0] if is_compiling() or overridden(q, k, v, segment_ids, q_positions, bias) else _native.attention_masked(*args)


# kinds of additive masks (mask_kind; the last one of mask_verdict only)
MASK_GENERAL, MASK_CAUSAL, MASK_PAIRS, MASK_PAIRS_CAUSAL = 0, 1, 2, 3


def mask_verdict(mask: Tensor) -> int:
  """``mask_kind``, or ``MASK_PAIRS_CAUSAL`` for a mask of kind ``MASK_PAIRS`` that is causality and padding: the pairs on
  and below the diagonal less rows and keys as a whole."""
  return _native.mask_verdict(mask)


def mask_kind(mask: Tensor) -> int:
  """What a (1|B, 1, Sq, Skv) additive mask is: ``MASK_CAUSAL`` (exactly 0 on and below the diagonal, -inf above),
  ``MASK_PAIRS`` (every entry 0 or one that lets its pair drop out of the softmax, and no row of finite such entries
  only: causality + padding) or ``MASK_GENERAL``.  Waits for the device."""
  return min(mask_verdict(mask), MASK_PAIRS)


def attention_pairs_fit(q: Tensor, k: Tensor, v: Tensor, mask: Tensor) -> bool:
  """The kernels behind ``attention_pairs``, forward and backward, take problems of these sizes (they keep lists of tiles
  in LDS and address a mask's bits with 32 bits); ``attention(bias=mask)`` goes further."""
  return _native.attention_pairs_fit(mask.shape[0], q.shape[2], k.shape[2], q.shape[3], v.shape[3])


def attention_pairs(q: Tensor, k: Tensor, v: Tensor, mask: Tensor, sm_scale: float, causal_padded: bool = False) -> Tensor:
  """Attention under an additive mask of kind ``MASK_PAIRS`` (1|B, 1, Sq, Skv): as ``attention(bias=mask)``, with the
  mask as one bit per pair, tiles without a pair left out and tiles with every pair unmasked.  bfloat16 and float16.
  ``causal_padded``: the mask is known to be causality and padding (``MASK_PAIRS_CAUSAL``); the backward shares out its
  work by that, the results are the same either way."""
  if is_compiling() or overridden(q, k, v, mask):
    return attn_fwd_pairs(q, k, v, mask, sm_scale, causal_padded)[0]
  return _native.attention_pairs(q, k, v, mask, sm_scale, causal_padded)


def l2norm(x: Tensor, eps: float) -> Tensor:
  """``(x.float() * rsqrt(mean(x.float()**2, -1) + eps)).type_as(x)`` over the last dim."""
  return l2norm_fwd(x, eps)[0] if is_compiling() or overridden(x) else _native.l2norm(x, eps)


def swiglu(gate: Tensor, up: Tensor) -> Tensor:
  """``silu(gate) * up`` with the eager roundings, one pass."""
  return swiglu_fwd(gate, up) if is_compiling() or overridden(gate, up) else _native.swiglu(gate, up)


def cross_entropy(logits: Tensor, labels: Tensor, ignore_index: int) -> Tensor:
  """Mean of ``logsumexp(logits[b, s]) - logits[b, s, labels[b, s+1]]`` over the labels that are not ``ignore_index``."""
  if is_compiling() or overridden(logits, labels):
    return cross_entropy_fwd(logits, labels, ignore_index, True)[0]
  return _native.cross_entropy(logits, labels, ignore_index)
