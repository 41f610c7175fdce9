"""Projections of one input through several ``nn.Linear`` modules (q, k, v; gate, up), as one call, and embedding lookups.

Small ones run as one HIP launch forward and one backward (``csrc/linear.hip``), large ones as the modules' own GEMMs;
the modules and their parameters stay what they are."""

from __future__ import annotations

import torch
from torch import nn
from torch.compiler import is_compiling
from torch.nn.modules import module as _module
from torch.overrides import has_torch_function_variadic as overridden

from .ops import _native

_GLOBAL_HOOKS = (
  _module._global_forward_hooks, _module._global_forward_pre_hooks, _module._global_backward_hooks, _module._global_backward_pre_hooks,
)  # fmt: skip


def plain(m: nn.Module, cls: type) -> bool:
  """``m`` is exactly a ``cls`` and nothing has to see its call: no hooks, no patched ``forward``."""
  d = m.__dict__
  return type(m) is cls and not (
    d["_forward_hooks"] or d["_forward_pre_hooks"] or d["_backward_hooks"] or d["_backward_pre_hooks"] or "forward" in d
  )


def global_hooks() -> bool:
  return any(_GLOBAL_HOOKS)


def weight_of(m: nn.Module):
  """The weight of a module that is nothing but ``x @ weight.T``, else None."""
  if not plain(m, nn.Linear):
    return None
  p = m.__dict__["_parameters"]
  return None if p.get("bias") is not None else p.get("weight")


def project(x: torch.Tensor, *modules: nn.Module) -> list[torch.Tensor]:
  """``[m(x) for m in modules]``."""
  if not is_compiling() and not global_hooks():
    ws = [weight_of(m) for m in modules]
    # (nor may the call be overridden: fx proxies, tensor subclasses and function modes see the modules' own calls)
    if all(w is not None for w in ws) and not overridden(x, *ws):
      return _native.linears(x, ws)
  return [m(x) for m in modules]


def embed(module: nn.Module, ids: torch.Tensor) -> torch.Tensor:
  """``module(ids)`` of an ``nn.Embedding``."""
  if not is_compiling() and plain(module, nn.Embedding) and not global_hooks():
    d = module.__dict__
    w = d["_parameters"]["weight"]
    if d["padding_idx"] is None and d["max_norm"] is None and not d["scale_grad_by_freq"] and not d["sparse"] and not overridden(ids, w):
      return _native.embedding(ids, w)
  return module(ids)
