"""Projections of one input through several ``nn.Linear`` modules (q, k, v; gate, up), as one call.

Small ones run as one HIP launch forward and one backward (``csrc/linear.hip``), large ones as the modules' own GEMMs;
the modules and their parameters stay what they are."""

from __future__ import annotations

import torch
from torch import nn
from torch.compiler import is_compiling
from torch.nn.modules import module as _module

from .ops import _native

_GLOBAL_HOOKS = (
  _module._global_forward_hooks, _module._global_forward_pre_hooks, _module._global_backward_hooks, _module._global_backward_pre_hooks,
)  # fmt: skip


def _weight(m: nn.Module):
  """The weight of a module that is nothing but ``x @ weight.T``, else None: a bias, hooks, a subclass or a patched
  ``forward`` have to see the call."""
  if type(m) is not nn.Linear:
    return None
  d = m.__dict__
  p = d["_parameters"]
  if p.get("bias") is not None or d["_forward_hooks"] or d["_forward_pre_hooks"] or d["_backward_hooks"] or d["_backward_pre_hooks"]:
    return None
  return None if "forward" in d else p.get("weight")


def project(x: torch.Tensor, *modules: nn.Module) -> list[torch.Tensor]:
  """``[m(x) for m in modules]``."""
  if not is_compiling() and not any(_GLOBAL_HOOKS):
    ws = [_weight(m) for m in modules]
    if all(w is not None for w in ws):
      return _native.linears(x, ws)
  return [m(x) for m in modules]
