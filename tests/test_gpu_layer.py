"""A small decoder layer as one native call (``LlamaDecoderLayer.forward_deferred``) against the same layer taken module
by module (a hook on one module forces that): the same kernels in the same order, so outputs and gradients are equal bit
for bit.  The one exception is the input's gradient where no residual comes in: the modules' two contributions are
rounded and then added by autograd, the native call adds them in fp32 and rounds once, so they differ by up to two
roundings of the larger contribution (2^-8 relative in bfloat16, 2^-11 in float16, 2^-23 in fp32)."""

import pytest
import torch

import torchprime_amd as tpa
from tests.util import randn

pytestmark = pytest.mark.gpu
DEV = "cuda"
ULP = {torch.bfloat16: 2.0**-8, torch.float16: 2.0**-11, torch.float32: 2.0**-23}


def _layer(hidden, heads, kv_heads, inter, kernel, dtype):
  cfg = tpa.Config(hidden_size=hidden, intermediate_size=inter, num_attention_heads=heads, num_key_value_heads=kv_heads,
                   hidden_act="silu", rms_norm_eps=1e-5, attention_dropout=False, attention_bias=False, attention_kernel=kernel)  # fmt: skip
  layer = tpa.LlamaDecoderLayer(cfg, 0).to(DEV).to(dtype)
  with torch.no_grad():
    for i, p in enumerate(layer.parameters()):
      p.copy_(randn(p.shape, 50 + i, dtype, 0.05) + (1 if p.dim() == 1 else 0))
  return layer


def _run(layer, x, res, mask, cs, grads):
  outs = layer.forward_deferred(x, res, attention_mask=mask, position_embeddings=cs)
  leaves = [x] + ([res] if res is not None else []) + list(layer.parameters())
  return outs, torch.autograd.grad(outs, leaves, grads)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("B,S,heads,kv_heads,D,inter,kernel,residual", [
  (2, 33, 8, 8, 64, 64, "splash_attention", False), (1, 130, 4, 2, 128, 72, "splash_attention", True),
  (3, 8, 4, 1, 64, 136, "eager causal", True), (2, 65, 2, 2, 64, 64, "eager full", False)])  # fmt: skip
def test_one_call_equals_the_modules(B, S, heads, kv_heads, D, inter, kernel, residual, dtype):
  H = heads * D
  layer = _layer(H, heads, kv_heads, inter, kernel if kernel.startswith("splash") else None, dtype)
  mask = torch.full((S, S), float("-inf"), device=DEV).triu(1)[None, None] if kernel == "eager causal" else None
  leaf = lambda seed: randn((B, S, H), seed, dtype).to(DEV).requires_grad_(True)  # noqa: E731
  x, res = leaf(1), leaf(2) if residual else None
  cs = tpa.LlamaRotaryEmbedding(D, 500000.0).to(DEV)(x, torch.arange(S, device=DEV)[None].float())
  grads = [randn((B, S, H), 3, dtype).to(DEV), randn((B, S, H), 4, dtype).to(DEV)]
  outs, got = _run(layer, x, res, mask, cs, grads)
  assert outs[0].grad_fn.name() == "TprimeLlamaLayerBackward"
  with torch.no_grad():
    plain = layer.forward_deferred(x, res, attention_mask=mask, position_embeddings=cs)
  assert all(torch.equal(a, b) for a, b in zip(plain, outs)) and plain[0].grad_fn is None

  layer.mlp.register_forward_hook(lambda m, a, o: None)
  want_outs, want = _run(layer, x, res, mask, cs, grads)
  assert want_outs[0].grad_fn.name() != "TprimeLlamaLayerBackward"
  for a, b in zip(outs, want_outs):
    assert torch.equal(a, b)
  first = 0 if residual else 1
  for a, b in zip(got[first:], want[first:]):
    assert torch.equal(a, b)
  if not residual:
    err = (got[0].double() - want[0].double()).abs().max().item()
    assert err <= ULP[dtype] * 2 * want[0].double().abs().max().item()


def test_frozen_parameters_and_unused_outputs():
  layer = _layer(128, 2, 2, 64, "splash_attention", torch.float32)
  for n, p in layer.named_parameters():
    p.requires_grad_("o_proj" in n or "input_layernorm" in n)
  x = randn((1, 20, 128), 1).to(DEV)
  cs = tpa.LlamaRotaryEmbedding(64, 500000.0).to(DEV)(x, torch.arange(20, device=DEV)[None].float())
  leaves = [p for p in layer.parameters() if p.requires_grad]
  g = randn((1, 20, 128), 2).to(DEV)
  one = torch.autograd.grad(layer.forward_deferred(x, None, position_embeddings=cs)[0], leaves, g)
  both = torch.autograd.grad(layer.forward_deferred(x, None, position_embeddings=cs), leaves, [g, torch.zeros_like(g)])
  assert all(torch.equal(a, b) for a, b in zip(one, both))
