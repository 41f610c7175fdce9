"""A small decoder layer as one native call (``LlamaDecoderLayer.forward_deferred``) against the same layer taken module
by module (a hook on one module forces that): the same kernels in the same order, so outputs and gradients are equal bit
for bit.  The one exception is the input's gradient where no residual comes in: the modules' two contributions are
rounded and then added by autograd, the native call adds them in fp32 and rounds once, so they differ by up to two
roundings of the larger contribution (2^-8 relative in bfloat16, 2^-11 in float16, 2^-23 in fp32)."""

import pytest
import torch

import torchprime_amd as tpa
from tests.util import off_address, randn

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


@pytest.mark.parametrize("trained,untouched", [
  ("down_proj", "q_proj k_proj v_proj o_proj gate_proj up_proj down_proj input_layernorm post_attention_layernorm tables"),
  ("gate_proj up_proj", "q_proj k_proj v_proj o_proj gate_proj up_proj input_layernorm post_attention_layernorm tables"),
  ("post_attention_layernorm", "q_proj k_proj v_proj o_proj input_layernorm tables"),
  ("o_proj", "q_proj k_proj v_proj o_proj input_layernorm tables"), ("k_proj", "q_proj k_proj v_proj input_layernorm"),
  ("input_layernorm", "")])  # fmt: skip
@pytest.mark.parametrize("residual", [False, True])
def test_a_frozen_lower_part_is_left_alone(trained, untouched, residual):
  """The backward of a layer whose lower part is frozen, from an input without a gradient, forms no gradient there and keeps
  nothing for it: what lies below may be changed in place after the forward, as with the modules, and the gradients are
  theirs bit for bit."""
  layer = _layer(128, 2, 2, 64, "splash_attention", torch.bfloat16)
  for n, p in layer.named_parameters():
    p.requires_grad_(any(t in n for t in trained.split()))
  leaves = [p for p in layer.parameters() if p.requires_grad]
  x, res = randn((1, 20, 128), 1, torch.bfloat16).to(DEV), randn((1, 20, 128), 2, torch.bfloat16).to(DEV) if residual else None
  cs = tpa.LlamaRotaryEmbedding(64, 500000.0).to(DEV)(x, torch.arange(20, device=DEV)[None].float())
  g = [randn((1, 20, 128), 3, torch.bfloat16).to(DEV), randn((1, 20, 128), 4, torch.bfloat16).to(DEV)]
  outs = layer.forward_deferred(x, res, position_embeddings=cs)
  assert outs[0].grad_fn.name() == "TprimeLlamaLayerBackward"
  hook = layer.mlp.register_forward_hook(lambda m, a, o: None)
  want_outs = layer.forward_deferred(x, res, position_embeddings=cs)
  hook.remove()
  used = [i for i, o in enumerate(want_outs) if o.requires_grad]  # (the modules' sum has no gradient if nothing below it has)
  want = torch.autograd.grad([want_outs[i] for i in used], leaves, [g[i] for i in used])
  with torch.no_grad():
    for n, p in layer.named_parameters():
      if any(t in n for t in untouched.split()):
        p.zero_()
    for t in cs if "tables" in untouched else ():
      t.zero_()
    if "input_layernorm" in untouched:
      x.zero_()
  for a, b in zip(torch.autograd.grad(outs, leaves, g), want):
    assert torch.equal(a, b)


def test_a_head_that_is_tuned_alone_keeps_only_its_input():
  norm, lm = tpa.LlamaRMSNorm(64).to(DEV).requires_grad_(False), torch.nn.Linear(64, 136, bias=False, device=DEV)
  x, res = randn((1, 9, 64), 1).to(DEV), randn((1, 9, 64), 2).to(DEV)
  logits = tpa.ops._native.llama_head(x, res, norm.weight, 1e-6, lm.weight)
  g = randn((1, 9, 136), 3).to(DEV)
  (want,) = torch.autograd.grad(logits, lm.weight, g, retain_graph=True)
  with torch.no_grad():
    for t in (x, res, norm.weight, lm.weight):
      t.zero_()
  assert torch.equal(torch.autograd.grad(logits, lm.weight, g)[0], want)


def test_gradients_at_odd_addresses():
  """Gradients of a layer, of the logits and of embedding rows that are contiguous but off the 16-byte addresses (pieces of
  a concatenation): the gradients of the same values at an allocation's start."""
  from torchprime_amd.linear import embed

  layer = _layer(128, 2, 2, 64, "splash_attention", torch.float32)
  x = randn((1, 20, 128), 1).to(DEV).requires_grad_(True)
  cs = tpa.LlamaRotaryEmbedding(64, 500000.0).to(DEV)(x, torch.arange(20, device=DEV)[None].float())
  g = [randn((1, 20, 128), 2).to(DEV), randn((1, 20, 128), 3).to(DEV)]
  for a, b in zip(_run(layer, x, None, None, cs, [off_address(t) for t in g])[1], _run(layer, x, None, None, cs, g)[1]):
    assert torch.equal(a, b)
  cfg = tpa.Config(vocab_size=136, num_hidden_layers=1, max_position_embeddings=512, hidden_size=128, intermediate_size=64,
                   num_attention_heads=2, num_key_value_heads=2, hidden_act="silu", initializer_range=0.02, rms_norm_eps=1e-5,
                   attention_dropout=False, attention_bias=False, rope_theta=500000.0, attention_kernel="splash_attention")  # fmt: skip
  model = tpa.LlamaForCausalLM(cfg).to(DEV)
  ids = torch.randint(136, (2, 37), generator=torch.Generator().manual_seed(1)).to(DEV)
  params, gl = list(model.parameters()), randn((2, 37, 136), 4).to(DEV)
  got, want = (torch.autograd.grad(model(ids)[0], params, t) for t in (off_address(gl), gl))
  assert all(torch.equal(a, b) for a, b in zip(got, want))
  m = torch.nn.Embedding(7, 64, device=DEV)
  ge = randn((2, 37, 64), 5).to(DEV)
  got, want = (torch.autograd.grad(embed(m, ids % 7), m.weight, t)[0] for t in (off_address(ge), ge))
  assert torch.equal(got, want)
  m.weight = torch.nn.Parameter(off_address(m.weight.detach()))
  assert torch.equal(embed(m, ids % 7), m(ids % 7))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_model_ends_equal_the_modules(dtype):
  """Embedding, final norm + lm_head + .float(): logits and gradients of the model against the same model with hooks on
  its body and its layers' mlp (the modules' own calls, over the same projection kernels)."""
  cfg = tpa.Config(vocab_size=136, num_hidden_layers=2, max_position_embeddings=512, hidden_size=256, intermediate_size=64,
                   num_attention_heads=4, num_key_value_heads=2, hidden_act="silu", initializer_range=0.02, rms_norm_eps=1e-5,
                   attention_dropout=False, attention_bias=False, rope_theta=500000.0, attention_kernel="splash_attention")  # fmt: skip
  model = tpa.LlamaForCausalLM(cfg).to(DEV).to(dtype)
  ids = torch.randint(136, (2, 37), generator=torch.Generator().manual_seed(1)).to(DEV)
  params = list(model.parameters())
  logits, loss = model(ids, labels=ids)
  assert logits.grad_fn.name() == "TprimeLlamaHeadBackward" and logits.dtype == torch.float32
  got = torch.autograd.grad(loss, params)
  for m in [model.model] + [layer.mlp for layer in model.model.layers]:
    m.register_forward_hook(lambda m, a, o: None)
  want_logits, want_loss = model(ids, labels=ids)
  assert want_logits.grad_fn.name() == "ToCopyBackward0" or dtype == torch.float32
  want = torch.autograd.grad(want_loss, params)
  assert torch.equal(logits, want_logits) and torch.equal(loss, want_loss)
  for (name, _), a, b in zip(model.named_parameters(), got, want):
    if "embed" in name:  # (its gradient is the first layer's input gradient: one rounding instead of two, see above)
      assert (a.double() - b.double()).abs().max() <= 4 * ULP[dtype] * b.double().abs().max()
    else:
      assert torch.equal(a, b), name


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("n,vocab,hidden", [(1, 3, 2), (255, 7, 510), (257, 300, 514), (1000, 2, 64)])
def test_embedding_of_a_small_vocabulary(n, vocab, hidden, dtype):
  """Rows exactly; the gradient against a float64 scatter: fp32 sums of up to n rows (n 2^-24 relative to the sum of
  magnitudes) and one rounding, half a unit in the last place: 2^-8 of the value for bfloat16's 8 significant bits, 2^-11
  for float16, 2^-24 for fp32 (a first version of this bound had halved them once more)."""
  from torchprime_amd.linear import embed

  m = torch.nn.Embedding(vocab, hidden, device=DEV, dtype=dtype)
  ids = torch.randint(vocab, (1, n), generator=torch.Generator().manual_seed(n)).to(DEV)
  out = embed(m, ids)
  assert out.grad_fn.name() == "TprimeEmbeddingBackward" and torch.equal(out, torch.nn.functional.embedding(ids, m.weight))
  g = randn(out.shape, 2, dtype).to(DEV)
  (dw,) = torch.autograd.grad(out, m.weight, g)
  zero = torch.zeros((vocab, hidden), dtype=torch.float64, device=DEV)
  ref = zero.index_add(0, ids[0], g[0].double())
  mag = zero.index_add(0, ids[0], g[0].double().abs())
  assert ((dw.double() - ref).abs() <= ULP[dtype] * ref.abs() + n * 2.0**-24 * mag + 1e-30).all()


@pytest.mark.parametrize("rows", [1, 3, 63, 65, 1024, 1025])
@pytest.mark.parametrize("hidden", [8, 72, 1000, 4096])
def test_norm_backward_of_few_rows(rows, hidden):
  """Both sides of the line between the one-launch backward and the row-walking one, against float64.  Bound: bfloat16
  results of fp32 arithmetic on bfloat16 inputs; dw also carries the normalised value's rounding."""
  x, r, w = randn((rows, hidden), 1, torch.bfloat16), randn((rows, hidden), 2, torch.bfloat16), 1 + randn((hidden,), 3, torch.bfloat16, 0.1)
  dy, dh = randn((rows, hidden), 4, torch.bfloat16), randn((rows, hidden), 5, torch.bfloat16)
  xs = [t.to(DEV).requires_grad_(True) for t in (x, r, w)]
  got = torch.autograd.grad(tpa.ops.add_rmsnorm(*xs, 1e-5), xs, [dy.to(DEV), dh.to(DEV)])
  h = (x + r).double().requires_grad_(True)
  wd = w.double().requires_grad_(True)
  y = wd * (h * torch.rsqrt(h.pow(2).mean(-1, keepdim=True) + 1e-5))
  dxr, dwr = torch.autograd.grad(y, [h, wd], dy.double())
  for a, b in ((got[0], dxr + dh.double()), (got[1], dxr + dh.double()), (got[2], dwr)):
    a = a.double().cpu()
    assert ((a - b).norm() / b.norm()).item() <= 1e-2


@pytest.mark.parametrize("unpack", ["as it was", "other strides"])
def test_saved_tensor_hooks(unpack):
  """Everything the nodes keep goes through the host and comes back, once in other strides than it went in."""
  cfg = tpa.Config(vocab_size=136, num_hidden_layers=2, max_position_embeddings=512, hidden_size=128, intermediate_size=64,
                   num_attention_heads=2, num_key_value_heads=2, hidden_act="silu", initializer_range=0.02, rms_norm_eps=1e-5,
                   attention_dropout=False, attention_bias=False, rope_theta=500000.0, attention_kernel="splash_attention")  # fmt: skip
  model = tpa.LlamaForCausalLM(cfg).to(DEV).to(torch.bfloat16)
  ids = torch.randint(136, (2, 37), generator=torch.Generator().manual_seed(1)).to(DEV)
  params = list(model.parameters())
  want = torch.autograd.grad(model(ids, labels=ids)[1], params)

  def back(t):
    t = t.to(DEV)
    return t if unpack == "as it was" or t.dim() < 2 else t.transpose(0, 1).contiguous().transpose(0, 1)

  with torch.autograd.graph.saved_tensors_hooks(lambda t: t.cpu(), back):
    logits, loss = model(ids, labels=ids)
    mlp = model.model.layers[0].mlp(logits.detach()[..., :128].to(torch.bfloat16))
  assert logits.grad_fn.name() == "TprimeLlamaHeadBackward"
  got = torch.autograd.grad(loss, params)
  assert all(torch.equal(a, b) for a, b in zip(got, want))
  w = list(model.model.layers[0].mlp.parameters())
  again = model.model.layers[0].mlp(logits.detach()[..., :128].to(torch.bfloat16))
  for a, b in zip(torch.autograd.grad(mlp.float().sum(), w), torch.autograd.grad(again.float().sum(), w)):
    assert torch.equal(a, b)


def test_a_function_mode_sees_the_modules():
  """Under an active function mode the model runs module by module, so that the mode sees every projection and lookup; the
  logits are the same but for the order of fp32 sums."""
  cfg = tpa.Config(vocab_size=136, num_hidden_layers=2, max_position_embeddings=512, hidden_size=128, intermediate_size=64,
                   num_attention_heads=2, num_key_value_heads=2, hidden_act="silu", initializer_range=0.02, rms_norm_eps=1e-5,
                   attention_dropout=False, attention_bias=False, rope_theta=500000.0, attention_kernel="splash_attention")  # fmt: skip
  model = tpa.LlamaForCausalLM(cfg).to(DEV)
  ids = torch.randint(136, (1, 37), generator=torch.Generator().manual_seed(1)).to(DEV)
  names = []

  class Seen(torch.overrides.TorchFunctionMode):
    def __torch_function__(self, func, types, args=(), kwargs=None):
      names.append(getattr(func, "__name__", str(func)))
      return func(*args, **(kwargs or {}))

  want, _ = model(ids)
  with Seen():
    got, _ = model(ids)
  assert names.count("linear") == 2 * 7 + 1 and names.count("embedding") == 1
  assert ((got - want).norm() / want.norm()).item() <= 1e-5  # (the library's fp32 products: sums in another order)


def test_a_recorded_backward_gives_the_gradients_and_no_second_ones():
  """create_graph: the same gradients as without it; differentiating through them raises."""
  cfg = tpa.Config(vocab_size=136, num_hidden_layers=2, max_position_embeddings=512, hidden_size=128, intermediate_size=64,
                   num_attention_heads=2, num_key_value_heads=2, hidden_act="silu", initializer_range=0.02, rms_norm_eps=1e-5,
                   attention_dropout=False, attention_bias=False, rope_theta=500000.0, attention_kernel="splash_attention")  # fmt: skip
  model = tpa.LlamaForCausalLM(cfg).to(DEV)
  ids = torch.randint(136, (1, 37), generator=torch.Generator().manual_seed(1)).to(DEV)
  params = list(model.parameters())
  logits, loss = model(ids, labels=ids)
  assert logits.grad_fn.name() == "TprimeLlamaHeadBackward"
  want = torch.autograd.grad(loss, params)
  got = torch.autograd.grad(model(ids, labels=ids)[1], params, create_graph=True)
  for (name, _), a, b in zip(model.named_parameters(), got, want):
    # (the embedding's gradient is the library's scatter then: fp32 sums in another order)
    same = (a - b).abs().max() <= 1e-5 * b.abs().max() if "embed" in name else torch.equal(a, b)
    assert same and a.requires_grad, name
  with pytest.raises((NotImplementedError, RuntimeError), match="not implemented"):
    torch.autograd.grad(sum(g.sum() for g in got), params)
