"""The autograd nodes behind the tprime operators: gradients of outputs that are not all used, graphs that are walked
twice or differentiated, saved-tensor hooks, and traces through the dispatcher.  Reference: the same operator with the
missing gradients passed as zeros, or run eagerly; the kernels are deterministic, so results are compared bit for bit."""

import pytest
import torch

import torchprime_amd as tpa
from tests.util import randn, ticks_during

pytestmark = pytest.mark.gpu
DEV = "cuda"
BF = torch.bfloat16


def _leaf(shape, seed, dtype=BF):
  return randn(shape, seed, dtype).to(DEV).requires_grad_(True)


@pytest.mark.parametrize("used", [0, 1])
def test_one_of_two_outputs_used(used):
  q, k = _leaf((1, 4, 9, 64), 1), _leaf((1, 2, 9, 64), 2)
  cos, sin = randn((1, 9, 64), 3, BF).to(DEV), randn((1, 9, 64), 4, BF).to(DEV)
  x, r, w = _leaf((5, 96), 5), _leaf((5, 96), 6), _leaf((96,), 7)
  for make, leaves in ((lambda: tpa.ops.rope_apply(q, k, cos, sin), [q, k]), (lambda: tpa.ops.add_rmsnorm(x, r, w, 1e-5), [x, r, w])):
    outs = make()
    g = [torch.zeros_like(o) for o in outs]
    g[used] = randn(outs[used].shape, 8, BF).to(DEV)
    want = torch.autograd.grad(outs, leaves, g)
    got = torch.autograd.grad(make()[used], leaves, g[used])
    for a, b in zip(got, want):
      assert torch.equal(a, b)


def test_second_walk_and_second_derivative():
  x, w = _leaf((5, 96), 1), _leaf((96,), 2)
  y = tpa.ops.rmsnorm(x, w, 1e-5).float().sum()
  a = torch.autograd.grad(y, [x, w], retain_graph=True)
  b = torch.autograd.grad(y, [x, w])
  assert all(torch.equal(s, t) for s, t in zip(a, b))
  with pytest.raises(RuntimeError, match="second time"):
    torch.autograd.grad(y, [x, w])
  (g,) = torch.autograd.grad(tpa.ops.rmsnorm(x, w, 1e-5).float().pow(2).sum(), x, create_graph=True)
  with pytest.raises(RuntimeError, match="not implemented"):
    g.float().sum().backward()


def test_saved_tensor_hooks_and_trace():
  from functorch.compile import aot_function, nop

  q = _leaf((1, 2, 70, 128), 1)
  x, w = _leaf((5, 96), 2), _leaf((96,), 3)

  def f(q, x, w):
    return tpa.ops.attention(q, q, q), tpa.ops.rmsnorm(x, w, 1e-5), tpa.ops.swiglu(x, x)

  def grads(outs):
    return torch.autograd.grad([o.float().sum() for o in outs], [q, x, w])

  want = f(q, x, w)
  g_want = grads(want)
  with torch.autograd.graph.saved_tensors_hooks(lambda t: t.cpu(), lambda t: t.to(DEV)):
    hooked = f(q, x, w)
  traced = aot_function(f, fw_compiler=nop, bw_compiler=nop)(q, x, w)
  for outs in (hooked, traced):
    assert all(torch.equal(a, b) for a, b in zip(outs, want))
    assert all(torch.equal(a, b) for a, b in zip(grads(outs), g_want))


def test_waits_for_the_device_let_other_threads_run():
  """The kind of a mask and the range of position ids are read back from the device, behind whatever is queued there."""
  a = randn((8192, 8192), 1, BF).to(DEV)
  b = torch.empty_like(a)
  q, pos = _leaf((1, 2, 9, 64), 1), torch.arange(9, device=DEV)[None]
  table = randn((16, 64), 2, BF).to(DEV)
  mask = torch.full((9, 9), float("-inf"), device=DEV).triu(1)[None, None]
  tpa.ops.mask_kind(mask), tpa.ops.rope_apply(q, q, table, table, pos.clone()), torch.mm(a, a, out=b)
  for call in (lambda: tpa.ops.mask_kind(mask), lambda: tpa.ops.rope_apply(q, q, table, table, pos)):
    torch.cuda.synchronize()
    for _ in range(150):  # 0.1 s and more
      torch.mm(a, a, out=b)
    n, took = ticks_during(call)
    assert took > 0.03 and n > 0, (n, took)


def test_attention_refuses_shapes_it_has_no_kernel_for():
  """The checks of the operators themselves, forward and (through the mask extensions) general, before any launch."""
  q = _leaf((1, 4, 8, 64), 1)
  for kw in ({}, {"soft_cap": 5.0}):
    for exc, args in ((ValueError, (q, q[:, :3], q[:, :3])), (ValueError, (q, q, q[:, :, :4])), (ValueError, (q[0], q[0], q[0])),
                      (NotImplementedError, (q[..., :32],) * 3), (TypeError, (q, q.float(), q.float())), (TypeError, (q.double(),) * 3)):
      with pytest.raises(exc):
        tpa.ops.attention(*args, sm_scale=0.1, **kw)
    with pytest.raises(NotImplementedError, match="not built"):
      tpa.ops.attention(*(torch.zeros((1, 2, 8, d), device=DEV) for d in (192, 192, 128)), **kw)
    with pytest.raises(AssertionError, match="Sharding along sequence dimension"):
      tpa.ops.attention(q, q, q, torch.zeros((1, 4), dtype=torch.int32, device=DEV), **kw)
