"""Grouped small projections (``linear.project``) against float64 products: edges of the 64 x 64 tiles and of the 64- / 32-
value steps of the contraction, one to three weights with a summed input gradient, gradients that are strided views or
missing.  Bound: the operands are exact, sums are float32, so an element is off by its one rounding (2^-9 relative for
bfloat16, 2^-12 for float16) and by at most K 2^-24 of the sum of magnitudes; on normal data both are far below
``2^-8`` / ``2^-11`` / ``1e-5`` of the tensor in the 2-norm."""

import pytest
import torch
from torch import nn

from tests.util import off_address, randn
from torchprime_amd.linear import project

pytestmark = pytest.mark.gpu
DEV = "cuda"
REL = {torch.bfloat16: 2.0**-8, torch.float16: 2.0**-11, torch.float32: 1e-5}


def _close(got, ref, dtype, name):
  got, ref = got.double().cpu(), ref.double()
  assert torch.isfinite(got).all(), name
  err = ((got - ref).norm() / ref.norm()).item()
  assert err <= REL[dtype], f"{name}: {err:.3e} > {REL[dtype]:.3e}"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("M,K,Ns", [(1, 64, (64,)), (16, 8, (8,)), (63, 72, (64, 8)), (65, 512, (512, 128, 128)), (130, 136, (72, 200)),
                                    (300, 512, (64, 64)), (513, 64, (512,))])  # fmt: skip
def test_forward_and_gradients(M, K, Ns, dtype):
  x = randn((M, K), 1, dtype)
  ws = [randn((n, K), 10 + i, dtype) for i, n in enumerate(Ns)]
  gs = [randn((M, n), 20 + i, dtype) for i, n in enumerate(Ns)]
  mods = [nn.Linear(K, n, bias=False, device=DEV, dtype=dtype) for n in Ns]
  with torch.no_grad():
    for m, w in zip(mods, ws):
      m.weight.copy_(w)
  xd = x.to(DEV).requires_grad_(True)
  outs = project(xd.view(1, M, K), *mods)
  assert all(o.grad_fn.name() == "TprimeLinearsBackward" and o.shape == (1, M, n) for o, n in zip(outs, Ns))
  for o, w in zip(outs, ws):
    _close(o[0], x.double() @ w.double().T, dtype, "out")
  # gradients as a caller may hand them over: contiguous, and the first as a strided view
  wide = torch.cat([gs[0], gs[0]], 1).to(DEV)
  grads = [wide[:, : Ns[0]][None]] + [g.to(DEV)[None] for g in gs[1:]]
  got = torch.autograd.grad(outs, [xd] + [m.weight for m in mods], grads, retain_graph=True)
  _close(got[0], sum(g.double() @ w.double() for g, w in zip(gs, ws)), dtype, "dx")
  for d, g in zip(got[1:], gs):
    _close(d, g.double().T @ x.double(), dtype, "dw")
  # only the last output used; only the input asked for
  (dx,) = torch.autograd.grad(outs[-1], xd, grads[-1])
  _close(dx, gs[-1].double() @ ws[-1].double(), dtype, "dx of one output")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_rows_far_apart_or_shared(dtype):
  """Rows whose span is past the launch's 32-bit offsets (the last token of each long sequence of a batch) and gradients
  whose rows are one row expanded: the results of the same values side by side, bit for bit."""
  K, N = 4096, 64
  m = nn.Linear(K, N, bias=False, device=DEV, dtype=dtype)
  far = torch.empty((2, 4096, K), dtype=dtype, device=DEV)
  far[:, -1] = randn((2, K), 1, dtype).to(DEV)
  x, near = (t.detach().requires_grad_(True) for t in (far[:, -1:], far[:, -1:].contiguous()))
  assert (2 + 64) * x.stride(0) * x.element_size() >= 2**31
  g = randn((1, 1, N), 2, dtype).to(DEV).expand(2, 1, N)
  got, want = project(x, m)[0], project(near, m)[0]
  assert got.grad_fn.name() == "TprimeLinearsBackward" and torch.equal(got, want)
  for a, b in zip(torch.autograd.grad(got, [x, m.weight], g), torch.autograd.grad(want, [near, m.weight], g.contiguous())):
    assert torch.equal(a, b)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_contiguous_at_an_odd_address(dtype):
  """Input and gradients that are contiguous pieces of larger tensors, off the 16-byte addresses: the results of the same
  values at an allocation's start, bit for bit."""
  a, b = (nn.Linear(64, n, bias=False, device=DEV, dtype=dtype) for n in (64, 8))
  leaves = [f(randn((3, 5, 64), 1, dtype).to(DEV)).detach().requires_grad_(True) for f in (off_address, torch.clone)]
  grads = [randn((3, 5, n), 2, dtype).to(DEV) for n in (64, 8)]
  got, want = (project(x, a, b) for x in leaves)
  assert all(o.grad_fn.name() == "TprimeLinearsBackward" for o in got) and all(torch.equal(s, t) for s, t in zip(got, want))
  for s, t in zip(torch.autograd.grad(got, [leaves[0], a.weight, b.weight], [off_address(g) for g in grads]),
                  torch.autograd.grad(want, [leaves[1], a.weight, b.weight], grads)):
    assert torch.equal(s, t)


def test_what_no_gradient_needs_may_change():
  """The input of frozen weights and the weight of an input without a gradient are not kept, as with the modules."""
  m = nn.Linear(64, 64, bias=False, device=DEV)
  x, g = randn((7, 64), 1).to(DEV).requires_grad_(True), randn((7, 64), 2).to(DEV)
  want = torch.autograd.grad(project(x, m)[0], [x, m.weight], g)
  m.weight.requires_grad_(False)
  h = x * 1
  y = project(h, m)[0]
  h.zero_()
  assert y.grad_fn.name() == "TprimeLinearsBackward" and torch.equal(torch.autograd.grad(y, x, g)[0], want[0])
  m.weight.requires_grad_(True)
  y = project(x.detach(), m)[0]
  with torch.no_grad():
    m.weight.zero_()
  assert torch.equal(torch.autograd.grad(y, m.weight, g)[0], want[1])


def test_a_weight_past_the_offsets_is_the_library_s():
  """2 GiB of weight and one token: little work, but more than the launch's 32-bit offsets reach."""
  m = nn.Linear(8192, 131072, bias=False, device=DEV, dtype=torch.bfloat16)
  x = randn((1, 8192), 1, torch.bfloat16).to(DEV)
  with torch.no_grad():
    assert torch.equal(project(x, m)[0], m(x))


def test_what_the_modules_have_to_see_themselves():
  """Hooks, a bias, autocast, a recorded backward: the results are the modules' own."""
  x = randn((7, 64), 1, torch.float32).to(DEV).requires_grad_(True)
  m, b = nn.Linear(64, 64, bias=False, device=DEV), nn.Linear(64, 64, device=DEV)
  seen = []
  h = m.register_forward_hook(lambda mod, args, out: seen.append(out.shape))
  project(x, m)
  assert seen == [(7, 64)]
  h.remove()
  assert torch.equal(project(x, b)[0], b(x))
  with torch.autocast("cuda", dtype=torch.bfloat16):
    assert project(x, m)[0].dtype == torch.bfloat16
  (g,) = torch.autograd.grad(project(x, m)[0].pow(2).sum(), x, create_graph=True)
  (gg,) = torch.autograd.grad(g.sum(), x)
  w = m.weight.detach().double().cpu()
  _close(gg, 2.0 * torch.ones(7, 64, dtype=torch.float64) @ w.T @ w, torch.float32, "second derivative")


def test_forward_mode_goes_to_the_modules():
  """Tangents of the input and of a weight: the library's product rule, not a product without it."""
  x, m = randn((7, 64), 1, torch.float32).to(DEV), nn.Linear(64, 64, bias=False, device=DEV)
  w, tx, tw = m.weight.detach(), randn((7, 64), 2, torch.float32).to(DEV), randn((64, 64), 3, torch.float32).to(DEV)
  with torch.autograd.forward_ad.dual_level():
    del m.weight
    m.register_parameter("weight", None)
    m._parameters["weight"] = torch.autograd.forward_ad.make_dual(w, tw)
    y = project(torch.autograd.forward_ad.make_dual(x, tx), m)[0]
    got = torch.autograd.forward_ad.unpack_dual(y).tangent
  assert got is not None
  _close(got, tx.double().cpu() @ w.double().cpu().T + x.double().cpu() @ tw.double().cpu().T, torch.float32, "tangent")
