"""Additive masks that only drop pairs (causality + padding, block patterns), which the attention module turns into bits:
kind of the mask, forward and backward against the oracle's eager attention at the edges of the 64-column tiles and the
128-row blocks.  Bounds: the ones every 16-bit attention test here uses (tests/util.py)."""

import pytest
import torch

import torchprime_amd as tpa
from oracle import tprime_oracle as orc
from tests.test_gpu_masks import _eager_grads, _padding_mask
from tests.util import assert_close, heads_view

pytestmark = pytest.mark.gpu
DEV = "cuda"
LOWEST = {dt: torch.finfo(dt).min for dt in (torch.bfloat16, torch.float16, torch.float32)}


def _blocks(B, Sq, Skv, seed, fill):
  """A random 0 / fill pattern whose blocks of 48 x 80 are full, empty or mixed; key 0 is seen by every row."""
  g = torch.Generator().manual_seed(seed)
  up = lambda t: t.repeat_interleave(48, 1).repeat_interleave(80, 2)[:, :Sq, :Skv]  # noqa: E731
  kind = up(torch.randint(0, 3, (B, (Sq + 47) // 48, (Skv + 79) // 80), generator=g))
  keep = (kind == 1) | ((kind == 2) & (torch.rand((B, Sq, Skv), generator=g) < 0.5))
  keep[:, :, 0] = True
  return torch.zeros((B, 1, Sq, Skv)).masked_fill_(~keep[:, None], fill)


def _check(B, Hq, Hkv, D, Dv, mask, dtype, seed=0):
  Sq, Skv = mask.shape[-2:]
  q, k, v, do = (heads_view(B, h, s, d, seed + i, dtype)
                 for i, (h, s, d) in enumerate(((Hq, Sq, D), (Hkv, Skv, D), (Hkv, Skv, Dv), (Hq, Sq, Dv))))  # fmt: skip
  qd, kd, vd = (t.to(DEV).requires_grad_(True) for t in (q, k, v))
  m = tpa.AttentionModule(tpa.Config(attention_kernel=None, num_attention_heads=Hq, num_key_value_heads=Hkv))
  out = m(qd, kd, vd, mask.to(DEV))
  assert out.grad_fn.name() == "TprimeAttnPairsBackward"
  out.backward(do.to(DEV))
  for got, ref, name in zip((out, qd.grad, kd.grad, vd.grad), _eager_grads(q, k, v, do, mask), ("out", "dq", "dk", "dv")):
    assert_close(got, ref, name, scale_abs=name != "out")


@pytest.mark.parametrize("D,Dv", [(128, 128), (64, 64), (192, 128)])
# (The smallest is 16: in a row with a single key dS = P (dP - delta) is 0 up to the 16-bit rounding of the output in delta,
# 2^-9 |dP|, against |dP| in other rows.  Where most rows are of that kind, as with 2 keys and padding, the relative bound
# of dq, 1e-2, is not one the arithmetic can meet; with 16 keys they are under a tenth of the rows: 2^-9 * 0.3 < 1e-3.)
@pytest.mark.parametrize("S", [16, 63, 64, 65, 128, 129, 333])
def test_causal_and_padding(S, D, Dv):
  lengths = [S, max(1, S // 2), max(1, S - 1)]
  _check(3, 4, 2, D, Dv, _padding_mask(3, S, S, lengths, causal=True, dtype=torch.bfloat16, fill=LOWEST[torch.bfloat16]), torch.bfloat16, S)
  _check(3, 4, 2, D, Dv, _padding_mask(3, S, S, lengths, causal=True, dtype=torch.float16, fill=LOWEST[torch.float16]), torch.float16, S)


@pytest.mark.parametrize("Sq,Skv", [(70, 300), (300, 70), (257, 257)])
@pytest.mark.parametrize("fill", [float("-inf"), LOWEST[torch.float32]])
def test_block_patterns(Sq, Skv, fill):
  _check(2, 4, 2, 128, 128, _blocks(2, Sq, Skv, Sq, fill), torch.bfloat16)
  _check(2, 4, 4, 64, 64, _blocks(1, Sq, Skv, Skv, fill), torch.float16)  # one mask for all batches


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_kind(dtype):
  kind = lambda m: tpa.ops.mask_kind(m.to(dtype).to(DEV))  # noqa: E731
  K = tpa.ops
  S, low = 130, LOWEST[dtype]
  causal = orc.causal_additive_mask(S)
  assert kind(causal) == K.MASK_CAUSAL
  assert kind(causal.clamp(min=low)) == K.MASK_PAIRS  # the same pairs, written with the lowest value
  one = causal.clone()
  one[..., 100, 7] = float("-inf")
  assert kind(one) == K.MASK_PAIRS
  for value in (-1.0, 0.5, float("nan")):
    one[..., 100, 7] = value
    assert kind(one) == K.MASK_GENERAL
  empty = causal.clone()
  empty[..., 64, :] = float("-inf")  # a row without a pair: zeros, as in the general kernels
  assert kind(empty) == K.MASK_PAIRS
  empty[..., 64, :] = low  # ... of finite entries: uniform weights
  assert kind(empty) == K.MASK_GENERAL


def test_more_masks_than_one_launch_takes():
  """65537 sequences of 4 tokens, each with its padding: kinds over all of them, and the last one's attention."""
  B, S, low = 65537, 4, float("-inf")
  causal = torch.full((S, S), low).triu(1)
  mask = causal.expand(B, 1, S, S).to(DEV, torch.bfloat16)
  assert tpa.ops.mask_kind(mask) == tpa.ops.MASK_CAUSAL
  mask = mask.clone()
  mask[-1, :, 3, 2] = low
  assert tpa.ops.mask_kind(mask) == tpa.ops.MASK_PAIRS
  q = heads_view(B, 1, S, 64, 1, torch.bfloat16).to(DEV)
  m = tpa.AttentionModule(tpa.Config(attention_kernel=None, num_attention_heads=1, num_key_value_heads=1))
  ref = orc.eager_attention(*(q[-1:].float().cpu(),) * 3, mask[-1:].float().cpu())
  assert_close(m(q, q, q, mask)[-1:], ref, "out")
  mask[-1, :, 3, 1] = 0.5
  assert tpa.ops.mask_kind(mask) == tpa.ops.MASK_GENERAL


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("Skv", [1, 3, 4, 5, 7, 8, 9, 63, 64, 65, 67, 68, 71, 72, 73, 100, 127, 128, 129])
def test_bits_at_the_rows_ends(Skv, dtype):
  """Every bit of a random mask whose rows end inside a tile; the entries behind a row's end (0: kept) must not show."""
  B, Sq = 2, 70
  g = torch.Generator().manual_seed(Skv)
  keep = torch.rand((B, Sq, Skv), generator=g) < 0.5
  memory = torch.zeros((B, 1, Sq, Skv + 5), dtype=dtype)
  memory[..., :Skv].masked_fill_(~keep[:, None], float("-inf"))
  q, k = (torch.zeros((B, 1, n, 64), dtype=torch.bfloat16, device=DEV) for n in (Sq, Skv))
  nkt, nqt, nqb, nkb = (Skv + 63) // 64, (Sq + 63) // 64, (Sq + 127) // 128, (Skv + 127) // 128
  for mask in (memory.to(DEV)[..., :Skv], memory[..., :Skv].contiguous().to(DEV)):
    pairs = torch.ops.tprime.attn_fwd_pairs(q, k, k, mask, 0.125)[2].cpu().numpy().tobytes()
    words = torch.frombuffer(bytearray(pairs[64:]), dtype=torch.int64)
    n = B * nkt * nqb * 128
    qbits, kbits = words[:n].view(B, nkt, nqb * 128), words[n : n + B * nqt * nkb * 128].view(B, nqt, nkb * 128)
    bit = torch.arange(64)
    got = ((qbits[..., None] >> bit) & 1).bool().permute(0, 2, 1, 3).reshape(B, nqb * 128, nkt * 64)
    assert torch.equal(got[:, :Sq, :Skv], keep) and not got[:, Sq:].any() and not got[:, :, Skv:].any()
    got = ((kbits[..., None] >> bit) & 1).bool().permute(0, 1, 3, 2).reshape(B, nqt * 64, nkb * 128)
    assert torch.equal(got[:, :Sq, :Skv], keep) and not got[:, Sq:].any() and not got[:, :, Skv:].any()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("Sq,Skv", [(3, 3), (5, 5), (64, 64), (65, 65), (129, 129), (200, 200), (4200, 4200), (70, 131), (131, 70)])
def test_causality_and_padding_are_told_from_other_pairs(Sq, Skv, dtype):
  """Causal masks less whole rows and keys; one pair more above the diagonal or one less below it, anywhere, makes the difference."""
  keep = torch.ones((2, 1, Sq, Skv), dtype=torch.bool, device=DEV).tril()
  keep[0, :, :, Skv // 2 + 1 :] = False  # padding on the right ...
  keep[1, :, :, : Skv // 3] = False  # ... and on the left, whose rows have no pair
  fill = lambda keep: torch.zeros(keep.shape, dtype=dtype, device=DEV).masked_fill_(~keep, float("-inf"))  # noqa: E731
  verdict = lambda keep: tpa.ops.mask_verdict(fill(keep))  # noqa: E731
  assert verdict(keep) == tpa.ops.MASK_PAIRS_CAUSAL and tpa.ops.mask_kind(fill(keep)) == tpa.ops.MASK_PAIRS
  m = min(Sq, Skv)
  for i, j in {(0, 1), (0, Skv - 1), (62, 63), (63, 64), (64, 65), (127, 128), (m - 2, m - 1), (Sq - 1, Sq), (4100, 4101)}:
    if 0 <= i < Sq and i < j < Skv:
      one = keep.clone()
      one[1, 0, i, j] = True
      assert verdict(one) == tpa.ops.MASK_PAIRS, ("above", i, j)
  for i, j in {(m - 1, m // 2), (Sq - 1, m // 2), (Sq // 2, Skv // 3), (64, 63), (63, 62), (64, 40), (128, 64), (128, 127), (4100, 4000)}:
    if i < Sq and j < min(i, Skv) and keep[0, 0, i, j] and int(keep[0, 0, i].sum()) > 1:
      one = keep.clone()
      one[0, 0, i, j] = False
      assert verdict(one) == tpa.ops.MASK_PAIRS, ("below", i, j)


def test_documents_and_windows_are_not_padding():
  S = 300
  i, j = torch.arange(S)[:, None], torch.arange(S)[None]
  for keep in (i // 100 == j // 100, (i // 100 == j // 100) & (j <= i), (j <= i) & (j > i - 50), (j <= i) | (j < 20), torch.ones((S, S), dtype=torch.bool),
               (j < 200) & (i >= 0)):  # fmt: skip
    mask = torch.zeros((1, 1, S, S)).masked_fill_(~keep, float("-inf")).to(DEV, torch.bfloat16)
    assert tpa.ops.mask_verdict(mask) == tpa.ops.mask_kind(mask) == tpa.ops.MASK_PAIRS


@pytest.mark.parametrize("causal", [True, False])
def test_the_backward_knows_the_kind(causal):
  """What the module's check says of the mask reaches the operator that plans the backward."""
  from torch.utils._python_dispatch import TorchDispatchMode

  seen = []

  class Calls(TorchDispatchMode):
    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
      if func is torch.ops.tprime.attn_bwd_pairs.default:
        seen.append(len(args) > 9 and args[9])
      return func(*args, **(kwargs or {}))

  q = torch.randn((2, 4, 300, 64), device=DEV, dtype=torch.bfloat16, requires_grad=True)
  mask = _padding_mask(2, 300, 300, [300, 100], causal=causal, dtype=torch.bfloat16, fill=LOWEST[torch.bfloat16]).to(DEV)
  m = tpa.AttentionModule(tpa.Config(attention_kernel=None, num_attention_heads=4, num_key_value_heads=4))
  with Calls():
    m(q, q, q, mask).sum().backward()
  assert seen == [causal]
