"""dK/dV with the walk of a key tile split over several workgroups (few key tiles): pieces that find nothing to do, because
segment ids or a pair mask leave most query tiles out, and key tiles that nobody sees.  Against the fp32 oracle, bounds as in
every 16-bit attention test here (tests/util.py); sums of pieces in another order are fp32 and far below them."""

import ctypes
import math

import pytest
import torch

import torchprime_amd as tpa
from oracle import tprime_oracle as orc
from tests.test_gpu_masks import _eager_grads
from tests.util import assert_close, heads_view
from torchprime_amd import _lib

pytestmark = pytest.mark.gpu
DEV = "cuda"
I3 = ctypes.c_int64 * 3


class _Problem(ctypes.Structure):  # tp_attn_bwd_problem
  _fields_ = [(n, ctypes.c_void_p) for n in ("dout", "q", "k", "v", "out", "lse", "seg", "q_positions", "bias")]
  _fields_ += [("bias_strides", I3), ("pairs", ctypes.c_void_p), ("mask_batches", ctypes.c_int)]
  _fields_ += [(n, ctypes.c_void_p) for n in ("dq", "dk", "dv", "ws", "parts")] + [("parts_bytes", ctypes.c_size_t)]
  _fields_ += [(n, ctypes.c_int) for n in ("B", "Hq", "Hkv", "Sq", "Skv", "Dqk", "Dv")]
  _fields_ += [(n, I3) for n in ("do_s", "q_s", "k_s", "v_s", "o_s", "dq_s", "dk_s", "dv_s")]
  _fields_ += [("sm_scale", ctypes.c_float)] + [(n, ctypes.c_int) for n in ("causal", "causal_offset", "window_left", "window_right")]
  _fields_ += [("soft_cap", ctypes.c_float), ("dtype", ctypes.c_int), ("pairs_causal", ctypes.c_int)]


def _assert_split(B, Hq, Hkv, S, Dqk, Dv, causal=False, pairs=False, soft_cap=0.0, ids=False, padded=False):
  p = _Problem(seg=16 if ids else None, B=B, Hq=Hq, Hkv=Hkv, Sq=S, Skv=S, Dqk=Dqk, Dv=Dv, causal=int(causal), window_left=-1, window_right=-1, sm_scale=0.1,
               soft_cap=soft_cap, pairs=16 if pairs else None, mask_batches=int(pairs), pairs_causal=int(padded))  # fmt: skip
  # (up to 1024 bytes: the counters of a queue, and no tile is split)
  assert _lib.load().tp_attn_bwd_parts_bytes(ctypes.byref(p)) > 1024


def _documents(S, lengths):
  """(1, S) ids of documents of the given lengths, over and over."""
  ids, doc = [], 0
  while len(ids) < S:
    ids += [doc] * lengths[doc % len(lengths)]
    doc += 1
  return torch.tensor([ids[:S]], dtype=torch.int32)


def _leaves(Hq, Hkv, S, Dqk, Dv, B=1):
  q, k, v, do = (heads_view(B, h, S, d, i, torch.bfloat16) for i, (h, d) in enumerate(((Hq, Dqk), (Hkv, Dqk), (Hkv, Dv), (Hq, Dv))))
  return (q, k, v, do), [t.to(DEV).requires_grad_(True) for t in (q, k, v)], do.to(DEV)


@pytest.mark.parametrize("Dqk,Dv", [(128, 128), (64, 64), (192, 128)])
@pytest.mark.parametrize("S,lengths", [(1500, (16, 70, 33)), (1536, (128,)), (1100, (700, 1, 9))])
@pytest.mark.parametrize("kw", [{"causal": True}, {"causal": False}, {"causal": True, "soft_cap": 4.0}])
def test_segment_ids(Dqk, Dv, S, lengths, kw):
  Hq, Hkv, scale = 4, 2, 1 / math.sqrt(Dv)
  _assert_split(1, Hq, Hkv, S, Dqk, Dv, ids=True, **kw)
  (q, k, v, do), leaves, dod = _leaves(Hq, Hkv, S, Dqk, Dv)
  seg = _documents(S, lengths)
  ext = {k: x for k, x in kw.items() if k != "causal"}
  out = tpa.ops.attention(*leaves, seg.to(DEV), scale, kw["causal"], **ext)
  got = torch.autograd.grad(out, leaves, dod)
  refs = orc.attention_grads_ref(q, k, v, do, seg, kw["causal"], scale, torch.float32, **ext)
  for name, a, b in zip(("out", "dq", "dk", "dv"), (out, *got), refs):
    assert_close(a, b, name, scale_abs=name != "out")


@pytest.mark.parametrize("Dqk,Dv", [(128, 128), (64, 64), (192, 128)])
@pytest.mark.parametrize("S,lengths,unseen", [(1500, (16, 70, 33), 0), (1536, (128,), 0), (1100, (700, 300, 9), 400)])
def test_pair_masks(Dqk, Dv, S, lengths, unseen):
  """Documents written as an additive mask; with ``unseen``, the last keys are dropped for every row that has others."""
  Hq, Hkv = 4, 2
  _assert_split(1, Hq, Hkv, S, Dqk, Dv, pairs=True)
  (q, k, v, do), leaves, dod = _leaves(Hq, Hkv, S, Dqk, Dv)
  seg = _documents(S, lengths)[0]
  keep = seg[:, None] == seg[None]
  if unseen:
    keep[:, S - unseen :] = False
    keep[:, 0] = True
  mask = torch.zeros((1, 1, S, S)).masked_fill_(~keep, float("-inf"))
  m = tpa.AttentionModule(tpa.Config(attention_kernel=None, num_attention_heads=Hq, num_key_value_heads=Hkv))
  out = m(*leaves, mask.to(DEV, torch.bfloat16))
  assert out.grad_fn.name() == "TprimeAttnPairsBackward"
  got = torch.autograd.grad(out, leaves, dod)
  for name, a, b in zip(("out", "dq", "dk", "dv"), (out, *got), _eager_grads(q, k, v, do, mask)):
    assert_close(a, b, name, scale_abs=name != "out")
  if unseen:
    assert not got[1][:, :, S - unseen :].any() and not got[2][:, :, S - unseen :].any()


@pytest.mark.parametrize("Dqk,Dv", [(128, 128), (64, 64)])
@pytest.mark.parametrize("what", ["causal", "padding", "ids"])
def test_more_groups_than_engines(Dqk, Dv, what):
  """Three groups of heads on some XCDs and two on the others, pieces that start by falling length; walks that padding or a
  short document ends before the plan's last piece, in some sequences only."""
  B, Hq, Hkv, S, scale = 5, 16, 4, 600, 1 / math.sqrt(Dv)
  _assert_split(B, Hq, Hkv, S, Dqk, Dv, causal=what != "padding", pairs=what == "padding", ids=what == "ids", padded=True)
  (q, k, v, do), leaves, dod = _leaves(Hq, Hkv, S, Dqk, Dv, B)
  if what == "padding":
    seen = torch.tensor([600, 1, 129, 64, 383])
    keep = (torch.arange(S) < seen[:, None])[:, None] & torch.ones(S, S, dtype=torch.bool).tril()
    mask = torch.zeros((B, 1, S, S)).masked_fill_(~keep[:, None], float("-inf"))
    m = tpa.AttentionModule(tpa.Config(attention_kernel=None, num_attention_heads=Hq, num_key_value_heads=Hkv))
    out = m(*leaves, mask.to(DEV, torch.bfloat16))
    refs = _eager_grads(q, k, v, do, mask)
  else:
    seg = torch.cat([_documents(S, n) for n in ((600,), (5, 200), (300,), (16, 70, 33), (599, 1))]) if what == "ids" else None
    out = tpa.ops.attention(*leaves, seg.to(DEV) if what == "ids" else None, scale, True)
    refs = orc.attention_grads_ref(q, k, v, do, seg, True, scale, torch.float32)
  got = torch.autograd.grad(out, leaves, dod)
  for name, a, b in zip(("out", "dq", "dk", "dv"), (out, *got), refs):
    assert_close(a, b, name, scale_abs=name != "out")
