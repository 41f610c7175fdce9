"""dK/dV with more key tiles than workgroups that run at once: the tiles come from a queue.  What a tile's sums are made of
does not depend on who computes it, so the gradients are those of a plain grid (no ``parts`` handed over) bit for bit, run
after run; rows of the outputs may be 8-byte aligned only, and nothing is written beyond them.  That the queue was in use, and gave
out every tile once, is read back from its counters."""

import ctypes
import math

import pytest
import torch

from oracle import tprime_oracle as orc
from tests.test_gpu_graph import REPLAYS, _capture, _same
from tests.test_gpu_split_walks import I3, _documents, _Problem
from tests.util import assert_close, heads_view, randn
from torchprime_amd import _lib

pytestmark = pytest.mark.gpu
DEV = "cuda"
FILL = 7.0

CASES = [  # (Dqk, Dv, B, Hq, Hkv, Sq, Skv, causal, window, mask)
  (192, 128, 1, 131, 131, 300, 300, True, -1, None),     # 131 groups: 17 for three XCDs, 16 for the others
  (192, 128, 1, 131, 131, 50, 300, False, -1, None),     # one query tile per key tile
  (192, 128, 1, 131, 131, 50, 300, True, -1, None),      # key tiles that no query sees
  (192, 128, 1, 131, 131, 290, 290, True, 3, None),
  (128, 128, 5, 16, 8, 1100, 1100, True, -1, "documents"),
  (128, 128, 5, 16, 8, 1025, 1025, False, -1, "documents"),
  (128, 128, 5, 16, 8, 1100, 1100, True, -1, "pairs"),
  (128, 128, 3, 33, 33, 513, 513, True, -1, None),
]


def _padded(B, H, S, D, pad, dtype):
  """(B, H, S, D) views of (B, S, H, D + pad) memory filled with FILL."""
  mem = torch.full((B, S, H, D + pad), FILL, dtype=dtype, device=DEV)
  return mem, mem[..., :D].transpose(1, 2)


def _problem(tensors, Sq, Skv, scale, causal, **more):
  """``tp_attn_bwd_problem`` of (dout, q, k, v, out, dq, dk, dv) and whatever else is handed over."""
  B, Hq, Dqk, Hkv, Dv = *(tensors["q"].shape[i] for i in (0, 1, 3)), *(tensors["v"].shape[i] for i in (1, 3))
  p = _Problem(B=B, Hq=Hq, Hkv=Hkv, Sq=Sq, Skv=Skv, Dqk=Dqk, Dv=Dv, causal=int(causal), window_left=-1, window_right=-1, sm_scale=scale,
               dtype={torch.bfloat16: 0, torch.float16: 1}[tensors["q"].dtype])  # fmt: skip
  for name, t in tensors.items():
    setattr(p, name, t.data_ptr() if t is not None else None)
  for name in ("dout", "q", "k", "v", "out", "dq", "dk", "dv"):
    setattr(p, {"dout": "do", "out": "o"}.get(name, name) + "_s", I3(*tensors[name].stride()[:3]))
  for name, x in more.items():
    setattr(p, name, x)
  return p


@pytest.mark.parametrize("pad", [0, 4])
@pytest.mark.parametrize("case,dtype", [(c, torch.bfloat16) for c in CASES] + [(CASES[i], torch.float16) for i in (0, 4, 6)])
def test_queue_is_the_grid(case, dtype, pad):
  Dqk, Dv, B, Hq, Hkv, Sq, Skv, causal, window, mask = case
  scale = 1 / math.sqrt(Dv)
  shapes = ((Hq, Sq, Dqk), (Hkv, Skv, Dqk), (Hkv, Skv, Dv), (Hq, Sq, Dv))
  host = [heads_view(B, h, s, d, i, dtype) for i, (h, s, d) in enumerate(shapes)]
  q, k, v, do = (t.to(DEV) for t in host)
  seg = _documents(Skv, (700, 1, 90)).repeat(B, 1).to(DEV) if mask == "documents" else None
  pairs = None
  if mask == "pairs":
    keys = torch.arange(Skv)
    real = keys[None] < torch.tensor([Skv, 700, 64, 1, 900])[:B, None]
    keep = (keys[None, :] <= keys[:, None])[None] & real[:, None, :]
    add = torch.zeros((B, 1, Sq, Skv)).masked_fill_(~keep[:, None], float("-inf")).to(DEV, dtype)
    out, lse, pairs = torch.ops.tprime.attn_fwd_pairs(q, k, v, add, scale)
  elif window >= 0:
    out, lse = torch.ops.tprime.attn_fwd_masked(q, k, v, None, None, scale, True, 0, window, -1, 0.0, None)
  else:
    out, lse = torch.ops.tprime.attn_fwd(q, k, v, seg, scale, causal)
  ws = torch.empty((_lib.load().tp_attn_bwd_workspace_bytes(B, Hq, Sq),), dtype=torch.uint8, device=DEV)
  results = []
  for queued in (True, False, True):
    (dqm, dq), (dkm, dk), (dvm, dv) = (_padded(B, h, s, d, pad, dtype) for h, s, d in shapes[:3])
    tensors = dict(dout=do, q=q, k=k, v=v, out=out, lse=lse, seg=seg, pairs=pairs, dq=dq, dk=dk, dv=dv, ws=ws)
    p = _problem(tensors, Sq, Skv, scale, causal and mask != "pairs", window_left=window, mask_batches=B if pairs is not None else 0)
    n = _lib.load().tp_attn_bwd_parts_bytes(ctypes.byref(p))
    assert n == 1024, "a queue, and no split walks"
    # (whatever the memory holds: it is cleared on the way)
    parts = torch.full((n,), 255, dtype=torch.uint8, device=DEV)
    p.parts, p.parts_bytes = (parts.data_ptr(), n) if queued else (None, 0)
    _lib.call("tp_attn_bwd_run", ctypes.byref(p), torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    if queued:  # (whoever is done with a tile asks for the next one, once)
      tiles = [(B * Hkv - x + 7) // 8 * ((Skv + 127) // 128) for x in range(8)]
      assert parts.view(torch.int32)[::32].tolist() == tiles
    for mem, d in ((dqm, Dqk), (dkm, Dqk), (dvm, Dv)):
      assert (mem[..., d:] == FILL).all()
    results.append([t.clone() for t in (dq, dk, dv)])
  for other in results[1:]:
    for a, b in zip(results[0], other):
      assert torch.equal(a, b)
  if mask is None and window < 0 and Sq == Skv:  # the last head, by itself, against the oracle
    refs = orc.attention_grads_ref(*(t[:, -1:].float() for t in host), None, causal, scale, torch.float32)
    for name, a, b in zip(("dq", "dk", "dv"), results[0], refs[1:]):
      assert_close(a[:, -1:], b, name, scale_abs=True)


@pytest.mark.parametrize("Hq,Hkv,S,Dqk,queue", [(32, 8, 1100, 128, False), (32, 8, 5000, 128, True), (8, 2, 900, 64, False)])
def test_less_scratch_than_a_plan_asks_for(Hq, Hkv, S, Dqk, queue):
  """Walks are not split then: the queue where its counters fit (and the problem has one), else a plain grid that leaves the
  scratch alone."""
  scale = 1 / math.sqrt(Dqk)
  q, k, v, do = (heads_view(1, h, S, Dqk, i, torch.bfloat16).to(DEV) for i, h in enumerate((Hq, Hkv, Hkv, Hq)))
  out, lse = torch.ops.tprime.attn_fwd(q, k, v, None, scale, True)
  ws = torch.empty((_lib.load().tp_attn_bwd_workspace_bytes(1, Hq, S),), dtype=torch.uint8, device=DEV)
  results = []
  for take in (lambda n: 0, lambda n: n - 16, lambda n: 1024, lambda n: 1008):
    dq, dk, dv = (torch.full_like(t, FILL) for t in (q, k, v))
    p = _problem(dict(dout=do, q=q, k=k, v=v, out=out, lse=lse, dq=dq, dk=dk, dv=dv, ws=ws), S, S, scale, True)
    n = _lib.load().tp_attn_bwd_parts_bytes(ctypes.byref(p))
    assert n > 2048, "split walks"
    parts = torch.full((n,), 255, dtype=torch.uint8, device=DEV)
    p.parts_bytes = take(n)
    p.parts = parts.data_ptr() if p.parts_bytes else None
    _lib.call("tp_attn_bwd_run", ctypes.byref(p), torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    counters, rest = parts[:1024].view(torch.int32)[::32], parts[1024:]
    assert (rest == 255).all()
    assert counters.tolist() == ([Hkv // 8 * ((S + 127) // 128)] * 8 if queue and p.parts_bytes >= 1024 else [-1] * 8)
    results.append((dq, dk, dv))
  for other in results[1:]:
    for a, b in zip(results[0], other):
      assert torch.equal(a, b)


def test_a_captured_queue():
  """The counters are cleared on every replay (by the kernel before: no memset node)."""
  B, H, S = 2, 24, 1000
  q, k, v, do = (torch.empty((B, H, S, 128), dtype=torch.bfloat16, device=DEV) for _ in range(4))
  p = _Problem(B=B, Hq=H, Hkv=H, Sq=S, Skv=S, Dqk=128, Dv=128, causal=1, window_left=-1, window_right=-1, sm_scale=0.1)
  assert _lib.load().tp_attn_bwd_parts_bytes(ctypes.byref(p)) == 1024

  def step():
    out, lse = torch.ops.tprime.attn_fwd(q, k, v, None, 0.1, True)
    return (out, *torch.ops.tprime.attn_bwd(do, q, k, v, out, lse, None, 0.1, True))

  def fill(seed):
    for i, t in enumerate((q, k, v, do)):
      t.copy_(randn(t.shape, seed + i, t.dtype))

  fill(0)
  graph, got = _capture(step)
  for r in range(REPLAYS):
    fill(10 * r + 1)
    want = [t.clone() for t in step()]
    torch.cuda.synchronize()
    graph.replay()
    torch.cuda.synchronize()
    _same(got, want, "queue")
