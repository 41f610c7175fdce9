"""dK/dV with more key tiles than workgroups that run at once: the tiles come from a queue.  What a tile's sums are made of
does not depend on who computes it, so the gradients are those of a plain grid (no ``parts`` handed over) bit for bit, run
after run; rows of the outputs may be 8-byte aligned only, and nothing is written beyond them."""

import ctypes
import math

import pytest
import torch

from oracle import tprime_oracle as orc
from tests.test_gpu_split_walks import I3, _documents, _Problem
from tests.util import assert_close, heads_view
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


def _padded(B, H, S, D, pad):
  """(B, H, S, D) views of (B, S, H, D + pad) memory filled with FILL."""
  mem = torch.full((B, S, H, D + pad), FILL, dtype=torch.bfloat16, device=DEV)
  return mem, mem[..., :D].transpose(1, 2)


@pytest.mark.parametrize("pad", [0, 4])
@pytest.mark.parametrize("case", CASES)
def test_queue_is_the_grid(case, pad):
  Dqk, Dv, B, Hq, Hkv, Sq, Skv, causal, window, mask = case
  scale = 1 / math.sqrt(Dv)
  shapes = ((Hq, Sq, Dqk), (Hkv, Skv, Dqk), (Hkv, Skv, Dv), (Hq, Sq, Dv))
  host = [heads_view(B, h, s, d, i, torch.bfloat16) for i, (h, s, d) in enumerate(shapes)]
  q, k, v, do = (t.to(DEV) for t in host)
  seg = _documents(Skv, (700, 1, 90)).repeat(B, 1).to(DEV) if mask == "documents" else None
  pairs = None
  if mask == "pairs":
    keys = torch.arange(Skv)
    real = keys[None] < torch.tensor([Skv, 700, 64, 1, 900])[:B, None]
    keep = (keys[None, :] <= keys[:, None])[None] & real[:, None, :]
    add = torch.zeros((B, 1, Sq, Skv)).masked_fill_(~keep[:, None], float("-inf")).to(DEV, torch.bfloat16)
    out, lse, pairs = torch.ops.tprime.attn_fwd_pairs(q, k, v, add, scale)
  elif window >= 0:
    out, lse = torch.ops.tprime.attn_fwd_masked(q, k, v, None, None, scale, True, 0, window, -1, 0.0, None)
  else:
    out, lse = torch.ops.tprime.attn_fwd(q, k, v, seg, scale, causal)
  ws = torch.empty((_lib.load().tp_attn_bwd_workspace_bytes(B, Hq, Sq),), dtype=torch.uint8, device=DEV)
  results = []
  for queued in (True, False, True):
    (dqm, dq), (dkm, dk), (dvm, dv) = (_padded(B, h, s, d, pad) for h, s, d in shapes[:3])
    p = _Problem(B=B, Hq=Hq, Hkv=Hkv, Sq=Sq, Skv=Skv, Dqk=Dqk, Dv=Dv, causal=int(causal and mask != "pairs"), window_left=window,
                 window_right=-1, sm_scale=scale, dtype=0, mask_batches=B if pairs is not None else 0)  # fmt: skip
    tensors = dict(dout=do, q=q, k=k, v=v, out=out, lse=lse, seg=seg, pairs=pairs, dq=dq, dk=dk, dv=dv, ws=ws)
    for name, t in tensors.items():
      setattr(p, name, t.data_ptr() if t is not None else None)
    for name, t in zip(("do_s", "q_s", "k_s", "v_s", "o_s", "dq_s", "dk_s", "dv_s"), (do, q, k, v, out, dq, dk, dv)):
      setattr(p, name, I3(*t.stride()[:3]))
    n = _lib.load().tp_attn_bwd_parts_bytes(ctypes.byref(p))
    assert n == 1024, "a queue, and no split walks"
    # (whatever the memory holds: it is cleared on the way)
    parts = torch.full((n,), 255, dtype=torch.uint8, device=DEV)
    p.parts, p.parts_bytes = (parts.data_ptr(), n) if queued else (None, 0)
    _lib.call("tp_attn_bwd_run", ctypes.byref(p), torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
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
