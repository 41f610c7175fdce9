"""How the backward's key tiles are handed out (``tp_attn_bwd_make_plan``), on the host."""

import ctypes
import time

import pytest

from tests.test_gpu_split_walks import _Problem
from torchprime_amd import _lib


class _Plan(ctypes.Structure):  # tp_attn_bwd_plan
  _fields_ = [("parts_bytes", ctypes.c_size_t), ("sizes", ctypes.c_int32 * 8)]
  _fields_ += [(n, ctypes.c_int32) for n in ("queue", "cap", "sums_at")] + [("first", ctypes.c_uint16 * 65), ("tile", ctypes.c_uint8 * 64)]


def _problem(B=1, Hq=32, Hkv=8, S=1024, Dqk=128, Dv=128, causal=True, ids=False, pairs=False):
  return _Problem(B=B, Hq=Hq, Hkv=Hkv, Sq=S, Skv=S, Dqk=Dqk, Dv=Dv, causal=int(causal), window_left=-1, window_right=-1, sm_scale=0.1,
                  seg=16 if ids else None, pairs=16 if pairs else None, mask_batches=int(pairs))  # fmt: skip


def _plan(p):
  plan = _Plan()
  assert _lib.load().tp_attn_bwd_make_plan(ctypes.byref(p), ctypes.byref(plan)) == plan.parts_bytes
  return plan


@pytest.mark.parametrize("ids", [False, True])
def test_a_plan_costs_the_host_in_proportion_to_its_tiles(ids):
  """32 and 64 key tiles (4096 and 8192 rows): at most twice the host's time.  (With every candidate's pieces put in order it
  took 2.5 times as long; the bound lies between.)"""
  def cost(S):
    p, plan = _problem(S=S, ids=ids), _Plan()
    at, to, make = ctypes.byref(p), ctypes.byref(plan), _lib.load().tp_attn_bwd_make_plan
    best = 1.0
    for _ in range(60):
      start = time.perf_counter()
      for _ in range(100):
        make(at, to)
      best = min(best, time.perf_counter() - start)
    return best
  ratio = min(cost(8192) / cost(4096) for _ in range(3))
  assert ratio < 2.15, ratio


def test_a_plan_is_for_its_sizes():
  lib, p = _lib.load(), _problem()
  plan = _plan(p)
  assert plan.cap and plan.parts_bytes == lib.tp_attn_bwd_parts_bytes(ctypes.byref(p)) > 1024
  # (whatever the plan, a problem without pointers is refused; other sizes are refused before that)
  assert lib.tp_attn_bwd_run_planned(ctypes.byref(p), ctypes.byref(plan), None, None) != 0 and b"null pointer" in lib.tp_last_error()
  for other in (dict(S=1025), dict(B=2), dict(Hq=16), dict(Dqk=192)):
    o = _problem(**other)
    assert lib.tp_attn_bwd_run_planned(ctypes.byref(o), ctypes.byref(plan), None, None) != 0 and b"other sizes" in lib.tp_last_error()
  assert lib.tp_attn_bwd_make_plan(None, ctypes.byref(plan)) == 0 and plan.parts_bytes == 0
  assert lib.tp_attn_bwd_make_plan(ctypes.byref(p), None) == 0
