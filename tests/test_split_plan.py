"""How the backward's key tiles are handed out (``tp_attn_bwd_make_plan``), on the host."""

import ctypes
import time

import pytest

from tests.test_gpu_split_walks import _Problem
from torchprime_amd import _lib


class _Plan(ctypes.Structure):  # tp_attn_bwd_plan
  _fields_ = [("parts_bytes", ctypes.c_size_t), ("sizes", ctypes.c_int32 * 8)]
  _fields_ += [(n, ctypes.c_int32) for n in ("queue", "cap", "sums_at")] + [("first", ctypes.c_uint16 * 65), ("tile", ctypes.c_uint8 * 64)]


def _problem(B=1, Hq=32, Hkv=8, S=1024, Dqk=128, Dv=128, causal=True, ids=False, pairs=False, padded=False):
  return _Problem(B=B, Hq=Hq, Hkv=Hkv, Sq=S, Skv=S, Dqk=Dqk, Dv=Dv, causal=int(causal), window_left=-1, window_right=-1, sm_scale=0.1,
                  seg=16 if ids else None, pairs=16 if pairs else None, mask_batches=int(pairs), pairs_causal=int(padded))  # fmt: skip


def _plan(p):
  plan = _Plan()
  assert _lib.load().tp_attn_bwd_make_plan(ctypes.byref(p), ctypes.byref(plan)) == plan.parts_bytes
  return plan


@pytest.mark.parametrize("ids", [False, True])
def test_a_plan_costs_the_host_in_proportion_to_its_tiles(ids):
  """32 and 64 key tiles (4096 and 8192 rows): about twice the host's time at most (1.5 without ids, 1.9 with).  (With every
  candidate's pieces put in order it took 2.5 times as long; the bound lies between.)"""
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


@pytest.mark.parametrize("B,Hq,Hkv,S,Dqk", [(4, 32, 8, 1000, 128), (1, 32, 8, 1024, 128), (1, 32, 8, 2047, 128), (2, 32, 8, 2048, 128), (1, 16, 16, 1472, 192),
                                            (1, 32, 8, 900, 64), (4, 8, 8, 333, 64)])  # fmt: skip
def test_pair_masks_are_planned_by_what_is_known_of_them(B, Hq, Hkv, S, Dqk):
  """Nothing known: every key tile may be seen by every query or by few, as under segment ids without causality.  Causality and
  padding: the causal plan."""
  sizes = dict(B=B, Hq=Hq, Hkv=Hkv, S=S, Dqk=Dqk, Dv=min(Dqk, 128))
  assert bytes(_plan(_problem(causal=False, pairs=True, **sizes))) == bytes(_plan(_problem(causal=False, ids=True, **sizes)))
  assert bytes(_plan(_problem(causal=False, pairs=True, padded=True, **sizes))) == bytes(_plan(_problem(causal=True, **sizes)))


@pytest.mark.parametrize("Dqk", [64, 128, 192])
def test_equal_walks_are_cut_alike(Dqk):
  """Under a pair mask of which nothing is known no key tile's workgroups walk more than the longest that one XCD's share allows:
  the tiles are cut into the same number of pieces, or none is."""
  for B in (1, 2, 4):
    for S in range(256, 2304, 128):
      plan = _plan(_problem(B=B, S=S, Dqk=Dqk, Dv=min(Dqk, 128), causal=False, pairs=True))
      if plan.cap:
        n = S // 128
        assert len({plan.first[t + 1] - plan.first[t] for t in range(n)}) == 1, (B, S)


@pytest.mark.parametrize("what", ["ids", "pairs"])
def test_all_pieces_of_tiles_that_are_planned_alike(what):
  """Without causality a tile's pieces are as many as planned however short documents or a mask leave its walk (a cap of one tile);
  under causality the walks' lengths say how many."""
  sizes = dict(Hq=32, Hkv=8, S=2047)
  plan = _plan(_problem(causal=False, **{what: True}, **sizes))
  assert plan.cap == 1 and plan.first[1] > 1
  assert _plan(_problem(causal=True, ids=True, **sizes)).cap > 1 and _plan(_problem(causal=False, pairs=True, padded=True, **sizes)).cap > 1


def test_no_counters_where_no_workgroup_loops():
  """Mask extensions other than a band run on the general instantiation, which takes one key tile per workgroup."""
  for more, queue in ((dict(), 1), (dict(window_left=500), 1), (dict(soft_cap=4.0), 0), (dict(bias=16), 0), (dict(q_positions=16), 0)):
    p = _problem(B=8, S=4096)
    for name, x in more.items():
      setattr(p, name, x)
    plan = _plan(p)
    assert (plan.queue, plan.cap, plan.parts_bytes) == (queue, 0, 1024 * queue), more


def test_the_bindings_structs():
  assert [(n, getattr(_Problem, n).offset) for n in ("pairs", "parts", "B", "sm_scale", "pairs_causal")] == [
    (n, getattr(_lib.AttnBwdProblem, n).offset) for n in ("pairs", "parts", "B", "sm_scale", "pairs_causal")]  # fmt: skip
  p, plan = _lib.AttnBwdProblem(), _lib.AttnBwdPlan()
  ctypes.memmove(ctypes.byref(p), ctypes.byref(_problem()), ctypes.sizeof(p))
  assert ctypes.sizeof(p) == ctypes.sizeof(_Problem) and _lib.load().tp_attn_bwd_make_plan(ctypes.byref(p), ctypes.byref(plan)) == plan.parts_bytes
  assert bytes(plan) == bytes(_plan(_problem())) and list(plan.sizes) == [1, 32, 8, 1024, 1024, 128, 128, 0]
