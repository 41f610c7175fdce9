"""The order of the attention workgroups (``xcd_map``, ``xcd_item``, ``groups_in_turns``), compiled for the host from the header:
whatever it is, every (tile, head of a group, group) comes up exactly once, in a plain grid and from a queue."""

import ctypes
import itertools
import os
import re
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "torchprime_amd", "csrc")
HOST = """
#include <algorithm>
#include <cstdint>
#define __device__
#define __forceinline__ inline
using std::min;
constexpr int SEG_NONE = 0, SEG_IDS = 1, SEG_PAIRS = 2;
static struct { int x; } blockIdx;
%s
template <int PER_CU, int SEG> static int grid(int nt, int ni, int ng, int turns, int* seen) {
  for (unsigned n = 0; n < xcd_grid(nt, ni, ng); n++) {
    blockIdx.x = (int)n;
    int t, i, g;
    if (!xcd_map<PER_CU, SEG>(nt, ni, ng, t, i, g, turns)) continue;
    if (t < 0 || t >= nt || i < 0 || i >= ni || g < 0 || g >= ng || g %% NUM_XCD != (int)(n %% NUM_XCD)) return 1;
    seen[(g * nt + t) * ni + i]++;
  }
  return 0;
}
extern "C" int plain(int per_cu, int seg, int nt, int ni, int ng, int turns, int* seen) {
  auto of = [&](auto f, auto g, auto h) { return (seg == SEG_NONE ? f : seg == SEG_IDS ? g : h)(nt, ni, ng, turns, seen); };
  return per_cu == 1 ? of(grid<1, SEG_NONE>, grid<1, SEG_IDS>, grid<1, SEG_PAIRS>) : of(grid<2, SEG_NONE>, grid<2, SEG_IDS>, grid<2, SEG_PAIRS>);
}
extern "C" int queued(int nt, int ni, int ng, int turns, int* seen) {
  for (int x = 0; x < NUM_XCD; x++) {
    int t, i, g, slot = 0;
    for (; xcd_item(slot, x, nt, ni, ng, t, i, g, turns); slot++) {
      if (t < 0 || t >= nt || i < 0 || i >= ni || g < 0 || g >= ng) return 1;
      seen[(g * nt + t) * ni + i]++;
    }
    if (slot != (ng - x + NUM_XCD - 1) / NUM_XCD * nt * ni || xcd_item(slot + 1000, x, nt, ni, ng, t, i, g, turns)) return 2;
  }
  return 0;
}
extern "C" int turns_of(int nt, int ni, int ng, int per_cu) { return groups_in_turns(nt, ni, ng, per_cu); }
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
  header = open(os.path.join(CSRC, "attn_common.hpp")).read()
  body = re.search(r"constexpr int NUM_XCD.*?inline unsigned xcd_grid\(.*?\n}\n", header, re.S).group(0)
  d = tmp_path_factory.mktemp("order")
  (d / "order.cpp").write_text(HOST % body)
  subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-o", str(d / "order.so"), str(d / "order.cpp")], check=True)
  return ctypes.CDLL(str(d / "order.so"))


SIZES = [*itertools.product((1, 2, 3, 5, 8, 13, 31, 64, 67), (1, 2, 4, 7), (1, 3, 7, 8, 9, 16, 21, 32))]


@pytest.mark.parametrize("per_cu", [1, 2])
@pytest.mark.parametrize("seg", [0, 1, 2])
def test_a_grid_does_everything_once(lib, per_cu, seg):
  for nt, ni, ng in SIZES:
    for turns in {0, 1, 2, (ng + 7) // 8, lib.turns_of(nt, ni, ng, per_cu)}:
      if turns <= (ng + 7) // 8:
        seen = (ctypes.c_int * (nt * ni * ng))()
        assert lib.plain(per_cu, seg, nt, ni, ng, turns, seen) == 0 and set(seen) == {1}, (nt, ni, ng, turns)


def test_a_queue_does_everything_once(lib):
  for nt, ni, ng in SIZES:
    for turns in {0, 1, (ng + 7) // 8, lib.turns_of(nt, ni, ng, 1)}:
      if turns <= (ng + 7) // 8:
        seen = (ctypes.c_int * (nt * ni * ng))()
        assert lib.queued(nt, ni, ng, turns, seen) == 0 and set(seen) == {1}, (nt, ni, ng, turns)
