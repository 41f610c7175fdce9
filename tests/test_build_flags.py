"""The library's Makefile with compilers that only note what they are called for: every object is built once, none when
nothing changed, and all of them again when a flag did (the switch for packed fp32 among them)."""

import os
import shutil
import subprocess

CSRC = os.path.join(os.path.dirname(__file__), "..", "torchprime_amd", "csrc")


def test_a_changed_flag_rebuilds_the_objects(tmp_path):
  csrc = tmp_path / "package" / "csrc"
  csrc.mkdir(parents=True)
  (tmp_path / "include").mkdir()
  (tmp_path / "include" / "tprime_hip.h").touch()
  shutil.copy(os.path.join(CSRC, "Makefile"), csrc)
  (csrc / "check_mfma_hazards.py").touch()
  for f in os.listdir(CSRC):
    if f.endswith((".hip", ".hpp", ".cpp")):
      (csrc / f).touch()
  cc = tmp_path / "cc"
  cc.write_text('#!/bin/sh\nwhile [ "$1" != -o ]; do shift; done\necho "$2" >> %s\ntouch "$2"\n' % (tmp_path / "log"))
  cc.chmod(0o755)

  def built(**flags):
    (tmp_path / "log").write_text("")
    args = [f"HIPCC={cc}", f"CXX={cc}"] + [f"{k}={v}" for k, v in flags.items()]
    subprocess.run(["make", "-C", str(csrc), *args], check=True, capture_output=True)
    return {o for o in (tmp_path / "log").read_text().split() if o.endswith(".o")}

  every = built()
  assert len(every) == 23 and "build/bf16_128_128/attn_bwd.o" in every and "build/torch_ops.o" in every
  assert built() == set()
  assert built(DEFS="-DX=1") == every and built(DEFS="-DX=1") == set()
  text = (csrc / "Makefile").read_text()
  (csrc / "Makefile").write_text(text.replace("EXTRA_rope := ", "EXTRA_rope := -DY "))
  assert built(DEFS="-DX=1") == every
