"""The head_dim 64 constants' rule (`csrc/consts_rule.h`) counts blocks per compute unit of the device
it launches on, whole or partitioned: compiled for the host."""
import os
import shutil
import subprocess

import pytest

SRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                   "sageattention-rdna4_amd", "csrc", "consts_rule.h")
_MAIN = r"""
#include "%s"
#include <cstdio>
int main() {
  const long cus[] = {256, 128, 64, 32, 0};
  for (long c : cus)
    for (int form = 0; form < 3; ++form)     // plain, causal, key split
      for (long blocks = 1; blocks <= 1000; ++blocks)
        if (sage::consts_from_lds(blocks, c, form == 1, form == 2)) {
          std::printf("%%ld ", blocks);
          break;
        }
  return 0;
}
"""


def test_blocks_per_compute_unit(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    src, exe = tmp_path / "rule.cpp", tmp_path / "rule"
    src.write_text(_MAIN % SRC)
    subprocess.run(["g++", "-O1", "-std=c++17", "-o", str(exe), str(src)], check=True)
    got = subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout.split()
    want = [n * c + 1 for c in (256, 128, 64, 32, 256) for n in (2, 3, 1)]
    assert [int(x) for x in got] == want


def test_the_launcher_asks_it_with_the_devices_count():
    text = open(os.path.join(os.path.dirname(SRC), "attn_fwd_pl.hip")).read()
    calls = [c for c in text.split("consts_from_lds(")[1:]]
    assert len(calls) == 2 and all("a.cus," in c.split(";")[0].split("\n")[0] for c in calls)
    assert "cus_of_current_device(&a.cus)" in open(os.path.join(os.path.dirname(SRC), "capi.hip")).read()
