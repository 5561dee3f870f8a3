"""The causal tile order (`csrc/tile_order.h`) is a permutation of the grid's tiles: compiled for the
host and run over every grid of up to 140 planes and 80 tiles per plane, and larger ones in steps."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = os.path.join(ROOT, "sageattention-rdna4_amd", "csrc", "tile_order.h")

_MAIN = r"""
#include "%s"
#include <cstdio>
#include <vector>
int main() {
  long grids = 0;
  for (int resident = 1; resident <= 4; ++resident)
    for (int planes = 1; planes <= 140; ++planes)
      for (int tiles = 1; tiles <= 420; tiles += tiles < 80 ? 1 : 13) {
        const int total = planes * tiles, span = total / 8 * 8;
        std::vector<char> seen(total, 0);
        for (int b = 0; b < total; ++b) {
          const sage::CausalTile t = sage::causal_tile(b, span, tiles, resident);
          if (t.bh < 0 || t.bh >= planes || t.rank < 0 || t.rank >= tiles ||
              seen[t.bh * tiles + t.rank]++) {
            std::printf("resident %%d planes %%d tiles %%d block %%d -> %%d %%d\n", resident, planes,
                        tiles, b, t.bh, t.rank);
            return 1;
          }
        }
        ++grids;
      }
  std::printf("grids %%ld\n", grids);
  return 0;
}
"""


def _run(tmp_path, header, main=_MAIN):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    src, exe = tmp_path / "order.cpp", tmp_path / "order"
    src.write_text(main % header)
    subprocess.run(["g++", "-O2", "-std=c++17", "-o", str(exe), str(src)], check=True)
    return subprocess.run([str(exe)], capture_output=True, text=True)


def test_every_tile_once(tmp_path):
    res = _run(tmp_path, SRC)
    assert res.returncode == 0, res.stdout
    assert int(res.stdout.split()[1]) > 50000


def test_a_repeated_tile_is_found(tmp_path):
    # planted in a copy: the second share of the blocks that start together keeps descending order
    # in the first half and ascends in the second
    text = open(SRC).read()
    old = "i = 2 * XCD_CUS + XCD_CUS - 1 - i;"
    assert old in text
    bad = tmp_path / "bad.h"
    bad.write_text(text.replace(old, "i = c < 16 ? i : 2 * XCD_CUS + XCD_CUS - 1 - i;"))
    assert _run(tmp_path, str(bad)).returncode == 1


_ORDER = r"""
#include "%s"
#include <cstdio>
#include <set>
#include <vector>
int main() {
  long grids = 0;
  for (int planes = 1; planes <= 140; ++planes)
    for (int tiles = 1; tiles <= 300; tiles += tiles < 40 ? 1 : 13) {
      const int total = planes * tiles;
      if (total / 8 <= 32) continue;              // a compute unit for each block
      const int P = planes / 8, R = planes %% 8, slots = 4 * 32;
      const int want = (slots + tiles - 1) / tiles;
      const int G = P * tiles <= slots || want >= P ? (P ? P : 1) : want;
      const int groups = P ? (P + G - 1) / G : 1;
      std::vector<char> seen(total, 0);
      std::vector<int> last(8, -1), falls(8, 0);
      std::vector<std::set<int>> used(8);
      for (int b = 0; b < total; ++b) {
        const sage::CausalTile t = sage::causal_tile(b, total, tiles, 1);
        const int x = b %% 8;
        if (t.bh < 0 || t.bh >= planes || t.rank < 0 || t.rank >= tiles ||
            seen[t.bh * tiles + t.rank]++) {
          std::printf("planes %%d tiles %%d block %%d: repeated\n", planes, tiles, b);
          return 1;
        }
        falls[x] += t.rank < last[x];
        last[x] = t.rank;
        used[x].insert(t.bh);
      }
      for (int x = 0; x < 8; ++x)
        if (falls[x] > groups - 1 || (int)used[x].size() > P + R) {
          std::printf("planes %%d tiles %%d xcd %%d: %%d falls, %%d planes\n", planes, tiles, x, falls[x],
                      (int)used[x].size());
          return 1;
        }
      ++grids;
    }
  std::printf("grids %%ld\n", grids);
  return 0;
}
"""


def test_longest_first_and_few_planes_per_xcd(tmp_path):
    # an XCD's tiles are in descending length, but for one fall back per group of planes, and come
    # from its own planes and the ones left over, for any number of planes
    res = _run(tmp_path, SRC, _ORDER)
    assert res.returncode == 0, res.stdout
    assert int(res.stdout.split()[1]) > 5000
