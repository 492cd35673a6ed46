"""Host-compiled checks (g++) of the tiled GEMM's token-tile rules (csrc/launch_rules.h):

* tile_even_rule: a group's equal tiles are whole 16-token columns of at most the limit, number
  ceil(count / limit), cover the group, and none is empty;
* tile_dense_rule: 128 where that gives every CU a tile, else the smallest multiple of 16 from 64 whose
  tiles fit the CUs; known answers for the Qwen3 projections on 256 CUs.
"""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "nki-moe-megakernel_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include "launch_rules.h"
using namespace mkd;
int main() {
  for (int c = 1; c <= 20000; ++c) {
    const int per = tile_even_rule(c, 160), tiles = (c + 159) / 160;
    if (per < 16 || per > 160 || per % 16 || (long long)per * tiles < c || (long long)per * (tiles - 1) >= c) {
      printf("even %d -> %d\n", c, per);
      return 1;
    }
  }
  const int cu_list[] = {0, 64, 256, 304}, g_list[] = {1, 6, 8, 20, 32, 80};
  for (int cus : cu_list)
    for (int g : g_list)
      for (int T = 1; T <= 4096; T += 37) {
        const int t = tile_dense_rule(g, T, cus), n = cus > 0 ? cus : 256;
        if (t < 64 || t > 128 || t % 16) return 2;
        auto tiles = [&](int x) { return (long long)((T + x - 1) / x) * g; };
        if (tiles(128) >= n ? t != 128 : tiles(t) > n) return 3;
        if (tiles(128) < n && t > 64 && tiles(t - 16) <= n) return 4;
      }
  // QKV (20 n tiles) and o_proj (8 n tiles, alone and in 4 K slices) at 2048 tokens
  if (tile_dense_rule(20, 2048, 256) != 128 || tile_dense_rule(8, 2048, 256) != 64 ||
      tile_dense_rule(32, 2048, 256) != 128 || tile_dense_rule(20, 1024, 256) != 96) return 5;
  return 0;
}
"""


@pytest.mark.skipif(not shutil.which("g++"), reason="g++ not available")
def test_tile_rules(tmp_path):
    src, exe = tmp_path / "r.cpp", tmp_path / "r"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, (r.returncode, r.stdout)
