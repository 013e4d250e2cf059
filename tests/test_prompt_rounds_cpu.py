"""The workgroups of a prompt's plain products whose last round goes out in halves (hyd_rounds.h, built for the host): every (chunk of 16 tokens, strip group) once,
none without tokens - an empty one has its turn on an XCD, whose units then idle while others' wait - and halves only behind whole rounds."""
import os
import subprocess

from tests.conftest import ROOT

PROGRAM = r"""
#include "hyd_rounds.h"
#include <cstdio>
#include <vector>
int main() {
  for (int cus : {256, 128, 32, 304})
    for (int groups = 1; groups <= 600; groups += groups < 70 ? 1 : 37)
      for (int m = 17; m <= 1024; ++m) {
        const int chunks = (m + 31) / 32;
        const long long pairs = (long long)groups * chunks;
        const HydRounds R = hyd_rounds(pairs, cus);
        auto bad = [&](const char* what, int b) { printf("%s: %d units, %d groups, %d tokens, workgroup %d\n", what, cus, groups, m, b); return 1; };
        if (R.full + R.left != pairs || (R.left && (R.full % cus || R.left > cus / 2))) return bad("rounds", 0);
        if (!R.left) continue;
        std::vector<int> seen((size_t)groups * ((m + 15) / 16));
        const int grid = hyd_rounds_grid(R, groups, m);
        for (int b = 0; b < grid; ++b) {
          const HydRound r = hyd_round(R, groups, b);
          if (r.base < 0 || r.base >= m || r.group < 0 || r.group >= groups || r.half != (b >= R.full)) return bad("place", b);
          for (int t = r.base; t < r.base + (r.half ? 16 : 32) && t < m; t += 16)
            if (seen[(size_t)r.group * ((m + 15) / 16) + t / 16]++) return bad("twice", b);
        }
        for (int s : seen)
          if (s != 1) return bad("never", grid);
      }
  if (hyd_rounds(1ll << 31, 256).left) return 1;
  return 0;
}
"""


def test_every_token_and_group_once_and_no_empty_workgroup(tmp_path):
    src, exe = tmp_path / "rounds.cpp", tmp_path / "rounds"
    src.write_text(PROGRAM)
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-I", os.path.join(ROOT, "deepseek.cpp_amd", "csrc"), str(src), "-o", str(exe)])
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
