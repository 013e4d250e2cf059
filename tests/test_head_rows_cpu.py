"""What a head of kernels_head.hip requests of its caches.  A value read behind the context's end has weight nothing and shows in no result, so the offsets are
checked where they are made (head_rows.h, built for the host) and the loads where they are compiled."""
import os
import re
import shutil
import subprocess

import pytest

from tests.conftest import ROOT

HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
CSRC = os.path.join(ROOT, "deepseek.cpp_amd", "csrc")

# every lane's requests of a context of kv_len positions: inside it, or an offset past the records that 32 bits hold; and every position in its place.
# Loads are of 8 bytes, keys at + 0, + 128, + 256 bytes.
PROGRAM = r"""
#include "head_rows.h"
#include <cstdio>
#include <vector>
typedef unsigned long long u64;
static int bad(const char* what, int H, int hd, int vd, int vn, int kv, u64 at) { printf("%s: H %d hd %d vd %d early %d kv_len %d at %llu\n", what, H, hd, vd, vn, kv, at); return 1; }
static int check(int H, int hd, int vd, int vn, int kv) {
  if (!head_rows_fit(kv, H, hd, vd)) return 0;
  const u64 krow = head_row_bytes(H, hd), vrow = head_row_bytes(H, vd);
  auto request = [&](unsigned lane_at, u64 moved, u64 row) {  // 0 in the context, 1 past it, 2 neither
    const u64 at = lane_at + moved;
    if (at >= 1ull << 32) return 2;
    return at + 8 <= row * kv ? 0 : at >= row * kv ? 1 : 2;
  };
  for (int h = 0; h < H; h += H > 1 ? H - 1 : 1) {
    for (int first = 0; first < kv; first += HEAD_KEY_STEP) {
      if (!head_step_there(first, kv)) return bad("key step", H, hd, vd, vn, kv, first);
      for (int pos = 0; pos < HEAD_KEY_STEP; ++pos)
        for (int sl = 0; sl < 16; ++sl)
          for (int j = 0; j < 3; ++j) {
            const unsigned at = head_key_at(pos, sl, H, h, hd);
            const int r = request(at, first * krow + 128 * j, krow);
            const bool used = pos + first < kv && 64 * j + sl * 4 < hd;
            if (r == 2 || (used && (r || at + first * krow + 128 * j != ((u64)(pos + first) * H + h) * hd * 2 + (64 * j + sl * 4) * 2)))
              return bad("key", H, hd, vd, vn, kv, at + first * krow + 128 * j);
          }
    }
    const int tpp = vd / 4, TG = 1024 / tpp;
    std::vector<int> steps;
    for (int j = 0; j < vn; ++j) steps.push_back(j * TG);
    for (int first = vn * TG; first < kv; first += 4 * TG)
      for (int j = 0; j < 4; ++j) steps.push_back(first + j * TG);
    for (int first : steps) {
      if (!head_step_there(first, kv)) continue;
      if ((u64)first * vrow >= vrow * kv) return bad("value step", H, hd, vd, vn, kv, first);
      for (int tid = 0; tid < 1024; ++tid) {
        const int g = tid / tpp, i4 = tid % tpp;
        const unsigned at = head_value_at(g, i4, TG, H, h, vd);
        const int r = request(at, first * vrow, vrow);
        const bool used = g < TG && g + first < kv;
        if (r == 2 || used != (r == 0) || (used && at + first * vrow != ((u64)(g + first) * H + h) * vd * 2 + i4 * 8)) return bad("value", H, hd, vd, vn, kv, at + first * vrow);
      }
    }
  }
  return 0;
}
int main() {
  const int shapes[][3] = {{16, 192, 128}, {128, 192, 128}, {3, 128, 128}, {2, 48, 128}, {1, 100, 96}, {5, 192, 256}, {7, 8, 4}, {4, 12, 20}};
  for (auto& s : shapes)
    for (int vn : {2, 4, 8})
      for (int kv : {1, 15, 63, 64, 65, 100, 127, 128, 129, 255, 256, 257, 300, 352, 353, 511, 513, 961, 1000, 1023, 1024, 4096})
        if (check(s[0], s[1], s[2], vn, kv)) return 1;
  const int most = 43690;  // 2^31 bytes of 128 heads of 192, not quite: the offsets' end
  if (!head_rows_fit(most, 128, 192, 128) || head_rows_fit(most + 1, 128, 192, 128)) return bad("fit", 128, 192, 128, 0, most, 0);
  return check(128, 192, 128, 8, most);
}
"""


def test_requests_stay_in_the_context_or_past_the_records(tmp_path):
    src, exe = tmp_path / "rows.cpp", tmp_path / "rows"
    src.write_text(PROGRAM)
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-I", CSRC, str(src), "-o", str(exe)])
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
def test_loads_of_rows_carry_their_whole_offset_in_the_lane(tmp_path):
    """the range check is of the lane's offset: a scalar one beside it must be 0"""
    out = tmp_path / "head.s"
    subprocess.check_call([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-x", "hip", "-S",
                           "--offload-device-only", os.path.join(CSRC, "kernels_head.hip"), "-o", str(out)], stderr=subprocess.DEVNULL)
    loads = re.findall(r"buffer_load_dwordx2 [^\n]*", out.read_text())  # (keys and values alone are 8 bytes)
    assert len(loads) > 100
    assert [x for x in loads if not re.search(r"\], 0 offen", x)] == []
