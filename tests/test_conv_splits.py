"""The input-channel split of conv3x3r_*: the cheapest allowed one by the estimate that also chooses the kernel, so that a
split is never taken that the choice of the kernel rates slower than none."""

import os
import subprocess

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = r"""
#include <cstdio>
#include "hrt_ops.h"
int main() {
  int bad = 0;
  const int hw[][2] = {{8, 8}, {16, 16}, {32, 32}, {48, 40}, {64, 96}, {96, 96}, {120, 72}};
  for (int64_t n = 1; n <= 4; ++n)
    for (int64_t i = 64; i <= 1280; i += 64)
      for (int64_t o = 128; o <= 1280; o += 32)
        for (auto& x : hw) {
          const int64_t best = hrt_conv3r_splits(n, i, o, x[0], x[1]);
          bad += best < 1 || i / 16 % best != 0;
          for (int64_t s = 1; s <= 8; ++s)
            if (i / 16 % s == 0 && (s == 1 || i / 16 / s >= 4))
              bad += hrt_conv3r_us(n, i, o, x[0], x[1], s) < hrt_conv3r_us(n, i, o, x[0], x[1], best);
        }
  printf("%d\n", bad);
  return bad != 0;
}
"""


def test_split_is_the_cheapest(tmp_path):
    (tmp_path / "t.cpp").write_text(SRC)
    subprocess.run(["g++", "-std=c++17", "-I", os.path.join(REPO, "include"), str(tmp_path / "t.cpp"), "-o", str(tmp_path / "t")], check=True)
    r = subprocess.run([str(tmp_path / "t")], stdout=subprocess.PIPE, text=True)
    assert r.returncode == 0, r.stdout
