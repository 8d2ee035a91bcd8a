"""Dispatch orders of the sweeps' waves (csrc/sgm_order.h, compiled for the host):
an order names every wave of its launch once, longest first, and a cached one is
reused only for the launch it was made for -- the four paths and the four pairs
of eight paths have equally many directions and the same first one."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <stdio.h>
#include <stdlib.h>
#include "sgm_order.h"
using namespace sgm;
static const int DX[8] = {1, -1, 0, 0, 1, -1, 1, -1}, DY[8] = {0, 0, 1, -1, 1, 1, -1, -1};
static WaveLayout of(const int *dirs, int n, int w, int h, int nd, int per) {
  int dx[8], dy[8];
  for (int i = 0; i < n; i++) dx[i] = DX[dirs[i]], dy[i] = DY[dirs[i]];
  return wave_layout(n, dx, dy, w, h, nd, per);
}
int main() {
  const int four[4] = {0, 1, 2, 3}, pairs[4] = {0, 2, 4, 5}, eight[8] = {0, 1, 2, 3, 4, 5, 6, 7};
  const int sizes[][2] = {{1600, 1067}, {5, 5}, {160, 31}, {13, 260}, {64, 64}};
  for (auto &s : sizes)
    for (int per : {1, 2, 4})
      for (int nd : {1, 2}) {
        const int w = s[0], h = s[1];
        const WaveLayout a = of(four, 4, w, h, nd, per), b = of(pairs, 4, w, h, nd, per),
                         c = of(eight, 8, w, h, nd, per);
        if (a == b || a == c || b == c || !(a == of(four, 4, w, h, nd, per)))
          return printf("layouts of %dx%d\n", w, h), 1;
        if (a == of(four, 4, w + 1, h, nd, per) || a == of(four, 4, w, h, 3 - nd, per)) return 1;
        for (const WaveLayout &L : {a, b, c}) {
          std::vector<int> order, seen(L.total, 0);
          wave_order(L, order);
          if ((int)order.size() != L.total) return printf("order of %dx%d\n", w, h), 1;
          int before = 1 << 30;
          for (int v : order) {
            if (v < 0 || v >= L.total || seen[v]++) return printf("wave %d\n", v), 1;
            int k = 0;
            while (k + 1 < L.ndirs && v >= L.begin[k + 1]) k++;
            const int n = wave_length(L.dx[k], L.dy[k], (v - L.begin[k]) % L.split[k], per, w, h);
            if (n < 1 || n > before) return printf("length of wave %d\n", v), 1;
            before = n;
          }
        }
      }
  puts("ok");
  return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_orders_belong_to_their_launch(tmp_path):
    src, exe = tmp_path / "order.cpp", tmp_path / "order"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-fsanitize=address,undefined", "-I",
                    os.path.join(ROOT, "pose_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
