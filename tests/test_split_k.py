"""The K splits of the GEMM launches (qwen-3.5_amd/csrc/split_k.h), compiled for the host: for every
step count and every split count a launcher may pick (at least two steps per split), the splits are
consecutive, cover K once, end at K, and none is empty, none longer than the cost model's ceiling.
A split that began at or past K read past the operands (its kernel loads the first step before its
loop): with ceil(steps / splits) steps each, 56 steps in 16 splits left two of them."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "qwen-3.5_amd", "csrc")

PROG = r"""
#include <cstdio>
#include "split_k.h"
int main() {
  long checked = 0;
  for (int splits = 1; splits <= 16; ++splits)
    for (int steps = splits; steps <= 2048; ++steps) {
      const q35::SplitK k = q35::split_k(steps, splits);
      const int most = (steps + splits - 1) / splits;
      int at = 0;
      for (int s = 0; s < splits; ++s) {
        const int b = q35::split_begin(k, s), e = q35::split_begin(k, s + 1);
        if (b != at || e <= b || e - b > most || b >= steps) {
          std::printf("steps %d splits %d: split %d takes [%d, %d)\n", steps, splits, s, b, e);
          return 1;
        }
        at = e;
        ++checked;
      }
      if (at != steps) {
        std::printf("steps %d splits %d: end at %d\n", steps, splits, at);
        return 1;
      }
    }
  std::printf("%ld\n", checked);
  return 0;
}
"""


def test_every_split_lies_inside_k(tmp_path):
    src, exe = tmp_path / "split.cpp", tmp_path / "split"
    src.write_text(PROG)
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
    assert int(r.stdout) > 250000
