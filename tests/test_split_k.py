"""The K splits of the GEMM launches (qwen-3.5_amd/csrc/split_k.h), compiled for the host.

Steps: for every step count and every split count a launcher may pick (at least two steps per split), the splits are
consecutive, cover K once, end at K, and none is empty, none longer than the cost model's ceiling.
A split that began at or past K read past the operands (its kernel loads the first step before its
loop): with ceil(steps / splits) steps each, 56 steps in 16 splits left two of them.

Room: the partials of a prompt pass hold a gate | up launch of up to 64 rows whatever the ratio of
ffn to hidden (they were sized for the hidden width alone, and the launch was refused past 6 times it)."""
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

ROOM = r"""
#include <cstdio>
#include "split_k.h"
int main() {
  for (int cap = 64; cap <= 1024; cap += 64)
    for (int hidden = 128; hidden <= 4096; hidden += 128)
      for (int ffn = 128; ffn <= 16 * hidden; ffn += 128) {
        const size_t need = (size_t)(cap < 64 ? cap : 64) * 2 * ffn;
        if (q35::prompt_part_floats(cap, hidden, ffn) < need) {
          std::printf("cap %d hidden %d ffn %d\n", cap, hidden, ffn);
          return 1;
        }
      }
  return 0;
}
"""


def run(tmp_path, prog):
    src, exe = tmp_path / "split.cpp", tmp_path / "split"
    src.write_text(prog)
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
    return r.stdout


def test_every_split_lies_inside_k(tmp_path):
    assert int(run(tmp_path, PROG)) > 250000


def test_prompt_partials_hold_gate_up(tmp_path):
    run(tmp_path, ROOM)
