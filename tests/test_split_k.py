"""The K splits of the GEMM launches (qwen-3.5_amd/csrc/split_k.h), compiled for the host.

Steps: for every step count and every split count a launcher may pick (at least two steps per split), the splits are
consecutive, cover K once, end at K, and none is empty, none longer than the cost model's ceiling.
A split that began at or past K read past the operands (its kernel loads the first step before its
loop): with ceil(steps / splits) steps each, 56 steps in 16 splits left two of them.

Room: the partials of a prompt pass hold a gate | up launch of up to 64 rows whatever the ratio of
ffn to hidden (they were sized for the hidden width alone, and the launch was refused past 6 times it).

Same splits: a call takes the splits that unlimited room would give it with the room that is asked for
its rows or for any larger call, so its bits do not depend on what a shared workspace grew to."""
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
        if (q35::prompt_part_floats(cap, hidden, ffn, 256) < need) {
          std::printf("cap %d hidden %d ffn %d\n", cap, hidden, ffn);
          return 1;
        }
      }
  return 0;
}
"""

SAME = r"""
#include <cstdio>
#include "split_k.h"
int main() {
  long more = 0;
  for (int cus : {256, 304, 64})
    for (int N : {128, 512, 1024, 2048, 4096, 6144, 8192, 12288})
      for (int K : {64, 576, 1024, 2048, 3584, 6144, 8192}) {
        size_t room = 0;
        for (int M = 1; M <= 1100; ++M) {
          const size_t r = q35::mb_part_room(M, N, cus);
          if (r < room) {
            std::printf("room falls at M %d N %d\n", M, N);
            return 1;
          }
          room = r;
          for (int d = 0; d < 2; ++d) {
            const int all = q35::mb_splits(M, N, K, cus, d, ~(size_t)0 >> 1);
            more += all > 4;
            if (q35::mb_splits(M, N, K, cus, d, r) != all || (all > 1 && (size_t)all * M * N > r)) {
              std::printf("M %d N %d K %d cus %d: %d splits, asked room gives %d\n", M, N, K, cus, all,
                          q35::mb_splits(M, N, K, cus, d, r));
              return 1;
            }
          }
        }
      }
  std::printf("%ld\n", more);
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


def test_asked_room_gives_the_same_splits(tmp_path):
    assert int(run(tmp_path, SAME)) > 1000
