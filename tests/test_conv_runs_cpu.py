"""How the short convolution's workgroups share the rows of a step out: conv_runs.h, which the kernel walks by, compiled for the
CPU.  Every row of a batch is some workgroup's exactly once, a sequence's first rows all one's, and the walk ends also where an
owner entry names a sequence that does not contain the row."""
import os
import shutil
import subprocess

import pytest

HEADER = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "vllm-splitwise_amd", "csrc", "mixers")

PROGRAM = r"""
#include "conv_runs.h"
#include <cstdio>
#include <cstdlib>
#include <vector>
using namespace swm;
static void need(bool ok, const char* what) { if (!ok) { std::printf("%s\n", what); std::exit(1); } }
int main() {
  std::srand(7);
  for (int trial = 0; trial < 20000; ++trial) {
    const int seqs = 1 + std::rand() % 6, keep = 1 + std::rand() % 3, run = trial % 2 ? 8 : 1;
    std::vector<int> start(1, 0), owner;
    for (int s = 0; s < seqs; ++s) {
      const int n = std::rand() % (trial % 3 ? 5 : 20);
      start.push_back(start.back() + n);
      owner.insert(owner.end(), n, s);
    }
    const bool bad = trial % 4 == 3;                     // padding rows, entries of somebody else
    if (bad) {
      for (int i = std::rand() % 5; i > 0; --i) owner.push_back(std::rand() % seqs);
      for (auto& o : owner) if (std::rand() % 6 == 0) o = std::rand() % seqs;
    }
    const long rows = (long)owner.size();
    std::vector<int> taken(rows, 0);
    for (long begin = 0; begin < rows; begin += run) {
      const long end = begin + run < rows ? begin + run : rows;
      long t = begin;
      for (int steps = 0; t < end; ++steps) {
        need(steps <= run, "more pieces than rows");
        const int s = owner[t];
        const ConvPiece p = conv_piece(t, end, start[s], start[s + 1], keep);
        need(p.next > t, "no way forward");
        if (p.what != kRowsElsewhere) {
          need(p.next <= rows, "beyond the step");
          for (long r = t; r < p.next; ++r) ++taken[r];
          if (p.what == kRowsInOrder) {
            need(t >= start[s] && p.next <= start[s + 1], "rows of another sequence");
            need(t > start[s] || p.next - t >= (keep < start[s + 1] - t ? keep : start[s + 1] - t), "first rows apart");
            need(t == start[s] || t >= start[s] + keep, "a carried input read after it may have moved on");
          }
        }
        t = p.next;
      }
    }
    if (!bad) for (long r = 0; r < rows; ++r) need(taken[r] == 1, "a row left out or taken twice");
  }
  std::printf("ok\n");
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_every_row_once_and_the_walk_ends(tmp_path):
    source = tmp_path / "runs.cpp"
    source.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", HEADER, str(source), "-o", str(tmp_path / "runs")], check=True)
    done = subprocess.run([str(tmp_path / "runs")], capture_output=True, text=True, timeout=60)
    assert done.returncode == 0 and done.stdout == "ok\n", done.stdout
