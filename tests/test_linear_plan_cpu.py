"""linear_plan.h, by which a linear-attention step is shared out between the decode kernels and the walk, compiled for the CPU:
its bounds hold for every batch, decoding sequences do not walk beside a prompt's portion, and a long run of few heads is cut."""
import os
import shutil
import subprocess

import pytest

HEADER = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "vllm-splitwise_amd", "csrc", "mixers")

PROGRAM = r"""
#include "linear_plan.h"
#include <cstdio>
#include <cstdlib>
#include <vector>
#include <algorithm>
using namespace swm;
static void need(bool ok, const char* what) { if (!ok) { std::printf("%s\n", what); std::exit(1); } }
int main() {
  std::srand(3);
  for (int trial = 0; trial < 200000; ++trial) {
    const int seqs = 1 + std::rand() % (trial % 5 ? 12 : 300), heads = 1 << std::rand() % 6;
    const int dim = 8 * (1 + std::rand() % 32), vdim = 1 + std::rand() % 256;
    std::vector<int> lens;
    const int kind = std::rand() % 4;
    for (int s = 0; s < seqs; ++s)
      lens.push_back(kind == 0 ? 1 : kind == 1 ? std::rand() % 40 : kind == 2 ? std::rand() % 3000 : s ? 1 : std::rand() % 40000);
    long rows = 0, most = 0;
    for (int n : lens) rows += n, most = std::max<long>(most, n);
    const LinearWalkPlan p = linear_walk_plan(trial % 2, rows, seqs, (int)most, heads, dim, vdim);
    if (p.at_most >= most) { need(p.floats == 0 && p.segment == 0, "scratch for nothing"); continue; }
    long runs = 0, chunks = 0, items = 0;
    for (int n : lens)
      if (n > p.at_most) {
        ++runs;
        chunks += (n + 31) / 32;
        items += p.segment ? (n + p.segment - 1) / p.segment : 1;
      }
    need(runs <= p.runs && chunks <= p.chunks && items <= p.items, "a bound that does not hold");
    need(p.segment % 32 == 0, "a segment that ends inside a chunk");
    const int64_t groups = linear_walk_groups(p, heads, vdim), walkers = linear_walkers(p, heads, dim, vdim), width = (vdim + 15) / 16;
    need(groups >= p.items * heads * width && walkers > 0 && walkers <= groups && walkers % (8 * width) == 0, "whole eights of workgroups");
    need(walkers == groups || (p.at_most > 0 && walkers >= 496), "workgroups that go on");
    const long dp = (dim + 31) / 32 * 32, vb = (vdim + 15) / 16;
    need(p.floats >= p.chunks * heads * (65 * dp + 1024) + (p.segment ? p.items * heads * (16 * vb * dp + dp) : 0), "scratch");
  }
  // many short runs fill the GPU: no prologue, no walk
  need(linear_walk_plan(true, 64 * 17, 64, 17, 16, 128, 128).floats == 0, "64 x 17 walk");
  need(linear_walk_plan(false, 64 * 100, 64, 100, 16, 128, 128).floats == 0, "64 x 100 walk");
  // few do not
  need(linear_walk_plan(true, 4 * 100, 4, 100, 4, 128, 128).at_most == 0, "4 x 100 do not walk");
  // decoding sequences beside a portion go their own way
  for (int portion : {300, 1000, 8000}) {
    const LinearWalkPlan p = linear_walk_plan(true, 250 + portion, 251, portion, 16, 128, 128);
    need(p.at_most == 16, "250 decoding sequences walk");
  }
  // ... and leave no queue of workgroups that find no piece: 251 sequences, 1250 rows may be 73 runs, 9344 workgroups, and are one run
  const LinearWalkPlan mixed = linear_walk_plan(true, 1250, 251, 1000, 16, 128, 128);
  need(linear_walk_groups(mixed, 16, 128) == 9344 && linear_walkers(mixed, 16, 128, 128) == 512, "250 decoding sequences' workgroups");
  // a long run of few heads is cut into as many pieces as the GPU has room for
  for (int n : {8000, 16000, 32000}) {
    const LinearWalkPlan p = linear_walk_plan(false, n, 1, n, 4, 128, 128);
    need(p.segment > 0 && p.segment <= n / 7, "one chain");
  }
  need(linear_walk_plan(true, 32 * 2000, 32, 2000, 16, 128, 128).segment == 0, "runs that fill the GPU are cut");
  std::printf("ok\n");
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_plan(tmp_path):
    source = tmp_path / "plan.cpp"
    source.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", HEADER, str(source), "-o", str(tmp_path / "plan")], check=True)
    done = subprocess.run([str(tmp_path / "plan")], capture_output=True, text=True, timeout=60)
    assert done.returncode == 0 and done.stdout == "ok\n", done.stdout
