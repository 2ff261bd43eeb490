"""attention_plan.h, by which a step of the paged attention finds its kernels, compiled for the CPU."""
import os
import shutil
import subprocess

import pytest

HEADER = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "vllm-splitwise_amd", "csrc", "mixers")

PROGRAM = r"""
#include "attention_plan.h"
#include <cstdio>
#include <cstdlib>
using namespace swm;
static void need(bool ok, const char* what) { if (!ok) { std::printf("%s\n", what); std::exit(1); } }
int main() {
  // one query row over few keys: the vector kernel (a page of 16 keys, a table of `width` pages)
  auto way = [](int mql, int heads, int kv, int dim, int width, int window = 0, int chunk = 0) {
    return attention_way(true, 4, mql, heads, kv, dim, dim, 16, width, window, chunk);
  };
  for (int dim : {16, 32, 40, 64, 72, 96, 104, 128}) need(way(1, 8, 8, dim, 1) == kGeneralAttention, "one row, a page of keys");
  need(way(1, 8, 8, 128, 32) == kGeneralAttention && way(1, 8, 8, 128, 33) == kDecodeOnMatrixCores, "one row of 128");
  need(way(1, 8, 8, 64, 16) == kGeneralAttention && way(1, 8, 8, 64, 17) == kDecodeOnMatrixCores, "one row of 64");
  // up to 64 wide: 512 sequences x heads are one round of the matrix kernel's workgroups, more are two
  auto many = [](int seqs, int width) { return attention_way(true, seqs, 1, 8, 8, 64, 64, 16, width, 0, 0); };
  need(many(64, 17) == kDecodeOnMatrixCores && many(65, 64) == kGeneralAttention && many(96, 64) == kGeneralAttention, "512 and more");
  need(many(97, 17) == kDecodeOnMatrixCores && many(97, 16) == kGeneralAttention && many(129, 20) == kGeneralAttention, "1024");
  need(way(1, 8, 8, 64, 500, 200) == kGeneralAttention && way(1, 8, 8, 64, 500, 0, 256) == kGeneralAttention, "one row, masks");
  // more rows: the matrix cores whatever the keys
  need(way(2, 8, 8, 64, 1) == kDecodeOnMatrixCores && way(1, 8, 4, 64, 1) == kDecodeOnMatrixCores, "two rows");
  need(way(1, 8, 1, 64, 1) == kDecodeOnMatrixCores && way(9, 8, 8, 64, 1) == kGeneralAttention, "eight and nine rows");
  need(way(33, 8, 8, 64, 1) == kPromptOnMatrixCores && way(0, 8, 8, 64, 1) == kPromptOnMatrixCores, "a prompt");
  for (int mql = 0; mql < 70; ++mql) need(attention_way(false, 4, mql, 8, 8, 64, 64, 16, 100, 0, 0) == kGeneralAttention, "no pieces");
  // the prompt kernel's places in a page have 32 bits
  auto paged = [](int mql, int page, int64_t k, int64_t v) {
    return attention_way(true, 4, mql, 8, 8, 64, 64, page, 4, 0, 0, attention_page_bytes(page, k, v));
  };
  need(paged(40, 1 << 20, 2040, 512) == kPromptOnMatrixCores && paged(40, 1 << 20, 2048, 512) == kGeneralAttention &&
           paged(40, 1 << 20, 512, 2048) == kGeneralAttention && paged(0, 16, 1ll << 32, 512) == kGeneralAttention &&
           paged(40, 16, 1024, 1024) == kPromptOnMatrixCores && paged(2, 1 << 20, 2048, 512) == kDecodeOnMatrixCores, "pages of 4 GiB");
  // two groups of waves a walk: 16 query heads on 4, 32 tokens a workgroup
  auto groups = [](int64_t rows, int seqs, int mql, int width, int window = 0, int chunk = 0) {
    return prompt_attention_groups(rows, seqs, mql, 16, 4, 16, width, window, chunk);
  };
  need(prompt_attention_workgroups(65, 2, 16, 4) == 20 && prompt_attention_workgroups(64, 2, 16, 4) == 16, "workgroups");
  need(groups(240, 1, 240, 15) == 1 && groups(240, 1, 240, 16) == 2 && groups(240, 1, 240, 99, 255) == 1 && groups(240, 1, 240, 99, 256) == 2 &&
           groups(240, 1, 240, 99, 0, 255) == 1 && groups(240, 1, 240, 99, 0, 256) == 2, "keys");
  need(groups(63 * 32, 1, 2016, 126) == 2 && groups(62 * 32, 2, 1000, 126, 300) == 2 && groups(62 * 32 + 1, 2, 1000, 126, 300) == 1 &&
           groups(62 * 32 + 1, 2, 1000, 126, 0, 300) == 1, "a compute unit each");
  need(groups(62 * 32 + 1, 2, 1100, 70) == 2 && groups(98 * 32, 2, 50 * 32, 100) == 2 && groups(98 * 32, 2, 49 * 32, 100) == 1, "half of the workgroups");
  need(groups(3000, 5, 2900, 182) == 2 && groups(3000, 7, 2900, 182) == 1, "sequences beside");
  need(groups(127 * 32, 1, 4064, 254) == 2 && groups(127 * 32, 1, 4064, 900) == 2 && groups(128 * 32, 1, 4096, 900) == 1 &&
           groups(128 * 32, 1, 4096, 321) == 2 && groups(128 * 32, 1, 4096, 322) == 1, "keys in front of the prompt");
  need(groups(139 * 32, 1, 139 * 32, 278) == 2 && groups(139 * 32 + 1, 1, 139 * 32 + 1, 279) == 1, "the last line");
  need(groups(3000, 1, 0, 188) == 1 && groups(2000, 1, 0, 125) == 2, "longest unknown");
  // what the matrix kernels can read
  need(attention_pieces(0, 128, 128, 1024, 1024) && attention_pieces(32, 8, 120, 8, 120), "pieces");
  need(!attention_pieces(8, 128, 128, 1024, 1024) && !attention_pieces(0, 132, 128, 1024, 1024) &&
           !attention_pieces(0, 60, 64, 1024, 1024) && !attention_pieces(0, 64, 64, 1028, 1024), "no pieces");
  // keys are only shared out where the matrix kernel has the step
  for (int trial = 0; trial < 100000; ++trial) {
    const int kv = 1 + std::rand() % 8, heads = kv * (1 + std::rand() % 8), mql = std::rand() % 12, width = 1 + std::rand() % 600;
    const int dim = 8 * (1 + std::rand() % 16), window = std::rand() % 3 ? 0 : 1 + std::rand() % 3000;
    const int seqs = 1 + std::rand() % 20, parts = decode_attention_parts(seqs, mql, heads, kv, 16, width, window, 0);
    need(parts >= 1 && parts <= 16, "parts");
    if (parts > 1) need(attention_way(true, seqs, mql, heads, kv, dim, dim, 16, width, window, 0) == kDecodeOnMatrixCores, "shared keys");
  }
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
