"""paged_plan.h, by which paged attention's launches have 4 or 8 waves a workgroup and write a step's tokens, compiled for the CPU: its
lines lie where they were measured."""
import ctypes
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "vllm-splitwise_amd", "csrc")
PROGRAM = r"""
#include "paged_plan.h"
extern "C" int wide(int workgroups, int key_bytes, int longest, int writes_all) { return sw::pa_wide(workgroups, key_bytes, longest, writes_all); }
extern "C" int writes_all(int tokens, int sequences) { return sw::pa_writes_all(tokens, sequences); }
"""


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    at = tmp_path_factory.mktemp("plan")
    (at / "plan.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC", "-I", CSRC, str(at / "plan.cpp"), "-o",
                    str(at / "plan.so")], check=True)
    return ctypes.CDLL(str(at / "plan.so"))


@pytest.mark.parametrize("workgroups,key_bytes,longest,writes_all,waves", [
    (2 * 32, 256, 700, 1, 8), (8 * 32, 256, 2000, 0, 8), (10 * 32, 256, 2500, 0, 4), (8 * 40, 128, 1800, 0, 8), (43 * 12, 128, 700, 0, 4),
    # contexts of one step of 4 waves: without a write, with tokens looked up, with all of them written by everyone
    (24 * 12, 128, 125, 0, 4), (40 * 12, 128, 50, 0, 4), (1, 256, 256, 0, 4), (1, 256, 257, 0, 8), (8 * 32, 256, 125, 1, 8), (16 * 12, 128, 125, 1, 8),
    (1, 256, 1, 1, 8), (16 * 32, 256, 125, 1, 4)])
def test_waves(plan, workgroups, key_bytes, longest, writes_all, waves):
    assert (8 if plan.wide(workgroups, key_bytes, longest, writes_all) else 4) == waves


@pytest.mark.parametrize("tokens,sequences,everyone", [(1, 1, 1), (4, 4, 1), (5, 5, 0), (16, 16, 0), (128, 128, 0), (5, 4, 1), (16, 1, 1), (3, 128, 1)])
def test_who_writes_all_tokens(plan, tokens, sequences, everyone):
    assert plan.writes_all(tokens, sequences) == everyone
