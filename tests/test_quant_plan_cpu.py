"""quant_plan.h, by which int4 GEMMs are shared out among the kernels, compiled for the CPU: the sizes that the GPU tests give each kernel
go there, every size goes to a kernel that takes it, and the rule's two lines lie where they were measured."""
import ctypes
import os
import subprocess

import pytest
import test_quant_gpu as gpu

CSRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "vllm-splitwise_amd", "csrc")
WAYS = ["kAcrossWaves", "k32x128", "k64x64", "k64x128", "k128x128", "k128x256", "k64Rows"]
PROGRAM = r"""
#include "quant_plan.h"
extern "C" int way(long m, long n, long k, long group, int on16, int room) { return (int)sw::int4_way(m, n, k, group, on16, room); }
"""


@pytest.fixture(scope="module")
def way(tmp_path_factory):
    at = tmp_path_factory.mktemp("plan")
    (at / "plan.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC", "-I", CSRC, str(at / "plan.cpp"), "-o",
                    str(at / "plan.so")], check=True)
    lib = ctypes.CDLL(str(at / "plan.so"))
    return lambda m, k, n, group=128, on16=1, room=1: WAYS[lib.way(*map(ctypes.c_long, (m, n, k, group)), on16, room)]


@pytest.mark.parametrize("name", WAYS)
def test_the_gpu_tests_sizes_go_to_the_kernel_that_they_name(way, name):
    assert gpu.ROUTES[name] and all(way(*shape) == name for shape in gpu.ROUTES[name])


@pytest.mark.parametrize("m,k,n,name", [
    # across waves: measured the faster one, or level
    (8, 28672, 8192, "kAcrossWaves"), (12, 5120, 5120, "kAcrossWaves"), (28, 5120, 5120, "kAcrossWaves"), (20, 8192, 5120, "kAcrossWaves"),
    (17, 14336, 4096, "kAcrossWaves"), (24, 11008, 4096, "kAcrossWaves"),
    (16, 8192, 10240, "k32x128"), (17, 12288, 6144, "k32x128"), (32, 11008, 4096, "k32x128"), (9, 28672, 8192, "k32x128"),
    # long walks above 64 rows, and what was measured the other way
    (256, 28672, 8192, "k128x128"), (224, 28672, 8192, "k128x128"), (256, 14336, 8192, "k128x128"), (65, 28672, 8192, "k128x128"),
    (64, 28672, 8192, "k64x64"), (160, 8192, 10240, "k64x128"), (96, 8192, 8192, "k64x64"), (192, 6912, 5064, "k64x64"),
    (256, 5120, 27648, "k128x256")])
def test_the_lines_lie_where_they_were_measured(way, m, k, n, name):
    assert way(m, k, n) == name


def test_every_size_goes_to_a_kernel_that_takes_it(way):
    import random
    rng = random.Random(4)
    for _ in range(20000):
        m, k, n = rng.randrange(1, 600), 32 * rng.choice([1, 3, 8, rng.randrange(1, 900)]), 8 * int(2 ** rng.uniform(0, 13.5))
        group = rng.choice([32, 64, 96, 128, k])
        on16, room = rng.randrange(2), rng.randrange(2)
        name = way(m, k, n, group, on16, room)
        if name not in ("kAcrossWaves",):
            assert k % 256 == 0
        if name in WAYS[1:5]:
            assert on16 or (room and m > 32)
        if name == "k128x256":
            assert group % 64 == 0 and m > 128
        if name == "k64Rows":
            assert m > 128
        if m > 128 and k % 256 == 0:
            assert name != "kAcrossWaves" or group % 16
