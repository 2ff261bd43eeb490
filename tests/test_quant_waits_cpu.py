"""The streamed int4 GEMM waits for its loads by their number, "all but the N newest": that holds only while the compiler leaves them as
they are written, with none added (a spilled register), split or moved behind a wait.  So every path through the loop of the built
kernels is followed: what may be in flight at each barrier is what the source says.  Reads the code that was built here."""
import os
import re
import struct
import subprocess

import pytest

LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "vllm-splitwise_amd", "splitwise_amd", "libsplitwise_hip.so")
TOOLS = "/opt/rocm/llvm/bin"


@pytest.fixture(scope="module")
def code(tmp_path_factory):
    """-> the path of the code object that holds the streamed kernels."""
    if not os.path.exists(LIB) or not os.path.exists(os.path.join(TOOLS, "llvm-objdump")):
        pytest.skip("needs the built library and llvm-objdump")
    with open(LIB, "rb") as f:
        data = f.read()
    for m in re.finditer(rb"__CLANG_OFFLOAD_BUNDLE__", data):
        at = m.start() + 32
        for _ in range(struct.unpack_from("<Q", data, m.start() + 24)[0]):
            offset, size, length = struct.unpack_from("<QQQ", data, at)
            part = data[m.start() + offset:m.start() + offset + size]
            if b"gfx950" in data[at + 24:at + 24 + length] and b"gptq_gemm_stream_kernel" in part:
                path = tmp_path_factory.mktemp("code") / "quant.elf"
                path.write_bytes(part)
                return str(path)
            at += 24 + length
    pytest.fail("no streamed kernel in the library")


def test_no_registers_are_spilled(code):
    notes = subprocess.run([os.path.join(TOOLS, "llvm-readelf"), "--notes", code], capture_output=True, text=True, check=True).stdout
    found = 0
    for kernel in notes.split("    .name:")[1:]:
        if "gptq_gemm_stream_kernel" in kernel.split("\n")[0]:
            found += 1
            for field in ("private_segment_fixed_size", "vgpr_spill_count"):
                assert re.search(rf"\.{field}:\s+(\d+)", kernel).group(1) == "0"
    assert found == 4


def _kernels(code):
    text = subprocess.run([os.path.join(TOOLS, "llvm-objdump"), "-d", code], capture_output=True, text=True, check=True).stdout
    parts = re.split(r"\n[0-9a-f]+ <([^>]*)>:\n", text)
    for name, body in zip(parts[1::2], parts[2::2]):
        if "gptq_gemm_stream_kernel" not in name:
            continue
        program = []                                         # (address, instruction, address of a branch's target)
        for line in body.split("\n"):
            m = re.match(r"\s+(\S[^/]*?)\s*// ([0-9A-F]+):", line)
            if m:
                target = re.search(r"<[^>+]*(?:\+0x([0-9a-f]+))?>\s*$", line)
                program.append((int(m.group(2), 16), m.group(1), int(target.group(1) or "0", 16) if target else None))
        yield name, program


def _check(program, rows, groups, ring):
    """Follows every path up to the wait for everything behind the loop.  In flight, oldest first: A for a load to LDS, w for one of a
    weight, scale or zero."""
    k = 256 // groups
    a, w = "A" * (rows * k // 128), "w" * (2 * (k // 32 // (8 // groups)) + 2)
    at_first, in_loop = w + (a + w) * (ring - 2) + a, w + (a + w) * (ring - 2)
    first = program[0][0]
    index = {address - first: i for i, (address, _, _) in enumerate(program)}
    todo, seen, barriers, ends = [(0, "")], set(), {}, 0
    while todo:
        i, flying = todo.pop()
        if (i, flying) in seen:
            continue
        seen.add((i, flying))
        assert len(flying) <= 63, "more in flight than the counter holds"
        _, op, target = program[i]
        name = op.split()[0]
        if name == "s_endpgm":                               # workgroups past the last tile
            assert flying == ""
            continue
        assert not name.startswith("scratch_"), "a spill"
        if re.match(r"(buffer|global|flat)_", name):
            assert re.match(r"buffer_load_dword(x2|x4)?$", name), op
            flying += "A" if re.search(r"\blds\b", op) else "w"
        if name == "s_waitcnt":
            count = re.search(r"vmcnt\((\d+)\)", op)
            if count:
                left = int(count.group(1))
                flying = flying[len(flying) - left:] if left else ""
                if left == 0:
                    ends += 1                                # the loop is through
                    continue
        if name == "s_barrier":
            barriers[i] = barriers.get(i, set()) | {flying}
        if name == "s_branch":
            todo.append((index[target], flying))
        else:
            if name.startswith("s_cbranch"):
                todo.append((index[target], flying))
            todo.append((i + 1, flying))
    assert ends and len(barriers) == 1 + ring
    assert barriers.pop(min(barriers)) == {at_first}
    assert all(flying == {in_loop} for flying in barriers.values())


def test_what_is_in_flight_at_every_barrier(code):
    found = []
    for name, program in _kernels(code):
        rows, groups, ring = map(int, re.search(r"ILi(\d+)ELi(\d+)ELi(\d+)ELi\d+E", name).groups())
        found.append((rows, groups, ring))
        _check(program, rows, groups, ring)
    assert sorted(found) == [(1, 2, 4), (2, 1, 3), (2, 2, 3), (4, 2, 3)]


@pytest.mark.parametrize("change", ["a spill", "a load more", "a load less", "a wait less", "a store"])
def test_a_changed_kernel_is_noticed(code, change):
    name, program = next(k for k in _kernels(code) if "ILi2ELi1ELi3E" in k[0])
    loads = [i for i, (_, op, _) in enumerate(program) if op.startswith("buffer_load_dwordx2")]
    waits = [i for i, (_, op, _) in enumerate(program) if "vmcnt(12)" in op]
    at = loads[5] if "wait" not in change else waits[-1]
    address, _, target = program[at]
    op = {"a spill": "scratch_load_dword v1, off, off", "a load more": program[at][1], "a load less": "s_nop 0",
          "a wait less": "s_nop 0", "a store": "global_store_dword v[0:1], v2, off"}[change]
    if change == "a load more":
        nops = [i for i in range(at + 1, len(program)) if program[i][1].startswith("v_")]
        at, (address, _, target) = nops[0], program[nops[0]]
    program[at] = (address, op, target)
    with pytest.raises(AssertionError):
        _check(program, 2, 1, 3)
