"""The launch of the matrix cores' paged attention asks for more than 64 KB of LDS by what it passes: so the kernels may hold none of
their own beside it.  Reads the code that was built here."""
import os
import re
import struct
import subprocess

import pytest

LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "vllm-splitwise_amd", "splitwise_amd", "libsplitwise_hip.so")
READELF = "/opt/rocm/llvm/bin/llvm-readelf"


def _fixed_lds(kernel, tmp_path):
    """{name: bytes} of the kernels whose name contains `kernel`, over the library's code objects."""
    with open(LIB, "rb") as f:
        data = f.read()
    out = {}
    for m in re.finditer(rb"__CLANG_OFFLOAD_BUNDLE__", data):
        at = m.start() + 32
        for _ in range(struct.unpack_from("<Q", data, m.start() + 24)[0]):
            offset, size, length = struct.unpack_from("<QQQ", data, at)
            part = data[m.start() + offset:m.start() + offset + size]
            if b"gfx950" in data[at + 24:at + 24 + length] and kernel.encode() in part:
                path = tmp_path / "code.elf"
                path.write_bytes(part)
                notes = subprocess.run([READELF, "--notes", str(path)], capture_output=True, text=True, check=True).stdout
                for entry in re.split(r"\n  - ", notes):
                    lds = re.search(r"\.group_segment_fixed_size:\s+(\d+)", entry)
                    if lds and kernel in entry:
                        out[re.findall(r"\.name:\s+(\S+)", entry)[-1]] = int(lds.group(1))
            at += 24 + length
    return out


@pytest.mark.skipif(not os.path.exists(LIB) or not os.path.exists(READELF), reason="needs the built library and llvm-readelf")
def test_matrix_kernels_hold_no_lds_of_their_own(tmp_path):
    found = _fixed_lds("paged_attention_mfma_kernel", tmp_path)
    assert len(found) == 4 * 2 * 2 * 2 * 2                # types, head sizes, blocks, waves, with and without the cache write
    assert not {k: v for k, v in found.items() if v}
