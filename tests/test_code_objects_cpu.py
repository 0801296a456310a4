"""Registers of the built kernels, where a launch's width hangs on them.

The built library carries a gfx950 code object per source; its notes name every kernel's vector registers."""
import os
import re
import shutil
import struct
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "jitllm_amd", "lib", "libjitllm_hip.so")
READELF = shutil.which("llvm-readelf") or "/opt/rocm/llvm/bin/llvm-readelf"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects(data):
    """The gfx950 images in clang's offload bundles: count, then offset, size and triple of each entry."""
    at = data.find(MAGIC)
    while at >= 0:
        count, = struct.unpack_from("<Q", data, at + len(MAGIC))
        pos = at + len(MAGIC) + 8
        for _ in range(count):
            offset, size, triple = struct.unpack_from("<QQQ", data, pos)
            name = data[pos + 24:pos + 24 + triple]
            pos += 24 + triple
            if b"gfx950" in name and size:
                yield data[at + offset:at + offset + size]
        at = data.find(MAGIC, at + 1)


@pytest.fixture(scope="module")
def registers(tmp_path_factory):
    """{mangled kernel name: vector registers}"""
    if not os.path.exists(READELF):
        pytest.skip("no llvm-readelf")
    if not os.path.exists(LIB):
        from jitllm_amd.build import build
        build()
    found = {}
    with open(LIB, "rb") as f:
        data = f.read()
    for i, image in enumerate(code_objects(data)):
        path = tmp_path_factory.mktemp("objects") / f"{i}.co"
        path.write_bytes(image)
        notes = subprocess.run([READELF, "--notes", str(path)], capture_output=True, text=True, check=True).stdout
        # (a kernel's keys come sorted: its name before its registers)
        for name, count in re.findall(r"\.name:\s+(_Z\S+)\n(?:(?!\.name:).)*?\.vgpr_count:\s+(\d+)", notes, re.S):
            found[name] = int(count)
    assert found
    return found


def tiles_kernel(ggml_type, rms, slices, part):
    """jl_gemv_tiles for rows of one weight, 256 threads."""
    flag = "Lb1E" if rms else "Lb0E"
    return f"jl_gemv_tilesILi{ggml_type}ELb0E{flag}Lb0ELi256ELi{slices}ELb0ELb{int(part)}ELb0ELb0EE"


@pytest.mark.parametrize("rms", [False, True])
@pytest.mark.parametrize("slices,part", [(16, True), (32, False), (32, True), (64, False), (64, True)])
def test_q4_k_rows_of_one_weight_leave_room_for_five_waves(registers, rms, slices, part):
    """512 registers a lane, given out by eights: five waves of up to 96.  The grid of a launch is as wide as that."""
    want = tiles_kernel(12, rms, slices, part)
    counts = [c for name, c in registers.items() if want in name]
    assert len(counts) == 1 and counts[0] <= 96, (want, counts)
