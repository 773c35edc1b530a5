"""Registers of the expert GEMM kernels, from the metadata that the compiler writes
into the built library: none may spill.  (With spills in its loops the Q4_1 prefill
took 1.3 to 1.5 times as long.)"""
import os
import re
import struct
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "pokitlms_amd", "libpokit_hip.so")
READELF = "/opt/rocm/llvm/bin/llvm-readelf"
EM_AMDGPU = 224


def code_objects(data):
    """The gfx950 ELF images inside the library (its own code only)."""
    at = data.find(b"\x7fELF", 1)
    while at >= 0:
        if struct.unpack_from("<H", data, at + 18)[0] == EM_AMDGPU:
            shoff, = struct.unpack_from("<Q", data, at + 40)
            shentsize, shnum = struct.unpack_from("<HH", data, at + 58)
            yield data[at:at + shoff + shentsize * shnum]
        at = data.find(b"\x7fELF", at + 4)


@pytest.fixture(scope="module")
def spills(tmp_path_factory):
    """Kernel name -> spilled vector registers."""
    if not os.path.exists(READELF) or not os.path.exists(LIB):
        pytest.skip("needs llvm-readelf and the built library")
    with open(LIB, "rb") as f:
        data = f.read()
    out, path = {}, str(tmp_path_factory.mktemp("co") / "co.elf")
    for image in code_objects(data):
        with open(path, "wb") as f:
            f.write(image)
        notes = subprocess.run([READELF, "--notes", path], capture_output=True, text=True).stdout
        names = re.findall(r"^    \.name: +(\S+)$", notes, re.M)
        counts = re.findall(r"^    \.vgpr_spill_count: +(\d+)$", notes, re.M)
        assert len(names) == len(counts)
        out.update(zip(names, map(int, counts)))
    return out


def test_expert_gemms_do_not_spill(spills):
    mine = {k: v for k, v in spills.items() if "k_expert_gemmI" in k}
    assert len(mine) == 13 and not any(mine.values()), mine  # 6 formats x gate/up and down, and precise Q4_K
