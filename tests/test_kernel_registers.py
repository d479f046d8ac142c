"""What the kernels of libbr_hip.so, as they were built, take of a compute unit: the figures their code objects state."""
import os
import re
import struct
import subprocess

import pytest

READELF = "/opt/rocm/llvm/bin/llvm-readelf"


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{mangled name: (registers of a lane, bytes of scratch of a lane)}"""
    from blackriver_amd import hip
    if not os.path.exists(READELF):
        pytest.skip("no llvm-readelf")
    found, part = {}, tmp_path_factory.mktemp("code") / "object"
    with open(hip.LIB_PATH, "rb") as f:
        lib = f.read()
    for at in (m.start() for m in re.finditer(b"\x7fELF", lib)):
        if struct.unpack_from("<H", lib, at + 18)[0] != 224:   # EM_AMDGPU
            continue
        sections, = struct.unpack_from("<Q", lib, at + 40)
        size, count = struct.unpack_from("<HH", lib, at + 58)
        part.write_bytes(lib[at:at + sections + size * count])
        notes = subprocess.run([READELF, "--notes", str(part)], capture_output=True, text=True, check=True).stdout
        for text in notes.split("- .agpr_count")[1:]:
            def value(key):
                return re.search(r"\.%s:\s+(\S+)" % key, text)[1]
            found[value("name")] = (int(value("vgpr_count")), int(value("private_segment_fixed_size")))
    return found


def test_no_kernel_uses_scratch(kernels):
    assert kernels and {k: v for k, v in kernels.items() if v[1]} == {}


def test_small_tiles_of_fp32_products_leave_room_for_two_waves_a_simd(kernels):
    """Loaded in quads and value by value, apart and in pairs: up to 256 of a SIMD's 512 registers.  With one wave to a SIMD nothing
    runs while it waits for its loads, and many tiles take up to 1.7 times as long."""
    fp32 = {k: v for k, v in kernels.items() if re.search(r"gemm_flex_(pair_)?kernelILi2E", k)}
    assert len(fp32) >= 36
    assert {k: v for k, v in fp32.items() if v[0] > 256} == {}
