"""What the compiler made of the GEMM kernels in the built library: registers, which decide how many workgroups share a CU."""
import os
import re
import struct
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "nano-vllm-hw3_amd", "nanovllm", "_lib", "libqlinear.so")
READELF = "/opt/rocm/llvm/bin/llvm-readelf"
BF16, I8, F8 = 0, 1, 2                                     # activations


def code_objects(path):
    """The gfx950 code objects inside a library."""
    data = open(path, "rb").read()
    at = data.find(b"__CLANG_OFFLOAD_BUNDLE__")
    while at >= 0:
        count, p = struct.unpack_from("<Q", data, at + 24)[0], at + 32
        for _ in range(count):
            offset, size, n = struct.unpack_from("<QQQ", data, p)
            if size and b"gfx950" in data[p + 24:p + 24 + n]:
                yield data[at + offset:at + offset + size]
            p += 24 + n
        at = data.find(b"__CLANG_OFFLOAD_BUNDLE__", at + 24)


@pytest.fixture(scope="module")
def registers(tmp_path_factory):
    """Vector registers by kernel name."""
    if not os.path.exists(READELF):
        pytest.skip("no llvm-readelf")
    if not os.path.exists(LIB):
        import __graft_entry__
        __graft_entry__.build()
    found, where = {}, str(tmp_path_factory.mktemp("code") / "object")
    for code in code_objects(LIB):
        with open(where, "wb") as f:
            f.write(code)
        notes = subprocess.run([READELF, "--notes", where], capture_output=True, text=True, check=True).stdout
        for kernel in notes.split("- .agpr_count:")[1:]:
            found[re.search(r"\.name:\s+(\S+)", kernel)[1]] = int(re.search(r"\.vgpr_count:\s+(\d+)", kernel)[1])
    return found


def decode_kernel(act, fp8_weights, mt, wn, wk, cp):
    return f"_ZN2ql12qgemm_kernelILi{act}ELb{fp8_weights}ELi{mt}ELi{wn}ELi{wk}ELi{cp}" + "ELb0" * 8 + "EEEvNS_10GemmParamsE"


@pytest.mark.parametrize("act,fp8_weights,tile,most", [
    # workgroups of 8 waves, three per CU (6 waves per SIMD)
    (F8, 1, (1, 1, 8, 4), 80),
    # two per CU
    (BF16, 0, (1, 1, 8, 4), 128), (BF16, 1, (1, 1, 8, 4), 128), (I8, 0, (1, 1, 8, 4), 128),
    # 4 waves, three per CU
    (F8, 1, (1, 1, 4, 8), 168)])
def test_decode_tiles_leave_room_for_their_neighbours(registers, act, fp8_weights, tile, most):
    assert registers[decode_kernel(act, fp8_weights, *tile)] <= most
