"""What the compiler made of the kernels in the built libraries: registers, which decide how many workgroups share a CU, and the states between a
matrix instruction and the first read of its result."""
import os
import re
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "tools"))

import mfma_waits  # noqa: E402

LIBS = os.path.join(ROOT, "nano-vllm-hw3_amd", "nanovllm", "_lib")
LIB = os.path.join(LIBS, "libqlinear.so")
READELF = "/opt/rocm/llvm/bin/llvm-readelf"
BF16, I8, F8 = 0, 1, 2                                     # activations


@pytest.fixture(scope="module")
def built():
    if not (os.path.exists(READELF) and os.path.exists(mfma_waits.OBJDUMP)):
        pytest.skip("no llvm-readelf or llvm-objdump")
    if not os.path.exists(LIB):
        import __graft_entry__
        __graft_entry__.build()


@pytest.fixture(scope="module")
def registers(built, tmp_path_factory):
    """Vector registers by kernel name."""
    found, where = {}, str(tmp_path_factory.mktemp("code") / "object")
    for code in mfma_waits.code_objects(LIB):
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


@pytest.mark.parametrize("lib,kernels", [("libqlinear.so", "qgemm_kernelILi2E"), ("libhymix.so", "outer_chunk")])
def test_results_of_matrix_instructions_are_whole_when_they_are_read(built, lib, kernels):
    """The kernels with matrix instructions of several lengths: fp8 x fp8 GEMMs, chunked recurrences (tools/mfma_waits.py looks at all)."""
    count = 0
    for code in mfma_waits.code_objects(os.path.join(LIBS, lib)):
        for name, instructions in mfma_waits.kernels(code, kernels):
            assert not mfma_waits.early_reads(instructions), name
            count += any(op.startswith("v_mfma") for op, _, _ in instructions)
    assert count > 5


K64, K16 = "v_mfma_scale_f32_32x32x64_f8f6f4", "v_mfma_f32_32x32x16_fp8_fp8"


@pytest.mark.parametrize("nops,early", [(5, [K64, K16]), (10, [K64]), (12, [K64]), (13, [])])
def test_a_read_behind_a_join_counts_from_the_longer_product(nops, early):
    """The K = 64 product on one path (a branch of five states behind it), the K = 16 one on the other: 19 states and 11."""
    code = [("s_cbranch_scc0", "2", 3), (K64, "v[2:17], v[20:27], v[28:35], v[2:17], v1, v1", None), ("s_branch", "1", 4),
            (K16, "v[2:17], v[20:21], v[28:29], v[2:17]", None), ("s_nop", str(nops), None), ("v_mov_b32_e32", "v40, v9", None), ("s_endpgm", "", None)]
    assert [f[0] for f in mfma_waits.early_reads(code)] == early
