"""Where the prefill tiles with groups hold weights for 128 k (csrc/wide_ring.h), on the CPU: the header itself compiled with the host compiler."""
import ctypes
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "nano-vllm-hw3_amd", "csrc")
SOURCE = """#include "wide_ring.h"
extern "C" int alone(long long rows, long long cols, long long k) { return wide_alone((rows + 95) / 96, (cols + 255) / 256, k); }
"""


@pytest.fixture(scope="module")
def alone(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host compiler")
    where = tmp_path_factory.mktemp("wide_ring")
    (where / "ring.cpp").write_text(SOURCE)
    subprocess.check_call([cxx, "-O1", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, str(where / "ring.cpp"), "-o", str(where / "ring.so")])
    fn = ctypes.CDLL(str(where / "ring.so")).alone
    fn.argtypes = [ctypes.c_longlong] * 3
    return fn


@pytest.mark.parametrize("M,N,K,held", [(264, 20224, 512, False), (488, 9728, 768, False), (352, 11008, 768, True), (352, 11008, 1280, True),     # few row tiles
                                        (768, 8192, 1152, True), (769, 7168, 1152, False), (2222, 2048, 1536, False),                            # short k
                                        (769, 7168, 2176, True), (5650, 1024, 7424, True), (24576, 256, 2176, True),                             # long k
                                        (24577, 256, 7424, False), (3072, 2304, 4096, False)])                                                   # two tiles for some CU
def test_which_tiles_hold_weights_for_128_k(alone, M, N, K, held):
    assert bool(alone(M, N, K)) == held
