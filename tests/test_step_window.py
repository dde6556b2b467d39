"""Buffer loads of steps past a walk's last one (csrc/step_window.h), on the CPU: the header itself compiled with the host compiler.  Whatever
a lane asks for lies inside the activations or is refused, under both readings of the range check: the resource's bytes less the
uniform offset in 32 bits, and the lane's offset against the bytes alone."""
import ctypes
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "nano-vllm-hw3_amd", "csrc")
SOURCE = """#include "step_window.h"
extern "C" long long outside(unsigned M, unsigned K, unsigned BM) {       // reads past the end of M rows of K 16-bit numbers; < 0: one missing
    const unsigned row = 2 * K, bytes = M * row;
    const int steps = row / 256;
    long long bad = 0;
    for (int t = 0; t < steps + 2; ++t) {
        const StepWindow w = step_window(t, steps, 256, bytes);
        for (unsigned r = 0; r < (M + BM - 1) / BM * BM; ++r)
            for (unsigned c = 0; c < 16; ++c) {
                const unsigned lane = r * row + 16 * c;
                const unsigned long long at = (unsigned long long)lane + w.at;
                const bool in = lane < w.bytes - w.at, loose = lane < w.bytes;
                if ((in || loose) && at + 16 > bytes) ++bad;
                if (t < steps && r < M && (!in || at != (unsigned long long)r * row + 256ull * t + 16 * c)) return -1;
            }
    }
    return bad;
}
"""


@pytest.fixture(scope="module")
def window(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host compiler")
    where = tmp_path_factory.mktemp("step_window")
    (where / "window.cpp").write_text(SOURCE)
    subprocess.check_call([cxx, "-O1", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, str(where / "window.cpp"), "-o", str(where / "window.so")])
    lib = ctypes.CDLL(str(where / "window.so"))
    lib.outside.restype = ctypes.c_longlong
    return lib


@pytest.mark.parametrize("BM", [64, 96, 128])
@pytest.mark.parametrize("M,K", [(1, 128), (64, 128), (65, 256), (97, 384), (128, 1024), (200, 2560)])
def test_nothing_is_read_past_the_activations(window, M, K, BM):
    assert window.outside(M, K, BM) == 0
