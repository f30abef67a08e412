"""The dynamic LDS allowance of the kernels (strixite_amd/csrc/lds_grant.hpp) on the CPU, against a stand-in for the HIP
runtime: asked for once a device and size, asked for again after a refusal."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include "lds_grant.hpp"
#include <cstdio>
static int device = 0, calls = 0;
static bool refuse = false;
extern "C" hipError_t hipGetDevice(int *d) { *d = device; return hipSuccess; }
extern "C" hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) {
    ++calls;
    return refuse ? hipErrorInvalidValue : hipSuccess;
}
int main() {
    int a, b;
    auto ask = [](int dev, const void *k, size_t n) {
        device = dev;
        const int before = calls;
        const hipError_t e = strix::kernels::allow_lds(k, n);
        std::printf("%d%d ", calls - before, e == hipSuccess);
    };
    ask(0, &a, 100000), ask(0, &a, 90000), ask(0, &a, 110000);  // first, less, more
    ask(1, &a, 100000), ask(1, &a, 100000);                     // another device of the process
    refuse = true, ask(0, &b, 100000);
    refuse = false, ask(0, &b, 100000), ask(0, &b, 100000);
}
"""


@pytest.mark.skipif(shutil.which("g++") is None or not os.path.exists("/opt/rocm/include/hip/hip_runtime_api.h"),
                    reason="needs g++ and the HIP headers")
def test_lds_allowed_once_a_device(tmp_path):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++20", "-D__HIP_PLATFORM_AMD__", "-I", "/opt/rocm/include", "-I",
                    os.path.join(ROOT, "strixite_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split()
    assert out == ["11", "01", "11", "11", "01", "10", "11", "01"]  # {runtime calls, success} of each ask
