"""The dense projections' choice of a kernel (strixite_amd/csrc/dense_plan.hpp) on the CPU."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include "dense_plan.hpp"
#include <cstdio>
using namespace strix::kernels::dnp;
int main() {
    long bits, G, M, N, K, f32;
    const char *name[] = {"tiles", "stream", "gemm"};
    while (std::scanf("%ld %ld %ld %ld %ld %ld", &bits, &G, &M, &N, &K, &f32) == 6)
        std::puts(name[(int)plan(bits, G, M, N, K, f32, K % 64 == 0 && G % 64 == 0 && K / G <= 48)]);
}
"""


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("needs g++")
    tmp = tmp_path_factory.mktemp("plan")
    (tmp / "p.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++20", "-O1", "-I", os.path.join(ROOT, "strixite_amd", "csrc"), str(tmp / "p.cpp"), "-o",
                    str(tmp / "p")], check=True)

    def ask(cases):  # (bits, G, M, N, K, FP32 outputs)
        text = "\n".join(" ".join(str(int(v)) for v in c) for c in cases)
        return subprocess.run([str(tmp / "p")], input=text, check=True, capture_output=True, text=True).stdout.split()

    return ask


def test_plans_can_run(plan):
    cases = [(bits, G, M, N, K, f32) for bits in (4, 8) for G in (32, 64, 128) for f32 in (0, 1)
             for M in (1, 16, 63, 64, 127, 128, 2000, 60000) for N in (16, 528, 4096, 151936) for K in (128, 2048, 4096, 32768)]
    for c, kernel in zip(cases, plan(cases), strict=True):
        bits, G, M, N, K, f32 = c
        if kernel == "gemm":
            assert G >= 64 and K // G <= 48 and M >= (128 if f32 else 64), c
        if kernel == "stream":
            assert K in (128, 2048), c
        if kernel != "tiles":
            assert max(N * K * bits // 8, 2 * M * K, M * N * (4 if f32 else 2)) < 1 << 31, c


# sizes where one kernel is clearly the fastest of the three (us: tiles, stream, GEMM)
@pytest.mark.parametrize("case,kernel", [
    ((4, 128, 100, 1024, 3072, 0), "tiles"),     # 10 / 25 / 41
    ((8, 64, 100, 4096, 4096, 0), "tiles"),      # more groups than the GEMM takes
    ((4, 128, 127, 4096, 3072, 0), "tiles"),     # 23 / 27 / 42
    ((8, 128, 100, 4096, 2048, 0), "stream"),    # 32 / 21 / 35
    ((4, 64, 127, 4096, 1024, 0), "stream"),     # 19 / 14 / 19
    ((8, 128, 1, 32768, 2048, 1), "stream"),     # 31 / 19 / 38
    ((4, 128, 1, 131072, 2048, 0), "stream"),    # 55 / 37 / 45
    ((4, 32, 1, 32768, 512, 0), "stream"),       # 15 / 11
    ((4, 32, 700, 4096, 3072, 0), "tiles"),      # 405 / 440
    ((8, 32, 560, 10464, 1408, 0), "tiles"),     # 275 / 412
    ((8, 128, 100, 4096, 1536, 0), "tiles"),     # 17 / 18
    ((8, 64, 2000, 4096, 3072, 1), "gemm"),
    ((4, 128, 64, 131072, 2048, 0), "gemm"),     # 246 / 229 / 52
    ((4, 128, 64, 131072, 3072, 1), "tiles"),    # FP32 outputs below 128 tokens: not the GEMM
])
def test_the_fastest_kernel(plan, case, kernel):
    assert plan([case]) == [kernel]
