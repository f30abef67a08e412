"""The hyper-connection mix's choice of a kernel (strixite_amd/csrc/hc_plan.hpp) on the CPU, at 256 CUs."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include "hc_plan.hpp"
#include <cstdio>
using namespace strix::kernels::hcp;
int main() {
    char what;
    long bits, f32, G, T, r, d;
    while (std::scanf(" %c %ld %ld %ld %ld %ld %ld", &what, &bits, &f32, &G, &T, &r, &d) == 7) {
        if (what == 'd') {
            const DownPlan p = plan_down(bits, f32, G, T, r, d, 256);
            const char *name[] = {"dots", "split", "tiles"};
            std::printf("%s %d %ld %zu %d\n", name[(int)p.kernel], p.split, (long)split_blocks(kSplits[p.split], T, r),
                        split_lds(kSplits[p.split], d, G), p.halves);
        } else {
            const UpPlan p = plan_up(bits, f32, T, d, r, G, 256);
            std::printf("%s%s 0 0 %zu\n", p.small ? "small" : "wide", p.two ? " two" : " one", up_lds(p.small ? 1 : 2, r, G));
        }
    }
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

    def ask(cases):  # (kind, bits, f32, G, T, rows (up: rank), d)
        text = "\n".join(" ".join(str(int(v) if not isinstance(v, str) else v) for v in c) for c in cases)
        out = subprocess.run([str(tmp / "p")], input=text, check=True, capture_output=True, text=True).stdout.splitlines()
        assert len(out) == len(cases)
        return [line.split() for line in out]

    return ask


def test_down_plans_can_run(plan):
    """Split-K blocks fit the LDS and the CUs, staged tiles have whole stages."""
    cases = [("d", bits, f32, G, T, R, d) for bits in (4, 8) for f32 in (0, 1) for G in (32, 64, 128)
             for T in (1, 2, 32, 33, 255, 256, 441, 1000, 4000, 65535) for R in (1, 20, 324, 1028)
             for d in (32, 96, 128, 160, 2560, 4096, 10240, 65536) if (4 * d) % G == 0]
    for c, (kernel, split, blocks, lds, _) in zip(cases, plan(cases)):
        _, _, f32, _, T, _, d = c
        if kernel == "split":
            assert not f32 and T > 32 and int(lds) <= 159 * 1024, c
            assert int(blocks) <= 256 or (split == "3" and d % 128), c
        elif kernel == "tiles":
            assert d % 128 == 0, c


def test_fp32_crossing_moves_with_the_rows(plan):
    """FP32 streams: lane dots cost tokens x rows, the staged tiles a K walk whatever the tokens, so the crossing in tokens
    falls as the rows grow (measured pairs of the kernels' times: dots cheaper below, tiles above)."""
    pairs = [(4, 2560, 68, 700, 8000), (4, 2560, 324, 400, 700), (4, 2560, 388, 400, 500), (4, 2560, 772, 128, 256),
             (4, 2560, 1024, 128, 256), (8, 2560, 388, 256, 439), (4, 1024, 324, 256, 439), (8, 2560, 1024, 64, 256)]
    below = plan([("d", b, 1, 64, lo, R, d) for b, d, R, lo, hi in pairs])
    above = plan([("d", b, 1, 64, hi, R, d) for b, d, R, lo, hi in pairs])
    assert [p[0] for p in below] == ["dots"] * len(pairs)
    assert [p[0] for p in above] == ["tiles"] * len(pairs)


def test_streams_too_wide_for_the_split_go_to_the_cheaper_kernel(plan):
    """BF16 streams whose split-K scale table does not fit the LDS: staged tiles where their K walk costs less than the lane
    dots' tokens x rows, the lane dots for few tokens and where a stream has no whole stages."""
    cases = [(4, 32, 1000, 324, 5120), (8, 32, 1000, 324, 5120), (4, 64, 1000, 324, 10240), (8, 64, 1000, 324, 10240),
             (4, 32, 1000, 324, 8192), (4, 32, 40, 8, 65536), (4, 32, 1000, 324, 5152)]
    got = plan([("d", b, 0, G, T, R, d) for b, G, T, R, d in cases])
    assert [p[0] for p in got] == ["tiles"] * 5 + ["dots"] * 2


def test_staged_tiles_take_k_in_halves_only_in_one_round_of_blocks(plan):
    """Q4, BF16: two halves of K where the blocks are at most the CUs (and with groups of 32), one where two blocks share a CU;
    one for Q8 and FP32 streams."""
    cases = [(4, 0, 64, 2000, 324), (4, 0, 64, 4000, 388), (4, 0, 128, 2000, 772), (4, 0, 32, 4000, 388), (8, 0, 64, 2000, 324),
             (4, 1, 64, 2000, 324)]
    got = plan([("d", b, f, G, T, R, 2560) for b, f, G, T, R in cases])
    assert [(p[0], p[4]) for p in got] == [("tiles", v) for v in "211211"]


def test_up_mix_shares_a_cu_only_where_the_lds_holds_two_blocks(plan):
    """The two-block variant: more blocks than CUs, twice the h tile within the 160 KB LDS, and not where it measured slower."""
    cases = [("u", bits, f32, G, T, r, 2560) for bits in (4, 8) for f32 in (0, 1) for G in (32, 64, 128)
             for T in (16, 17, 500, 2000) for r in (128, 320, 384, 448, 512, 768, 896) if r % G == 0]
    for c, (tile, blocks, _, _, lds) in zip(cases, plan(cases)):
        _, bits, f32, _, T, r, _ = c
        assert (tile == "small") == (T == 16 or r > 768), c
        want = tile == "wide" and T >= 500 and r <= 384 and (bits == 4 or (not f32 and r <= 128))
        assert (blocks == "two") == want and (not want or 2 * int(lds) <= 160 * 1024), c
