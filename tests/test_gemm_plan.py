"""The rule that picks a prefill GEMM's output tile (fe_gemm_plan, host arithmetic), compiled here: what it takes for 256 CUs where the forms
were timed against each other on an MI355X and differ by more than 5 %."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
MAIN = r"""
#include <cstdio>
#include <cstdlib>
#include <string>
#include "fe_internal.h"
int main(int argc, char **argv) {
    for (int i = 1; i + 3 < argc; i += 4) {
        const std::string form = argv[i];
        const uint32_t m = atoi(argv[i + 1]), n = atoi(argv[i + 2]), k = atoi(argv[i + 3]);
        const bool f8 = form == "fp8", bf = form == "bf16";
        const FeGemmCost &c = form == "trellis" ? kFeCostTrellis : form == "nvfp4" ? kFeCostNvfp4 : f8 ? kFeCostFp8 : kFeCostBf16;
        const FeGemmPlan p = fe_gemm_plan(m, n, k / (f8 ? 128 : 64), 256, 1, (size_t)512 * kFeGemmPartBytes, 1, 8192, 8, bf ? 0 : 1, !f8 && !bf, c, FeGemmTileOptions{});
        printf("%u\n", p.tile);
    }
}
"""
# (form, rows, columns, K): the tile (0: 256 x 256, 1: 128 x 256, 2: 128 x 128); us of the taken form and of the other
TIMED = {
    ("trellis", 1424, 5632, 2048): 0,   # 68.2, 128 x 128 79.2
    ("trellis", 1536, 5632, 2048): 0,   # 69.5, 79.9
    ("trellis", 1650, 5632, 2048): 2,   # 81.1, 256 x 256 86.2
    ("trellis", 1408, 5632, 2048): 1,   # 51.7, 68.4
    ("trellis", 1280, 8704, 2560): 2,   # 95.2, 100.1
    ("nvfp4", 1536, 5632, 2048): 2,     # 52.5, 60.5
    ("nvfp4", 1100, 8704, 5120): 2,     # 111, 124
    ("bf16", 192, 5120, 17408): 1,      # 59 in 6 pieces of K, 67
    ("bf16", 1280, 5120, 8704): 1,      # 114, 124
    ("fp8", 777, 17408, 5120): 1,       # 80, 88
    ("fp8", 2048, 5120, 8704): 1,       # 110, 118
    ("bf16", 640, 5120, 17408): 0,      # 116; nearest small tile 129
}


def test_the_tile_that_was_timed_faster(tmp_path):
    src = tmp_path / "plan.cpp"
    src.write_text(MAIN)
    exe = str(tmp_path / "plan")
    # (the header's device buffers refer to the library, which the plan does not touch)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", os.path.join(ROOT, "ferrite_amd", "csrc"), "-I", os.path.join(ROOT, "include"), str(src), "-o", exe,
                    "-Wl,--unresolved-symbols=ignore-all"], check=True)
    args = [str(v) for key in TIMED for v in key]
    got = [int(v) for v in subprocess.run([exe, *args], stdout=subprocess.PIPE, text=True, check=True).stdout.split()]
    for key, tile in zip(TIMED, got):
        assert tile == TIMED[key], key
