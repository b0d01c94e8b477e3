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


FORM = r"""
#include <cstdio>
#include <cstdlib>
#include "fe_internal.h"
int main(int argc, char **argv) {
    for (int i = 1; i + 2 < argc; i += 3) {
        const uint32_t rows = atoi(argv[i]), n = atoi(argv[i + 1]), k = atoi(argv[i + 2]);
        const FeRgemmPlan p = fe_rgemm_plan(rows, k, &n, 1, 256, (size_t)512 * kFeGemmPartBytes, 0, 0);
        const FeGemmPlan g = fe_gemm_plan(rows, n, k / 64, 256, 1, (size_t)512 * kFeGemmPartBytes, 1, 8192, 8, 1, true, kFeCostTrellis, FeGemmTileOptions{});
        printf("%d\n", (int)fe_rgemm_takes(p, fe_rgemm_other_us(g, 256), 1));
    }
}
"""
# (rows, columns, K): whether a trellis prompt takes the GEMM that decodes into registers; us of the one that decodes through LDS and of this one
FORMS = {
    (507, 2048, 2048): 0,    # 20.2, 23.7
    (512, 1024, 2816): 0,    # 19.2, 22.2
    (1416, 896, 1664): 0,    # 21.2, 23.5
    (915, 2176, 640): 0,     # 14.8, 17.0
    (65, 2048, 5632): 1,     # 20.1, 14.8
    (309, 512, 8448): 1,     # 26.3, 19.5
    (128, 1024, 5120): 1,    # 18.4, 14.3
    (203, 5120, 17408): 1,   # 66.4, 52.3
    (512, 5120, 17408): 1,   # 105, 100
    (2048, 17408, 5120): 1,  # 339, 336
}


def test_the_trellis_gemm_that_was_timed_faster(tmp_path):
    src = tmp_path / "form.cpp"
    src.write_text(FORM)
    exe = str(tmp_path / "form")
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", os.path.join(ROOT, "ferrite_amd", "csrc"), "-I", os.path.join(ROOT, "include"), str(src), "-o", exe,
                    "-Wl,--unresolved-symbols=ignore-all"], check=True)
    args = [str(v) for key in FORMS for v in key]
    got = [int(v) for v in subprocess.run([exe, *args], stdout=subprocess.PIPE, text=True, check=True).stdout.split()]
    assert dict(zip(FORMS, got)) == FORMS


RGEMM = r"""
#include <cstdio>
#include "fe_internal.h"
// every plan covers its tiles once, within the workspace, with the row groups that kernels exist for
int main() {
    unsigned seed = 1;
    auto rnd = [&](unsigned lo, unsigned hi) { seed = seed * 1664525u + 1013904223u; return lo + (unsigned)((unsigned long long)(seed >> 8) * (hi - lo + 1) >> 24); };
    for (int i = 0; i < 200000; i++) {
        const uint32_t rows = rnd(0, 3) ? rnd(65, 2303) : rnd(65, 300), k = 128 * rnd(1, 140), count = rnd(1, 4), cus = rnd(0, 3) ? 256 : rnd(1, 304);
        uint32_t n[4];
        for (auto &v : n) v = 128 * rnd(1, 140);
        const uint32_t form = rnd(0, 3) ? 0 : rnd(1, 2), pieces = rnd(0, 3) ? 0 : rnd(1, 12);
        const size_t part = rnd(0, 9) ? (size_t)512 * 262144 : (size_t)rnd(0, 64) * 262144;
        const FeRgemmPlan p = fe_rgemm_plan(rows, k, n, count, cus, part, form, pieces);
        const uint32_t tiles = p.tiles_m * p.tiles_n, rest = tiles - p.full;
        uint32_t tn = 0;
        for (uint32_t j = 0; j < count; j++) tn += (n[j] / 128 + p.blocks - 1) / p.blocks;
        bool ok = p.us < 1e29f && (p.blocks == 1 || p.blocks == 2) && (rows <= 128 ? p.blocks == 1 : !form || p.blocks == form) && p.rg % 2 == 0 && p.rg <= 16 && p.rg >= (p.blocks == 1 ? 6u : 10u);
        ok = ok && p.tiles_n == tn && p.tiles_m * 16 * p.rg >= rows && (p.tiles_m - 1) * 16 * p.rg < rows && p.full <= tiles && p.k == k;
        ok = ok && 16 * (p.rg - 2) < rows;  // no piece of A lies past the end of the rows by its scalar offset alone
        const uint32_t loaders = 4 * p.blocks, pieces_a = (2 * p.rg + loaders - 1) / loaders;
        ok = ok && (uint64_t)(pieces_a - 1) * 16 * loaders * k + 2 * k - 128 < (uint64_t)rows * k * 2;
        ok = ok && (rest == 0) == (p.runs == 0) && p.runs <= rest * p.steps();
        ok = ok && (!rest || (size_t)(p.runs + rest) * p.blocks * p.rg * 16 * 512 <= part);
        if (!ok) return printf("%u x %u x %u: %u %u\n", rows, k, n[0], form, pieces), 1;
    }
    return 0;
}
"""


def test_every_plan_of_the_register_gemm_covers_its_tiles(tmp_path):
    src = tmp_path / "rgemm.cpp"
    src.write_text(RGEMM)
    exe = str(tmp_path / "rgemm")
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", os.path.join(ROOT, "ferrite_amd", "csrc"), "-I", os.path.join(ROOT, "include"), str(src), "-o", exe,
                    "-Wl,--unresolved-symbols=ignore-all"], check=True)
    subprocess.run([exe], check=True)


WHOLE = r"""
#include <cstdio>
#include "fe_internal.h"
int main() {
    for (uint32_t upb = 1; upb <= 9; upb++)
        for (uint32_t nb = 1; nb <= 24; nb++)
            for (uint32_t programs = 1; programs <= upb * nb; programs++)
                for (uint32_t per = 1; per <= 2; per++) {
                    const uint32_t units = upb * nb, base = units / programs, rem = units % programs;
                    bool start[9 * 24 + 1] = {};
                    for (uint32_t q = 0; q < programs; q += per) start[q * base + (q < rem ? q : rem)] = true;
                    uint32_t cut = 0;
                    for (uint32_t b = 0; b < nb; b++) {
                        bool c = false;
                        for (uint32_t u = 1; u < upb; u++) c = c || start[b * upb + u];
                        cut += c;
                    }
                    if (cut != fe_gemv_cut_blocks(units, programs, upb, per)) return printf("%u %u %u %u\n", upb, nb, programs, per), 1;
                }
    return 0;
}
"""


def test_which_column_blocks_are_cut(tmp_path):
    src = tmp_path / "whole.cpp"
    src.write_text(WHOLE)
    exe = str(tmp_path / "whole")
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", os.path.join(ROOT, "ferrite_amd", "csrc"), "-I", os.path.join(ROOT, "include"), str(src), "-o", exe,
                    "-Wl,--unresolved-symbols=ignore-all"], check=True)
    subprocess.run([exe], check=True)
