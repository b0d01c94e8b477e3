"""The choice of a prefill GEMM's row tiles where lower ones exist (fe_gemm_plan with `low`, host arithmetic), compiled here."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
MAIN = r"""
#include <cstdio>
#include <cstdlib>
#include <string>
#include "fe_internal.h"
int main(int argc, char **argv) {
    for (int i = 1; i + 4 < argc; i += 5) {
        const std::string form = argv[i];
        const uint32_t m = atoi(argv[i + 1]), n = atoi(argv[i + 2]), k = atoi(argv[i + 3]), slots = atoi(argv[i + 4]);
        const bool f8 = form == "fp8", bf = form == "bf16";
        const FeGemmCost &c = form == "nvfp4" ? kFeCostNvfp4 : f8 ? kFeCostFp8 : kFeCostBf16;
        const uint32_t ktiles = k / (f8 ? 128 : 64);
        const FeGemmPlan p = fe_gemm_plan(m, n, ktiles, 256, 1, (size_t)slots * kFeGemmPartBytes, 1, 8192, 8, bf ? 0 : 1, !f8 && !bf, c, FeGemmTileOptions{0, 0, true});
        uint32_t pieces = 0, whole = 0, each = 1;
        if (p.tile == 1 || p.tile == 2) pieces = p.splits > 1 ? p.tiles * p.splits : 0, whole = p.splits > 1 ? 0 : p.tiles, each = p.splits;
        else if (!p.big.stream_k) pieces = p.big.split.cut() * p.big.split.splits, whole = p.big.split.full, each = p.big.split.splits;
        printf("%u %d %u %u %u %zu\n", p.tile, (int)p.big.stream_k, whole, pieces, each, (size_t)pieces * kFeGemmTileM[p.tile] * kFeGemmTileN[p.tile] * 4);
    }
}
"""


def plans(tmp_path, calls):
    src, exe = tmp_path / "plan.cpp", str(tmp_path / "plan")
    src.write_text(MAIN)
    # (the header's device buffers refer to the library, which the plan does not touch)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", os.path.join(ROOT, "ferrite_amd", "csrc"), "-I", os.path.join(ROOT, "include"), str(src), "-o", exe,
                    "-Wl,--unresolved-symbols=ignore-all"], check=True)
    out = subprocess.run([exe, *(str(v) for c in calls for v in c)], stdout=subprocess.PIPE, text=True, check=True).stdout.splitlines()
    return [tuple(int(v) for v in line.split()) for line in out]


# (form, rows, columns, K): tile (3, 4, 5: 224, 192, 160 rows), stream-K; us of the taken form and of the nearest other
TIMED = {
    ("nvfp4", 400, 34816, 5120): (3, 0),   # 130, stream-K 144
    ("nvfp4", 200, 34816, 5120): (0, 1),   # 94, one piece 102
    ("nvfp4", 2048, 5120, 17408): (0, 1),  # 265, one piece 277
    ("nvfp4", 160, 34816, 5120): (5, 0),   # 76, 256 rows 93
    ("nvfp4", 320, 34816, 5120): (5, 0),   # 102, 256 rows 126
    ("nvfp4", 1024, 34816, 5120): (0, 0),  # 267, stream-K 277
    # FP8: where every lower tile would be cut, and with short K and a ratio near 1, the small tiles
    ("fp8", 1100, 5120, 17408): (1, 0),   # 88.6, 192 rows cut in two 91.7
    ("fp8", 1216, 5120, 17408): (1, 0),   # 92.7, 224 rows cut in two 103.6
    ("fp8", 1216, 2048, 8192): (1, 0),    # 28.8, 160 rows cut in four 30.5
    ("fp8", 1536, 2048, 8192): (1, 0),    # 32.9, 160 rows cut in three 35.4
    ("fp8", 512, 5120, 6144): (1, 0),     # 25.0, 160 rows cut in three 28.5
    ("fp8", 1024, 3072, 9216): (1, 0),    # 35.0, 160 rows cut in three 38.0
    ("fp8", 1024, 8192, 2048): (2, 0),    # 19.7, 160 rows whole 20.7
    # and the lower tiles where they are ahead
    ("fp8", 420, 17408, 5120): (5, 0),    # 38.6, 128 rows 46.7
    ("fp8", 250, 34816, 5120): (5, 0),    # a round and 16 tiles cut in seven 66.5, 128 rows 82.8
    ("fp8", 155, 18944, 8448): (5, 0),    # one row tile, cut in three 45.9, 128 rows 53.5
    ("fp8", 1100, 8192, 2048): (5, 0),    # 21.0, 128 x 128 23.7
    ("fp8", 1300, 17408, 5120): (4, 0),   # 93.4, 128 rows 103.3
    ("fp8", 777, 5120, 17408): (3, 0),    # each cut in three 74.2, 256 rows so 76.4
}


def test_the_height_that_was_timed_faster(tmp_path):
    for key, got in zip(TIMED, plans(tmp_path, [(*k, 512) for k in TIMED])):
        assert got[:2] == TIMED[key], (key, got)


def test_every_choice_covers_the_tiles_and_fits_its_slots(tmp_path):
    height, width = (256, 128, 128, 224, 192, 160), (256, 256, 128, 256, 256, 256)
    calls = [(f, m, n, k, s) for f in ("nvfp4", "fp8", "bf16") for m in (65, 130, 161, 225, 390, 777, 1025, 2048, 2049)
             for n, k in ((128, 256), (1024, 2816), (5120, 17408), (34816, 5120), (8704, 5120)) for s in (0, 1, 40, 512)]
    for call, (tile, sk, whole, pieces, each, used) in zip(calls, plans(tmp_path, calls)):
        f, m, n, k, s = call
        assert used <= s * 256 * 1024 and (m <= 2048 or tile < 3), call
        if not sk:
            assert whole + pieces // each == -(-m // height[tile]) * -(-n // width[tile]), call
        else:
            assert tile == 0 and not (f == "nvfp4" and m <= 2048 and -(-m // 256) * -(-n // 256) > 256), call
