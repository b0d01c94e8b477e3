"""Host arithmetic of the handles' options and dispatch rules (no GPU): the sources compiled here against the built library, which serves what they call elsewhere."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


def run_host(tmp_path, source, main):
    """The lines that `main` prints, compiled behind csrc/`source`."""
    src, exe, lib = tmp_path / "main.cpp", str(tmp_path / "main"), os.path.join(ROOT, "ferrite_amd")
    if not os.path.exists(os.path.join(lib, "libferrite_amd.so")):
        from ferrite_amd import build
        build.build()
    src.write_text(f'#include <cstdio>\n#include "{source}"\n{main}')
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(lib, "csrc"), "-I", os.path.join(ROOT, "include"), "-I", os.path.join(ROCM, "include"),
                    str(src), "-o", exe, "-L", lib, "-lferrite_amd", "-L", os.path.join(ROCM, "lib"), "-lamdhip64", f"-Wl,-rpath,{lib}:{os.path.join(ROCM, 'lib')}"], check=True)
    return subprocess.run([exe], stdout=subprocess.PIPE, text=True, check=True).stdout.splitlines()


@pytest.mark.parametrize("handle,most", [("fp4", 6), ("bf16", 6), ("exl3", 3)])
def test_a_tile_that_does_not_exist_is_refused(tmp_path, handle, most):
    """gemm_tile picks a row of the tables of tiles and kernels: what lies past them is refused and changes nothing."""
    lines = run_host(tmp_path, f"fe_{handle}.cpp", f"""
int main() {{
    fe_{handle}_kernels k;
    auto set = [&](int v) {{
        const int c = fe_{handle}_kernels_set_option(&k, "gemm_tile", v);
        printf("%d %u\\n", c == FE_ERR_ARG ? 1 : c, k.tile.force_tile);
    }};
    for (int v = 0; v <= {most}; v++) set(v);
    for (int v : {{-1, {most} + 1, 1000, (int)0x80000000}}) set(v);
}}
""")
    assert lines == [f"0 {v}" for v in range(most + 1)] + [f"1 {most}"] * 4


def test_asking_for_the_one_launch_block_sets_no_error(tmp_path):
    """Operands that the one launch of gate, up and SwiGLU does not take go another way, which may succeed: the library's last error is left as it was."""
    lines = run_host(tmp_path, "fe_bf16.cpp", """
int main() {
    const fe_bf16_kernels k;
    const fe_devptr_t big = 0x1000000, act = 0x2000000, x = 0x3000000, gate = 0x4000000, up = 0x5000000;
    fe_set_error(1, "kept", "");
    for (uint32_t off : {0u, 4u, 16u}) printf("%d", fe_bf16_gemv_swiglu_takes(&k, big + off, act, x, gate, up, 4, 512, 256, 0, false));
    printf("%d%d\\n", fe_bf16_gemv_swiglu_takes(&k, big, act, x + 8, gate, up, 4, 512, 256, 0, false), fe_bf16_gemv_swiglu_takes(&k, big, act, x, 0, up, 4, 512, 256, 0, false));
    printf("%s\\n", fe_hip_last_error());
    const int code = fe_bf16_linear_forward(&k, nullptr, big, 12, x, 96, gate, 0, 1, 12, 96, 0);
    printf("%d %s\\n", code == FE_ERR_SHAPE, fe_hip_last_error());
}
""")
    assert lines[:2] == ["10100", "kept:  (1)"]
    assert lines[2].startswith("1 fe_bf16_linear_forward: bf16 linear n 12 k 96 (n % 8 == 0, k % 64 == 0)")


def test_what_the_gemm_refuses_stays_refused_at_few_rows(tmp_path):
    """17 to 32 rows that are no decode rows may go through the GEMV, but not where the GEMM they went through before refuses the operands. (No case here reaches a launch.)"""
    lines = run_host(tmp_path, "fe_bf16.cpp", """
int main() {
    fe_bf16_kernels k;
    k.cus = 256;
    const fe_devptr_t y = 0x1000000, x = 0x2000000, w = 0x3000000;
    auto refused = [&](uint32_t n, uint32_t kk, uint32_t lda, uint32_t m, uint32_t dec) {
        return fe_bf16_linear_forward(&k, nullptr, y, n, x, lda, w, 0, m, n, kk, dec) == FE_ERR_UNSUPPORTED;
    };
    printf("%d%d%d\\n", refused(262144, 8192, 8192, 17, 0), refused(524288, 4096, 4096, 32, 0), refused(512, 256, 1u << 27, 17, 0));
    auto pair = [&](uint32_t m, uint32_t inter, uint32_t kk, uint32_t dec, bool over_gemm) {
        return fe_bf16_gemv_swiglu_takes(&k, 0x1000, 0x7000000000000ull, x, w, w, m, inter, kk, dec, over_gemm);
    };
    printf("%d%d%d%d%d\\n", pair(17, 262144, 8192, 0, false), pair(17, 131072, 8192, 0, true), pair(17, 131072, 8192, 0, false), pair(17, 131064, 8192, 0, true), pair(17, 262144, 8192, 17, false));
}
""")
    assert lines == ["111", "00111"]


def test_the_schedule_query_tells_what_a_launch_asks(tmp_path):
    """fe_gemm_schedule_query with the mode its comment names is the 256 x 256 schedule of an NVFP4 launch: mode 0 for up to 2048 rows and more tiles than CUs, else 1."""
    lines = run_host(tmp_path, "fe_fp4.cpp", """
int main() {
    uint32_t asked = 0, differ = 0, stream_k[2] = {};
    for (uint32_t m : {300u, 777u, 1024u, 1536u, 2048u, 2049u, 2304u, 4096u})
        for (uint32_t n : {5120u, 16384u, 17408u, 34816u})
            for (uint32_t k : {2048u, 5120u, 17408u}) {
                const uint32_t tiles = (m + 255) / 256 * ((n + 255) / 256), cus = 256;
                const int mode = m <= 2048 && tiles > cus ? 0 : 1;
                FeGemmTileOptions whole{0, 0, true};
                const FeGemmPlan p = fe_gemm_plan(m, n, k / 64, cus, 1, (size_t)cus * kFeGemmSlotsPerCu * kFeGemmPartBytes, 1, tiles, 8, 1, true, kFeCostNvfp4, whole);
                if (p.tile) continue;
                uint32_t sk, programs, full, splits, run, rem;
                fe_gemm_schedule_query(tiles, k / 64, cus, mode, 1, &sk, &programs, &full, &splits, &run, &rem);
                asked++, stream_k[mode] += sk;
                differ += sk != p.big.stream_k || programs != p.big.programs || full != p.big.args.full_tiles || run != p.big.args.sk_base || rem != p.big.args.sk_rem ||
                          splits != (sk ? 1 : p.big.split.splits);
            }
    printf("%d %u %d %d\\n", asked > 20, differ, stream_k[0] == 0, stream_k[1] > 4);
}
""")
    assert lines == ["1 0 1 1"]


def test_every_wide_form_of_nvfp4_is_one_that_a_rule_or_an_option_reaches(tmp_path):
    """The GEMV of 1..16 rows: whatever the shape, the rows and gemv_cols, the form picked is one that is built, and each that is built is picked somewhere."""
    lines = run_host(tmp_path, "fe_fp4.cpp", """
int main() {
    fe_fp4_kernels K;
    K.cus = 256;
    size_t built = 0, picked = 0, missing = 0;
    bool seen[2][2][4][7] = {};
    for (int q = 0; q < 2; q++)
        for (int e = 0; e < 2; e++)
            for (int i = 0; i < (q ? 3 : 4); i++)
                for (int j = 0; j < 7; j++)
                    if (wide_built(kWideColForms[j], e, q)) built++, (q ? K.wide_q[e][i] : K.wide[e][i])[j] = (fe_function_t)(size_t)(1 + ((q * 2 + e) * 4 + i) * 7 + j);
    fe_fp4_linear l;
    for (uint32_t cols : {0u, 8u, 16u, 24u, 32u, 40u, 48u, 72u, 1000u})
        for (uint32_t n = 128; n < 120000; n += n < 20000 ? 256 : 8192)
            for (uint32_t k : {256u, 1792u, 2048u, 5120u, 17408u})
                for (uint32_t m = 1; m <= 16; m++)
                    for (int q = 0; q < (m <= 8 ? 2 : 1); q++) {
                        l.n = n, l.k = k, K.gemv_cols = cols;
                        const size_t f = (size_t)wide_form(&l, &K, m, q).f;
                        if (!f) missing++;
                        else if (bool &s = (&seen[0][0][0][0])[f - 1]; !s) s = true, picked++;
                    }
    printf("%zu %d\\n", missing, picked == built);
}
""")
    assert lines == ["0 1"]


# (columns, K, rows): us with the quantizer's launch and with every program quantizing all of the activations
QUANT = {(152064, 1280, 8): (35.7, 48.4), (98304, 1280, 8): (25.4, 33.2), (65536, 2560, 4): (23.3, 27.5), (152064, 5120, 1): (74.6, 82.3), (65536, 5120, 2): (34.7, 38.6),
         (16384, 1280, 8): (7.8, 8.6), (28672, 1280, 8): (11.8, 13.5), (24576, 1280, 8): (10.9, 13.7), (1024, 2560, 8): (6.4, 7.1), (5120, 2560, 8): (7.9, 8.5),
         (5120, 5120, 1): (8.5, 6.7), (17408, 5120, 1): (13.9, 12.5), (34816, 5120, 2): (22.2, 21.1), (5120, 17408, 1): (14.6, 14.0), (24576, 512, 8): (8.4, 5.4),
         (28672, 1024, 2): (9.6, 7.1), (4096, 4096, 5): (7.2, 6.9), (40960, 5120, 1): (26.2, 25.2), (1024, 1024, 8): (5.1, 4.1)}


def test_programs_quantize_only_where_that_was_timed_faster(tmp_path):
    calls = ", ".join("{%du, %du, %du}" % c for c in QUANT)
    lines = run_host(tmp_path, "fe_fp4.cpp", f"""
int main() {{
    fe_fp4_kernels K;
    K.cus = 256;
    fe_fp4_linear l;
    fe_fp4_workspace ws;
    const uint32_t calls[][3] = {{{calls}}};
    for (auto &c : calls) {{
        l.n = c[0], l.k = c[1];
        printf("%d\\n", fp4_quants_itself(&l, &K, &ws, 0x1000000, l.n, 0x2000000000ull, l.k, c[2]));
    }}
}}
""")
    assert [int(v) for v in lines] == [int(inside < launch) for launch, inside in QUANT.values()]


# (form, rows, columns, K): us of a small tile (128 x 256 or 128 x 128) and of the lower one that the heights' estimate names in its place
LOWER = {("nvfp4", 636, 5248, 256): (9.2, 13.1), ("nvfp4", 449, 768, 1536): (14.9, 18.3), ("nvfp4", 163, 256, 2560): (12.1, 14.7),
         ("fp8", 315, 11136, 256): (9.1, 11.6), ("fp8", 584, 6784, 512): (11.2, 13.8), ("fp8", 180, 1024, 4864): (15.8, 18.5),
         ("bf16", 210, 256, 1536): (7.8, 10.3), ("bf16", 228, 25984, 256): (9.4, 10.4), ("bf16", 79, 512, 1792): (8.2, 9.7),
         ("nvfp4", 1686, 5888, 4096): (102.1, 83.7), ("nvfp4", 774, 37248, 2816): (188.2, 162.4), ("fp8", 868, 9856, 3584): (51.4, 43.4),
         ("bf16", 1423, 5888, 2048): (47.3, 37.6), ("bf16", 721, 25984, 1280): (67.4, 57.7),
         ("bf16", 1231, 1024, 8960): (36.4, 43.2), ("bf16", 1303, 768, 15104): (41.9, 52.6), ("bf16", 864, 1792, 16384): (56.8, 89.7), ("bf16", 424, 1792, 7936): (27.2, 33.0),
         ("bf16", 764, 2304, 8704): (40.8, 48.0), ("fp8", 711, 33536, 2048): (65.2, 70.8), ("fp8", 1516, 28672, 1792): (92.8, 102.6), ("nvfp4", 1313, 11008, 768): (33.5, 37.9),
         ("bf16", 1035, 8192, 1792): (42.1, 33.1), ("bf16", 1041, 4608, 7680): (88.7, 73.5), ("bf16", 469, 16640, 1280): (33.7, 25.5), ("fp8", 1253, 7168, 2560): (38.2, 32.3),
         ("nvfp4", 1159, 6912, 3328): (72.2, 58.6), ("nvfp4", 1528, 3840, 9216): (119.5, 98.4),
         ("bf16", 365, 38400, 5632): (179.6, 162.4), ("bf16", 195, 33280, 3840): (80.6, 72.5), ("nvfp4", 839, 25600, 1792): (87.7, 74.5), ("nvfp4", 840, 25856, 3328): (148.2, 130.3),
         ("front", 147, 512, 1024): (19.5, 15.0), ("front", 91, 768, 1024): (19.2, 14.5), ("front", 82, 1024, 1280): (16.7, 15.0), ("front", 165, 1024, 1024): (19.9, 16.2)}


def test_a_lower_tile_takes_a_small_ones_place_where_that_was_timed_faster(tmp_path):
    calls = ", ".join('{"%s", %d, %d, %d}' % c for c in LOWER)
    lines = run_host(tmp_path, "fe_fp4.cpp", f"""
int main() {{
    struct {{ const char *form; uint32_t m, n, k; }} calls[] = {{{calls}}};
    for (auto &c : calls) {{
        const bool f8 = c.form[0] == 'f' && c.form[1] == 'p', front = c.form[0] == 'f' && !f8, bf = c.form[0] == 'b';
        const FeGemmPlan p = fe_gemm_plan(c.m, c.n, c.k / (f8 ? 128 : 64), 256, 1, (size_t)512 * kFeGemmPartBytes, 1, 8192, 8, bf || front ? 0 : 1, !f8 && !bf,
                                          f8 ? kFeCostFp8 : bf ? kFeCostBf16 : kFeCostNvfp4, FeGemmTileOptions{{0, 0, true, front}});
        printf("%d\\n", p.tile >= 3 ? 1 : p.tile ? 0 : 2);
    }}
}}
""")
    assert [int(v) for v in lines] == [int(lower < small) for small, lower in LOWER.values()]


# (columns, K, rows): us of the FP8 GEMV and of the GEMM
FP8 = {(11776, 12288, 58): (44.6, 36.7), (34176, 3840, 53): (40.2, 31.1), (21120, 512, 49): (12.5, 9.0), (35328, 2304, 61): (30.6, 25.4),
       (26368, 512, 27): (10.7, 8.9), (37632, 384, 59): (16.6, 10.5), (27904, 256, 55): (12.0, 7.9), (2048, 19328, 58): (25.7, 22.0), (128, 2048, 52): (6.2, 11.5),
       (1024, 1024, 43): (5.1, 10.2), (384, 640, 15): (4.5, 7.4), (1152, 10752, 17): (9.3, 14.8), (1024, 896, 20): (4.7, 8.8), (768, 1536, 53): (5.8, 12.4),
       (768, 512, 53): (5.3, 8.0), (1920, 2432, 58): (7.3, 13.6), (3328, 49664, 27): (42.3, 32.7), (46336, 5376, 28): (47.1, 39.5), (3200, 63744, 26): (51.0, 39.7),
       (38272, 3840, 32): (31.0, 26.1), (4480, 17664, 18): (19.2, 23.4), (4480, 17664, 9): (16.4, 23.2)}


def test_fp8_rows_take_the_gemv_where_that_was_timed_faster(tmp_path):
    calls = ", ".join("{%du, %du, %du}" % c for c in FP8)
    lines = run_host(tmp_path, "fe_fp4.cpp", f"""
int main() {{
    const uint32_t calls[][3] = {{{calls}}};
    for (auto &c : calls) {{
        const uint32_t n = c[0], k = c[1], m = c[2];
        const FeGemmPlan p = fe_gemm_plan(m, n, k / 128, 256, 1, (size_t)512 * kFeGemmPartBytes, 1, 8192, 8, 1, false, kFeCostFp8, FeGemmTileOptions{{0, 0, true}});
        printf("%d\\n", fe_gemv_ahead(kFeGemvFp8, m, n, k, k / 128, 256, 4, p));
    }}
}}
""")
    assert [int(v) for v in lines] == [int(gemv < gemm) for gemv, gemm in FP8.values()]


# SwiGLU fronts (columns of gate and up together, K, rows): us of the GEMV and of the GEMM
SWIGLU = {(512, 4992, 45): (18.4, 13.8), (1536, 4480, 38): (19.1, 14.6), (4864, 4224, 40): (23.1, 18.7), (512, 2176, 38): (14.4, 12.4), (1280, 8832, 35): (20.6, 18.5),
          (2304, 17536, 45): (30.5, 28.0), (6912, 3200, 48): (21.8, 19.3), (512, 3712, 33): (17.7, 12.8), (40192, 512, 46): (15.0, 21.6), (29184, 2688, 20): (19.7, 29.6),
          (8704, 4096, 20): (15.4, 22.8), (1536, 1152, 28): (11.2, 17.8), (13824, 1024, 18): (12.1, 17.8), (35072, 9088, 24): (66.8, 114.9), (8960, 256, 20): (8.0, 11.7),
          (512, 4992, 12): (10.4, 13.1)}  # up to 16 rows in any case


def test_swiglu_fronts_take_the_gemv_where_that_was_timed_faster(tmp_path):
    calls = ", ".join("{%du, %du, %du}" % c for c in SWIGLU)
    lines = run_host(tmp_path, "fe_fp4.cpp", f"""
int main() {{
    fe_fp4_kernels K;
    K.cus = 256;
    fe_fp4_linear l;
    fe_fp4_workspace ws;
    ws.part.bytes = (size_t)512 * kFeGemmPartBytes;
    const uint32_t calls[][3] = {{{calls}}};
    for (auto &c : calls) {{
        l.n = c[0], l.k = c[1], l.w_sr = 32;
        const FeGemmPlan p = fe_gemm_plan(c[2], l.n, l.k / 64, 256, 1, ws.part.bytes, 1, 8192, 8, 0, true, kFeCostNvfp4, K.tile);
        printf("%d\\n", swiglu_takes_gemv(&l, &K, c[2], gemv_splits(&K, &ws, l.n, l.k), p));
    }}
}}
""")
    assert [int(v) for v in lines] == [int(gemv < gemm) for gemv, gemm in SWIGLU.values()]


# bf16 linears and gate|up fronts (columns, K, rows): us of the GEMV and of the GEMM
BF16 = {(61728, 256, 31): (15.8, 7.6), (55304, 256, 27): (14.5, 7.2), (24672, 512, 29): (9.8, 6.5), (53672, 1536, 31): (33.4, 27.7), (26952, 512, 17): (9.1, 6.6), (48152, 1280, 24): (26.2, 21.7),
        (24936, 256, 22): (7.6, 4.9), (3520, 18432, 32): (33.7, 27.9), (104, 2304, 21): (3.8, 7.9), (12312, 768, 29): (5.8, 7.6), (264, 4608, 23): (6.3, 8.8), (8368, 512, 30): (4.0, 6.1),
        (2488, 2816, 23): (6.0, 9.8), (144, 1280, 17): (3.2, 8.8), (5344, 1024, 20): (4.1, 8.5), (80048, 4096, 28): (114.0, 144.5), (28360, 6144, 22): (61.8, 84.9)}
BF16_PAIR = {(28480, 256, 22): (18.8, 7.8), (15168, 256, 21): (9.8, 5.6), (27072, 1280, 20): (29.8, 24.1), (64, 18432, 26): (36.4, 17.4), (320, 10752, 20): (22.4, 12.9), (640, 14336, 22): (32.4, 19.2),
             (384, 6400, 24): (15.0, 10.5), (640, 512, 20): (4.4, 6.2), (320, 1280, 21): (4.9, 8.1), (3072, 512, 30): (3.9, 6.8), (1280, 2560, 20): (7.0, 9.5), (2112, 1280, 20): (6.7, 10.3)}


def test_bf16_rows_take_the_gemv_where_that_was_timed_faster(tmp_path):
    calls = ", ".join("{%du, %du, %du, %d}" % (*c, pair) for t, pair in ((BF16, 0), (BF16_PAIR, 1)) for c in t)
    lines = run_host(tmp_path, "fe_bf16.cpp", f"""
int main() {{
    struct {{ uint32_t n, k, m; int pair; }} calls[] = {{{calls}}};
    for (auto &c : calls) {{
        const FeGemmPlan p = fe_gemm_plan(c.m, c.pair ? 2 * c.n : c.n, c.k / 64, 256, 1, (size_t)512 * kFeGemmPartBytes, 0, 0, 8, 0, false, kFeCostBf16, FeGemmTileOptions{{0, 0, true}});
        printf("%d\\n", fe_gemv_ahead(c.pair ? kFeGemvBf16Pair : kFeGemvBf16, c.m, c.n, c.k, c.k / 64, 256, 2, p, (c.pair ? 4.0f : 2.0f) * c.n * c.k));
    }}
}}
""")
    assert [int(v) for v in lines] == [int(gemv < gemm) for t in (BF16, BF16_PAIR) for gemv, gemm in t.values()]


# NVFP4 (columns, K, rows): us of the GEMV in two passes and of the GEMM
NVFP4_PASSES = {(768, 68864, 62): (53.5, 66.4), (256, 74496, 58): (53.4, 70.0), (256, 59136, 53): (45.5, 56.7), (384, 53248, 51): (42.9, 51.9), (4736, 20224, 53): (45.5, 33.6),
                (3712, 35328, 59): (55.5, 42.3), (34816, 5120, 64): (83.0, 63.0), (5120, 17408, 64): (43.0, 30.0), (2048, 6144, 64): (27.0, 14.0)}


def test_nvfp4_takes_two_passes_where_that_was_timed_faster(tmp_path):
    calls = ", ".join("{%du, %du, %du}" % c for c in NVFP4_PASSES)
    lines = run_host(tmp_path, "fe_fp4.cpp", f"""
int main() {{
    fe_fp4_kernels K;
    fe_fp4_linear l;
    const uint32_t calls[][3] = {{{calls}}};
    for (auto &c : calls) {{
        l.n = c[0], l.k = c[1];
        printf("%d\\n", takes_gemv(&l, &K, c[2], true));
    }}
}}
""")
    assert [int(v) for v in lines] == [int(gemv < gemm) for gemv, gemm in NVFP4_PASSES.values()]
