// fe_bf16: host side of the plain bf16 linear (see include/fe_bf16.h). Follows crates/fe-model/src/model.rs:310-345;
// the kernels are ferrite_amd/csrc/kernels/k_bf16.hip.
#include "fe_bf16.h"

#include <cstdio>
#include <cstdlib>

#include "fe_exl3.h"  // error codes
#include <string>

#include "fe_internal.h"

namespace {
// dynamic LDS by form (256 x 256, unused, 128 x 256, 128 x 128, 224, 192, 160 x 256): the k tiles in flight, three of W and two of A (128 x 256:
// three), A in whole loads of 64 rows
constexpr uint32_t kGemmLds[kFeGemmForms] = {160 * 1024, 0, 144 * 1024, 80 * 1024, 160 * 1024, 144 * 1024, 144 * 1024};
constexpr uint32_t kGemmThreads = 512;
constexpr uint32_t kTileM = 256;                         // rows of the largest output tile
constexpr uint32_t kGemvRows = 8;                        // rows of one fe_bf16_gemv call (model.rs:326)
constexpr uint32_t kGemvPass = 64;                       // rows of one pass over the weights
constexpr uint32_t kSmallBatch = 16;                     // X3_ROWS: batches up to here are decode rows (model.rs:172)
}  // namespace

struct fe_bf16_kernels {
    fe_module_t module = nullptr;
    fe_function_t gemm[kFeGemmForms] = {}, reduce[kFeGemmTiles] = {}, swiglu[kFeGemmForms] = {}, swiglu_reduce[kFeGemmTiles] = {};  // by form; by tile (fe_gemm_launch)
    fe_function_t interleave = nullptr;
    fe_function_t gemv[5][7] = {}, gemv_swiglu[5][7] = {};  // [kGemvRowForms][kGemvColForms]
    uint32_t cus = 0;
    FeBuf part;
    // Switches, read from the environment once at load (fe_bf16_kernels_set_option changes them afterwards)
    int32_t nc = -1;           // columns a GEMV program takes, rounded up to 8, 16, .. 48, 72; -1 = by the shape (FE_BF16_NC)
    int32_t raster_group = -1; // raster group of the GEMM; -1 = by the shape (FE_BF16_GROUP)
    uint32_t gemm_splits = 8;  // most pieces a cut output tile takes (FE_GEMM_SPLITS; 1: never cut)
    FeGemmTileOptions tile{0, 0, true};  // "gemm_tile", "gemm_pieces"
};

// Raster of the GEMM's output tiles (gemm_raster). Weights at least as large as the activations: column tiles are dealt
// to the XCDs (group 0), each weight panel through one L2, the smaller activations through all of them; else row tiles
// in groups of 8. Measured at M = 2048 in alternation with groups of 8: 5120 x 17408 323 against 344 us,
// 17408 x 5120 342 against 365 us, 5120 x 34816 618 against 648 us.
static uint32_t bf16_raster_group(uint32_t m, uint32_t n, uint32_t k, uint32_t tiles_m) {
    (void)k;
    return n >= m ? 0 : tiles_m < 8 ? tiles_m : 8;
}

// Why a linear's operands are refused (0: they are not). Sets no error: rules of a dispatch ask it, too.
static int refusal(fe_devptr_t y, uint32_t ldy, fe_devptr_t x, uint32_t lda, fe_devptr_t w, fe_devptr_t res, uint32_t n, uint32_t k, const char **why) {
    if (!y || !x || !w) return *why = "null pointer", FE_ERR_ARG;
    if (!n || !k || n % 8 || k % 64) return *why = "n % 8 == 0, k % 64 == 0", FE_ERR_SHAPE;
    if (lda % 8 || lda < k || x % 16 || w % 16) return *why = "x / w rows must be 16-byte aligned, lda >= k", FE_ERR_ARG;
    if (ldy % 4 || ldy < n || y % 8 || (res && res % 8)) return *why = "y / res rows must be 8-byte aligned, ldy >= n", FE_ERR_ARG;
    return 0;
}
static int check(const char *fn, fe_devptr_t y, uint32_t ldy, fe_devptr_t x, uint32_t lda, fe_devptr_t w, fe_devptr_t res,
                 uint32_t n, uint32_t k) {
    const char *why = nullptr;
    const int code = refusal(y, ldy, x, lda, w, res, n, k, &why);
    if (!code) return 0;
    char msg[120];
    if (code == FE_ERR_SHAPE) snprintf(msg, sizeof msg, "bf16 linear n %u k %u (%s)", n, k, why);
    return fe_set_error(code, fn, code == FE_ERR_SHAPE ? msg : why);
}

// Operands of 4 GB and more the GEMM refuses, also where few rows could go another way.
static bool gemm_reaches(uint32_t m, uint32_t n, uint32_t k, uint32_t lda) { return (uint64_t)m * lda * 2 < (1ull << 32) && (uint64_t)n * k * 2 < (1ull << 32); }
static FeGemmPlan gemm_plan(const fe_bf16_kernels *kern, uint32_t m, uint32_t n, uint32_t k) {
    return fe_gemm_plan(m, n, k / 64, kern->cus, kern->part.p, kern->part.bytes, 0, 0, kern->gemm_splits, 0, false, kFeCostBf16, kern->tile);
}
// Whether all of a call's rows go through the GEMV: a batch of decode rows, or 17..32 rows where its one read of the weights is ahead of the GEMM's
// tiles (kFeGemvBf16).
static bool rows_take_gemv(const fe_bf16_kernels *kern, uint32_t m, uint32_t n, uint32_t k, uint32_t lda, uint32_t dec) {
    if (m <= kSmallBatch || dec >= m) return true;
    if (m > 32 || k % 256 || !gemm_reaches(m - dec, n, k, lda)) return false;
    return fe_gemv_ahead(kFeGemvBf16, m, n, k, k / 64, std::max(kern->cus, 1u), 2, gemm_plan(kern, m - dec, n, k), (float)n * (float)k * 2.0f, dec);
}

bool fe_bf16_gemv_swiglu_takes(const fe_bf16_kernels *kern, fe_devptr_t big, fe_devptr_t act, fe_devptr_t x, fe_devptr_t gate, fe_devptr_t up, uint32_t m, uint32_t inter,
                               uint32_t k, uint32_t dec, bool over_gemm) {
    if (!kern || !m || m > kGemvPass || !inter || !k || inter % 8 || k % 256 || (uint64_t)m * k * 2 >= (1ull << 32)) return false;
    // (against the GEMM with SwiGLU: kFeGemvBf16Pair. Against gate, up and fe_silu_mul, where there are no such weights, it is ahead wherever those
    // go through the GEMV: 5120 x 8704 at 26 / 32 rows 63.0 -> 58.0, 63.9 -> 58.6, 5120 x 6144 at 30 53.0 -> 48.4, 7168 x 2048 at 25 32.7 -> 28.0)
    if (over_gemm && m > kSmallBatch && dec < m) {
        if (m > 32 || !gemm_reaches(m - dec, 2 * inter, k, k)) return false;
        if (!fe_gemv_ahead(kFeGemvBf16Pair, m, inter, k, k / 64, std::max(kern->cus, 1u), 2, gemm_plan(kern, m - dec, 2 * inter, k), (float)inter * (float)k * 4.0f, dec)) return false;
    } else if (!rows_take_gemv(kern, m, inter, k, k, dec)) {
        return false;
    }
    const char *why;
    if (refusal(big, inter, x, k, gate, 0, inter, k, &why) || refusal(big, inter, x, k, up, 0, inter, k, &why)) return false;
    // programs that are done write act while others read x and the weights
    const uint64_t bytes = (uint64_t)m * inter * 2, weights = (uint64_t)inter * k * 2;
    auto apart = [&](fe_devptr_t p, uint64_t size) { return act + bytes <= p || p + size <= act; };
    return act % 4 == 0 && apart(x, (uint64_t)m * k * 2) && apart(gate, weights) && apart(up, weights);
}

int fe_bf16_gemv_swiglu(const fe_bf16_kernels *kern, fe_stream_t s, fe_devptr_t act, fe_devptr_t x, fe_devptr_t gate, fe_devptr_t up, uint32_t m, uint32_t inter, uint32_t k) {
    const uint32_t form = gemv_row_form(m), xo = kGemvRowForms[form];
    const uint32_t cols = gemv_cols(m, inter, k, xo, std::max(kern->cus, 1u), kern->nc), co = kGemvColForms[cols];
    uint32_t pc = gemv_even(inter, 8 * co, std::max(kern->cus, 1u), 2, kern->nc > 0 || m <= 2);
    void *args[] = {&act, &x, &gate, &up, &m, &inter, &k, &k, &pc};
    return fe_hip_launch(kern->gemv_swiglu[form][cols], (inter + pc - 1) / pc, 1, 1, 256, 1, 1, gemv_lds(xo, co), s, args);
}

extern "C" {

int fe_bf16_kernels_load(fe_bf16_kernels **out) {
    if (!out) return fe_set_error(FE_ERR_ARG, "fe_bf16_kernels_load", "null out");
    auto *k = new fe_bf16_kernels;
    int c = fe_load_module(&k->module, "FE_BF16_HSACO", fe_k_bf16_hsaco, fe_k_bf16_hsaco_end);
    for (uint32_t tile = 0; tile < kFeGemmTiles && !c; tile++) {
        static const char *suffix[] = {"", "_s1", "_s2", "_h7", "_h6", "_h5"};
        const uint32_t form = tile ? tile + 1 : 0;
        const std::string s = suffix[tile];
        c = fe_hip_module_get_function(&k->gemm[form], k->module, ("fe_gemm_bf16" + s).c_str());
        if (!c) c = fe_hip_func_set_max_dyn_lds(k->gemm[form], kGemmLds[form]);
        if (!c) c = fe_hip_module_get_function(&k->swiglu[form], k->module, ("fe_gemm_bf16_swiglu" + s).c_str());
        if (!c) c = fe_hip_func_set_max_dyn_lds(k->swiglu[form], kGemmLds[form]);
        if (!c) c = fe_hip_module_get_function(&k->reduce[tile], k->module, ("fe_gemm_bf16_reduce" + s).c_str());
        if (!c) c = fe_hip_module_get_function(&k->swiglu_reduce[tile], k->module, ("fe_gemm_bf16_swiglu_reduce" + s).c_str());
    }
    if (!c) c = fe_hip_module_get_function(&k->interleave, k->module, "fe_interleave_gu");
    for (uint32_t i = 0; i < 5 && !c; i++)
        for (uint32_t j = 0; j < 7 && !c; j++) {
            const uint32_t xo = kGemvRowForms[i], co = kGemvColForms[j];
            if (!gemv_form(xo, co)) continue;
            for (int pair = 0; pair < 2 && !c; pair++) {
                char nm[40];
                snprintf(nm, sizeof nm, "fe_gemv_bf16%s_r%u_c%u", pair ? "_swiglu" : "", xo, co);
                fe_function_t &f = (pair ? k->gemv_swiglu : k->gemv)[i][j];
                c = fe_hip_module_get_function(&f, k->module, nm);
                if (!c) c = fe_hip_func_set_max_dyn_lds(f, gemv_lds(xo, co));
            }
        }
    int cus = 0;
    if (!c) c = fe_hip_cu_count(&cus);
    k->cus = (uint32_t)cus;
    if (const char *e = getenv("FE_BF16_NC")) k->nc = atoi(e);
    if (const char *e = getenv("FE_BF16_GROUP")) k->raster_group = atoi(e);
    if (const char *e = getenv("FE_GEMM_SPLITS")) k->gemm_splits = (uint32_t)atoi(e);
    if (!c) c = k->part.alloc((size_t)kFeGemmSlotsPerCu * k->cus * kFeGemmPartBytes);
    if (c) {
        fe_bf16_kernels_destroy(k);
        return c;
    }
    *out = k;
    return 0;
}

int fe_bf16_kernels_destroy(fe_bf16_kernels *k) {
    if (!k) return 0;
    k->part.release();
    if (k->module) fe_hip_module_unload(k->module);
    delete k;
    return 0;
}

int fe_bf16_kernels_set_option(fe_bf16_kernels *k, const char *name, int32_t value) {
    if (!k || !name) return fe_set_error(FE_ERR_ARG, "fe_bf16_kernels_set_option", "null argument");
    const std::string nm = name;
    if (nm == "nc") k->nc = value;
    else if (nm == "raster_group") k->raster_group = value;
    else if (nm == "gemm_splits") k->gemm_splits = (uint32_t)value;
    else if (nm == "gemm_tile") return k->tile.set(value) ? 0 : fe_set_error(FE_ERR_ARG, "fe_bf16_kernels_set_option", "gemm_tile: 0..6");
    else if (nm == "gemm_pieces") k->tile.force_pieces = (uint32_t)value;
    else return fe_set_error(FE_ERR_ARG, "fe_bf16_kernels_set_option", name);
    return 0;
}

// One pass over the weights, operands checked, m in 1..kGemvPass.
static int launch_gemv(const fe_bf16_kernels *kern, fe_stream_t s, fe_devptr_t y, uint32_t ldy, fe_devptr_t x, uint32_t lda,
                       fe_devptr_t w, fe_devptr_t res, uint32_t m, uint32_t n, uint32_t k) {
    if (m > 1 && (uint64_t)m * lda * 2 >= (1ull << 32)) {  // rows that lie further apart than an offset reaches
        for (uint32_t r = 0; r < m; r++)
            FE_TRY(launch_gemv(kern, s, y + (size_t)r * ldy * 2, ldy, x + (size_t)r * lda * 2, lda, w, res ? res + (size_t)r * ldy * 2 : 0, 1, n, k));
        return 0;
    }
    const uint32_t form = gemv_row_form(m), xo = kGemvRowForms[form];
    const uint32_t cols = gemv_cols(m, n, k, xo, std::max(kern->cus, 1u), kern->nc), co = kGemvColForms[cols];
    uint32_t pc = gemv_even(n, 8 * co, std::max(kern->cus, 1u), 2, kern->nc > 0 || m <= 2);
    void *args[] = {&y, &x, &w, &res, &m, &n, &k, &lda, &ldy, &pc};
    return fe_hip_launch(kern->gemv[form][cols], (n + pc - 1) / pc, 1, 1, 256, 1, 1, gemv_lds(xo, co), s, args);
}

int fe_bf16_gemv(const fe_bf16_kernels *kern, fe_stream_t s, fe_devptr_t y, uint32_t ldy, fe_devptr_t x, uint32_t lda,
                 fe_devptr_t w, fe_devptr_t res, uint32_t m, uint32_t n, uint32_t k) {
    const char *fn = "fe_bf16_gemv";
    if (!kern) return fe_set_error(FE_ERR_ARG, fn, "null kernels");
    if (m == 0) return 0;
    if (m > kGemvRows) return fe_set_error(FE_ERR_ARG, fn, "at most 8 rows a call");
    FE_TRY(check(fn, y, ldy, x, lda, w, res, n, k));
    return launch_gemv(kern, s, y, ldy, x, lda, w, res, m, n, k);
}

int fe_bf16_gemm(const fe_bf16_kernels *kern, fe_stream_t s, fe_devptr_t y, uint32_t ldy, fe_devptr_t x, uint32_t lda,
                 fe_devptr_t w, fe_devptr_t res, uint32_t m, uint32_t n, uint32_t k) {
    const char *fn = "fe_bf16_gemm";
    if (!kern) return fe_set_error(FE_ERR_ARG, fn, "null kernels");
    if (m == 0) return 0;
    FE_TRY(check(fn, y, ldy, x, lda, w, res, n, k));
    if (!gemm_reaches(m, n, k, lda)) return fe_set_error(FE_ERR_UNSUPPORTED, fn, "operand of 4 GB or more");
    const uint32_t tiles_m = (m + kTileM - 1) / kTileM;
    uint32_t group = bf16_raster_group(m, n, k, tiles_m);
    if (kern->raster_group >= 0) group = (uint32_t)kern->raster_group;
    if (group > tiles_m) group = tiles_m;
    const FeGemmPlan plan = gemm_plan(kern, m, n, k);
    return fe_gemm_launch(
        plan,
        [&](uint32_t form, uint32_t programs, FeGemmSchedArgs sched) {
            void *args[] = {&y, &x, &w, &res, &m, &n, &k, &lda, &ldy, &group, &sched};
            return fe_hip_launch(kern->gemm[form], programs, 1, 1, kGemmThreads, 1, 1, kGemmLds[form], s, args);
        },
        [&](uint32_t tile, uint32_t grid, uint32_t first, uint32_t splits) {
            fe_devptr_t part = kern->part.p;
            void *args[] = {&y, &part, &res, &m, &n, &ldy, &group, &first, &splits};
            return fe_hip_launch(kern->reduce[tile], grid, 1, 1, fe_reduce_threads(tile), 1, 1, 0, s, args);
        });
}

int fe_bf16_interleave_gu(const fe_bf16_kernels *kern, fe_stream_t s, fe_devptr_t dst, fe_devptr_t gate, fe_devptr_t up,
                          uint32_t inter, uint32_t k) {
    const char *fn = "fe_bf16_interleave_gu";
    if (!kern || !dst || !gate || !up) return fe_set_error(FE_ERR_ARG, fn, "null argument");
    if (!inter || !k || inter % 8 || k % 8 || dst % 16 || gate % 16 || up % 16)
        return fe_set_error(FE_ERR_SHAPE, fn, "inter % 8 == 0, k % 8 == 0, 16-byte aligned rows");
    void *args[] = {&dst, &gate, &up, &k};
    return fe_hip_launch(kern->interleave, 2 * inter, 1, 1, 256, 1, 1, 0, s, args);
}

int fe_bf16_gemm_swiglu(const fe_bf16_kernels *kern, fe_stream_t s, fe_devptr_t act, fe_devptr_t x, uint32_t lda,
                        fe_devptr_t w, uint32_t m, uint32_t inter, uint32_t k) {
    const char *fn = "fe_bf16_gemm_swiglu";
    if (!kern) return fe_set_error(FE_ERR_ARG, fn, "null kernels");
    if (m == 0) return 0;
    uint32_t n = 2 * inter;
    FE_TRY(check(fn, act, n, x, lda, w, 0, n, k));  // act rows have stride inter = n / 2, a multiple of 8
    if (n % 16) return fe_set_error(FE_ERR_SHAPE, fn, "inter % 8 == 0");
    if (!gemm_reaches(m, n, k, lda)) return fe_set_error(FE_ERR_UNSUPPORTED, fn, "operand of 4 GB or more");
    const uint32_t tiles_m = (m + kTileM - 1) / kTileM;
    uint32_t group = bf16_raster_group(m, n, k, tiles_m);
    if (kern->raster_group >= 0) group = (uint32_t)kern->raster_group;
    if (group > tiles_m) group = tiles_m;
    const FeGemmPlan plan = gemm_plan(kern, m, n, k);
    return fe_gemm_launch(
        plan,
        [&](uint32_t form, uint32_t programs, FeGemmSchedArgs sched) {
            void *args[] = {&act, &x, &w, &m, &n, &k, &lda, &group, &sched};
            return fe_hip_launch(kern->swiglu[form], programs, 1, 1, kGemmThreads, 1, 1, kGemmLds[form], s, args);
        },
        [&](uint32_t tile, uint32_t grid, uint32_t first, uint32_t splits) {
            fe_devptr_t part = kern->part.p;
            void *args[] = {&act, &part, &m, &n, &group, &first, &splits};
            return fe_hip_launch(kern->swiglu_reduce[tile], grid, 1, 1, fe_reduce_threads(tile), 1, 1, 0, s, args);
        });
}

int fe_bf16_linear_forward(const fe_bf16_kernels *kern, fe_stream_t s, fe_devptr_t y, uint32_t ldy, fe_devptr_t x,
                           uint32_t lda, fe_devptr_t w, fe_devptr_t res, uint32_t m, uint32_t n, uint32_t k, uint32_t dec) {
    const char *fn = "fe_bf16_linear_forward";
    if (!kern) return fe_set_error(FE_ERR_ARG, fn, "null kernels");
    if (m == 0) return 0;
    FE_TRY(check(fn, y, ldy, x, lda, w, res, n, k));
    // decode / verify rows: the GEMV, so that a row's bits do not depend on the batch
    uint32_t d = rows_take_gemv(kern, m, n, k, lda, dec) ? m : dec;
    if (k % 256) d = 0;
    for (uint32_t r = 0; r < d; r += kGemvPass) {
        const uint32_t mr = d - r < kGemvPass ? d - r : kGemvPass;
        FE_TRY(launch_gemv(kern, s, y + (size_t)r * ldy * 2, ldy, x + (size_t)r * lda * 2, lda, w,
                            res ? res + (size_t)r * ldy * 2 : 0, mr, n, k));
    }
    if (d == m) return 0;
    return fe_bf16_gemm(kern, s, y + (size_t)d * ldy * 2, ldy, x + (size_t)d * lda * 2, lda, w,
                        res ? res + (size_t)d * ldy * 2 : 0, m - d, n, k);
}

}  // extern "C"
