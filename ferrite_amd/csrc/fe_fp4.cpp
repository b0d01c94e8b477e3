// fe_fp4: host side of the NVFP4 prompt linear (see include/fe_fp4.h). Follows crates/fe-fp4/src/lib.rs; the kernels
// are ferrite_amd/csrc/kernels/k_fp4.hip.
#include "fe_fp4.h"

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <vector>

#include "fe_exl3.h"  // error codes
#include "fe_internal.h"

namespace {
constexpr uint32_t kTile = 128;                 // crates/fe-fp4/src/lib.rs:28
// dynamic LDS by form (256 x 256, its stream-K form, 128 x 256, 128 x 128, 224, 192, 160 x 256): the k tiles in flight, A in whole loads of 64 rows.
// Packed weights: three of A (128 bytes a row; 128 x 256: five) and three of W (36 bytes, 64 in the fp16 form of FP8; 128 x 256: six, 128 x 128:
// four). FP8 codes: two of A (128 x 256: three), three of W, 128 bytes a row.
constexpr uint32_t kGemmLds[kFeGemmForms] = {144 * 1024, 144 * 1024, 136 * 1024, 68 * 1024, 144 * 1024, 120 * 1024, 120 * 1024};
constexpr uint32_t kGemmLds8[kFeGemmForms] = {160 * 1024, 160 * 1024, 144 * 1024, 80 * 1024, 160 * 1024, 144 * 1024, 144 * 1024};
// Forms of the GEMV over programs of 8 CO columns: rows / 2 and CO
constexpr uint32_t kWideRowForms[4] = {1, 2, 4, 8}, kWideColForms[7] = {1, 2, 3, 4, 5, 6, 9};
// Fp4Wide<XP, CO, Q, WV>::LDS of k_fp4.hip; Q (rows m of k quantized by the program itself): with its wavefronts' activations in the place of a stage's
uint32_t wide_lds(uint32_t xp, uint32_t co, uint32_t waves, bool q = false, uint32_t m = 0, uint32_t k = 0) {
    const uint32_t cg = (co + 1) / 2, stage = (co + (q ? 0 : xp)) * 1024 + cg * 256, x = q ? ((k / 256 + waves - 1) / waves * m + 1) / 2 * 1024 * waves : 0;
    return std::max(waves * std::max(2u, std::min((q ? 60 : 80) * 1024 / (waves * stage), 6u)) * stage + x, 64 * waves * (16 * cg + 4));
}
constexpr uint32_t kCuLds = 160 * 1024;
constexpr uint32_t kQuantValues = 10240;
// The wavefronts of a form: eight where K is summed in eighths and two stages of eight wavefronts fit the LDS.
uint32_t wide_waves(uint32_t xp, uint32_t co, bool eighths, bool q = false) { return eighths && co <= 6 && (q || xp <= 2 || (xp == 4 && co <= 4)) ? 8 : 4; }
// Which widths exist: those that a rule or "gemv_cols" may pick. Nine octets pay with 9..16 rows of more columns than six octets a CU; a program of
// eight wavefronts that quantizes takes two octets rather than one (wide_form).
constexpr bool wide_built(uint32_t co, bool eighths, bool q) { return co == 9 ? !eighths && !q : co > 1 || !eighths || !q; }
constexpr uint32_t kGemmThreads = 512;
constexpr uint32_t kTileM = 256;                        // GM_BM
}  // namespace

struct fe_fp4_kernels {
    fe_module_t module = nullptr;
    fe_function_t quant4 = nullptr, gemv4[2][3] = {}, gemv_swiglu4[2][3] = {};  // the GEMVs: [weight tiles, rows as they lie][rows / 16]
    // by form (256 x 256, stream-K, 128 x 256, 128 x 128) and by tile (fe_gemm_launch); gemm8: the fp16 form, 256 x 256 only
    fe_function_t gemm4[kFeGemmForms] = {}, swiglu4[kFeGemmForms] = {}, gemm8c[kFeGemmForms] = {}, gemm8[2] = {};
    fe_function_t reduce4[kFeGemmTiles] = {}, swiglu_reduce4[kFeGemmTiles] = {}, reduce8c[kFeGemmTiles] = {};
    fe_function_t wide[2][4][7] = {};    // the GEMV over programs of 8 CO columns, [quarters or eighths of K][kWideRowForms][kWideColForms]
    fe_function_t wide_q[2][3][7] = {};  // the same, quantizing its activations itself
    fe_function_t gemv8[5][7] = {};  // the FP8 GEMV, [kGemvRowForms][kGemvColForms]
    fe_function_t quant8 = nullptr, expand8 = nullptr;
    uint32_t cus = 0;
    // Switches of the launch paths: read from the environment once, at load; fe_fp4_kernels_set_option changes them
    // afterwards. No forward call reads the environment.
    uint32_t group_m = 8;      // raster group height in row tiles; 0 = all (FE_FP4_GROUP, lib.rs:31-32, 68)
    uint32_t gemv = 1;         // few rows run the GEMV (takes_gemv, fe_gemv_ahead; FE_FP4_NO_GEMV=1: the GEMM's single tile row)
    uint32_t gemv_sk = 0;      // K splits of the GEMV over weight tiles; 0 = two programs a CU (FE_FP4_GEMV_SK)
    uint32_t gemv_strips = 1;  // up to 16 rows run programs of some columns over all of K; 0: weight tiles and K splits, as more rows do (FE_FP4_NO_STRIPS=1)
    // most values (rows x k) that the four wavefronts of the GEMV for up to 16 rows quantize themselves, in every program; eight take twice as many;
    // -1: by the shape, at most kQuantValues (FE_FP4_GEMV_QUANT)
    int32_t gemv_quant = -1;
    uint32_t gemv_cols = 0;    // columns a program of the GEMV for up to 16 rows, or of the FP8 GEMV, takes, rounded up to 8, 16, .. 48, 72; 0 = by the shape (FE_FP4_GEMV_COLS)
    int32_t xcd = -1;          // column tiles dealt to the XCDs: -1 = where the weights are the larger operand (FE_FP4_XCD)
    uint32_t fp8_f16 = 0;      // FP8 linears as fp16 expansion on the 16-bit matrix instruction (FE_FP8_F16=1)
    uint32_t gemm_splits = 8;  // most pieces a cut output tile takes (FE_GEMM_SPLITS; 1: never cut)
    int32_t gemm_sk = 1;       // stream-K schedule of the GEMMs: 0 never, 1 where measured faster, 2 always (FE_GEMM_SK)
    FeGemmTileOptions tile{0, 0, true};  // "gemm_tile", "gemm_pieces"
};

struct fe_fp4_linear {
    std::string name;
    uint32_t n = 0, k = 0;
    float g = 1.0f;
    bool fp8 = false;  // Kind::Fp8 (e4m3 codes [n][k], no block scales), else Kind::Nvfp4 (lib.rs:229-233)
    FeBuf w, sw, alpha;
    // byte strides of the codes / scales of (128-row tile, 64-wide k tile, row in tile); see fe_gemm_nvfp4
    uint32_t w_snt = 0, w_skt = 0, w_sr = 0, s_snt = 0, s_skt = 0, s_sr = 0;
};

struct fe_fp4_workspace {
    uint32_t max_rows = 0, max_k = 0;
    FeBuf codes, sf, aq, part, counters;  // part: partial sums of the GEMM (one slot a CU) or of the GEMV's splits
};
constexpr uint32_t kGemvRows = 48;      // rows of one fe_gemv_nvfp4 pass (three groups of 16)
constexpr uint32_t kGemvMaxRows = 64;   // up to here the GEMV may run (two passes above 48 rows: takes_gemv); above, the GEMM
constexpr uint32_t kGemvCounters = 8192;  // arrival counters: weight tiles of 128 rows (n <= 1 M)

extern "C" {

int fe_fp4_kernels_load(fe_fp4_kernels **out) {
    if (!out) return fe_set_error(FE_ERR_ARG, "fe_fp4_kernels_load", "null out");
    auto *k = new fe_fp4_kernels;
    int c = fe_load_module(&k->module, "FE_FP4_HSACO", fe_k_fp4_hsaco, fe_k_fp4_hsaco_end);
    if (!c) c = fe_hip_module_get_function(&k->quant4, k->module, "fe_fp4_quant");
    auto get = [&](fe_function_t *f, const std::string &nm, uint32_t lds) {
        if (!c) c = fe_hip_module_get_function(f, k->module, nm.c_str());
        if (!c && lds) c = fe_hip_func_set_max_dyn_lds(*f, lds);
    };
    static const char *form_sfx[] = {"", "_sk", "_s1", "_s2", "_h7", "_h6", "_h5"}, *tile_sfx[] = {"", "_s1", "_s2", "_h7", "_h6", "_h5"};
    for (uint32_t i = 0; i < kFeGemmForms; i++) {
        get(&k->gemm4[i], std::string("fe_gemm_nvfp4") + form_sfx[i], kGemmLds[i]);
        get(&k->swiglu4[i], std::string("fe_gemm_nvfp4_swiglu") + form_sfx[i], kGemmLds[i]);
        get(&k->gemm8c[i], std::string("fe_gemm_fp8_codes") + form_sfx[i], kGemmLds8[i]);
        if (i < 2) get(&k->gemm8[i], std::string("fe_gemm_fp8") + form_sfx[i], kGemmLds[i]);
    }
    for (uint32_t i = 0; i < kFeGemmTiles; i++) {
        get(&k->reduce4[i], std::string("fe_gemm_nvfp4_reduce") + tile_sfx[i], 0);
        get(&k->swiglu_reduce4[i], std::string("fe_gemm_nvfp4_swiglu_reduce") + tile_sfx[i], 0);
        get(&k->reduce8c[i], std::string(i < 3 ? "fe_gemm_fp8_codes_reduce" : "fe_gemm_nvfp4_reduce") + tile_sfx[i], 0);  // (one layout of the lower tiles)
    }
    for (int i = 0; i < 6; i++) {
        const std::string form = "x" + std::to_string(i % 3 + 1) + (i / 3 ? "_v" : "");
        get(&k->gemv4[i / 3][i % 3], "fe_gemv_nvfp4_" + form, 0);
        get(&k->gemv_swiglu4[i / 3][i % 3], "fe_gemv_nvfp4_swiglu_" + form, 0);
    }
    for (uint32_t i = 0; i < 8; i++)
        for (uint32_t j = 0; j < 7; j++) {
            const uint32_t xp = kWideRowForms[i % 4];
            const std::string nm = std::to_string(xp) + "_c" + std::to_string(kWideColForms[j]) + (i / 4 ? "_e" : "");
            if (!wide_built(kWideColForms[j], i / 4, false)) continue;
            get(&k->wide[i / 4][i % 4][j], "fe_gemv_nvfp4_r" + nm, wide_lds(xp, kWideColForms[j], wide_waves(xp, kWideColForms[j], i / 4)));
            if (i % 4 < 3 && wide_built(kWideColForms[j], i / 4, true)) get(&k->wide_q[i / 4][i % 4][j], "fe_gemv_nvfp4_q" + nm, kCuLds);
        }
    for (uint32_t i = 0; i < 5; i++)
        for (uint32_t j = 0; j < 7; j++) {
            const uint32_t xo = kGemvRowForms[i], co = kGemvColForms[j];
            if (gemv_form(xo, co)) get(&k->gemv8[i][j], "fe_gemv_fp8_r" + std::to_string(xo) + "_c" + std::to_string(co), gemv_lds(xo, co));
        }
    if (!c) c = fe_hip_module_get_function(&k->quant8, k->module, "fe_fp8_quant");
    if (!c) c = fe_hip_module_get_function(&k->expand8, k->module, "fe_fp8_expand");
    int cus = 0;
    if (!c) c = fe_hip_cu_count(&cus);
    k->cus = (uint32_t)cus;
    if (const char *g = getenv("FE_FP4_GROUP")) k->group_m = (uint32_t)atoi(g);
    if (const char *e = getenv("FE_FP4_NO_GEMV")) k->gemv = atoi(e) ? 0 : 1;
    if (const char *e = getenv("FE_FP4_GEMV_SK")) k->gemv_sk = (uint32_t)atoi(e);
    if (const char *e = getenv("FE_FP4_NO_STRIPS")) k->gemv_strips = atoi(e) ? 0 : 1;
    if (const char *e = getenv("FE_FP4_GEMV_QUANT")) k->gemv_quant = atoi(e);
    if (const char *e = getenv("FE_FP4_GEMV_COLS")) k->gemv_cols = (uint32_t)atoi(e);
    if (const char *e = getenv("FE_FP4_XCD")) k->xcd = atoi(e) ? 1 : 0;
    if (const char *e = getenv("FE_FP8_F16")) k->fp8_f16 = atoi(e) ? 1 : 0;
    if (const char *e = getenv("FE_GEMM_SPLITS")) k->gemm_splits = (uint32_t)atoi(e);
    if (const char *e = getenv("FE_GEMM_SK")) k->gemm_sk = atoi(e);
    if (c) {
        fe_fp4_kernels_destroy(k);
        return c;
    }
    *out = k;
    return 0;
}

int fe_fp4_kernels_destroy(fe_fp4_kernels *k) {
    if (!k) return 0;
    if (k->module) fe_hip_module_unload(k->module);
    delete k;
    return 0;
}

int fe_fp4_kernels_set_option(fe_fp4_kernels *k, const char *name, int32_t value) {
    if (!k || !name) return fe_set_error(FE_ERR_ARG, "fe_fp4_kernels_set_option", "null argument");
    const std::string nm = name;
    if (nm == "group_m") k->group_m = (uint32_t)value;
    else if (nm == "gemv") k->gemv = value ? 1 : 0;
    else if (nm == "gemv_sk") k->gemv_sk = (uint32_t)value;
    else if (nm == "gemv_quant") k->gemv_quant = value;
    else if (nm == "gemv_cols") k->gemv_cols = value;
    else if (nm == "gemv_strips") k->gemv_strips = (uint32_t)value;
    else if (nm == "gemv_once" || nm == "gemv_waves") (void)value;  // of a kernel that is no more: accepted, without effect
    else if (nm == "xcd") k->xcd = value;
    else if (nm == "fp8_f16") k->fp8_f16 = value ? 1 : 0;
    else if (nm == "gemm_splits") k->gemm_splits = (uint32_t)value;
    else if (nm == "gemm_sk") k->gemm_sk = value;
    else if (nm == "gemm_tile") return k->tile.set(value) ? 0 : fe_set_error(FE_ERR_ARG, "fe_fp4_kernels_set_option", "gemm_tile: 0..6");
    else if (nm == "gemm_pieces") k->tile.force_pieces = (uint32_t)value;
    else return fe_set_error(FE_ERR_ARG, "fe_fp4_kernels_set_option", name);
    return 0;
}

int fe_gemm_schedule_query(uint32_t tiles, uint32_t ktiles, uint32_t cus, int32_t mode, int32_t small_b, uint32_t *stream_k,
                           uint32_t *programs, uint32_t *whole, uint32_t *splits, uint32_t *run, uint32_t *run_rem) {
    if (!tiles || !ktiles || !cus || !stream_k || !programs || !whole || !splits || !run || !run_rem)
        return fe_set_error(FE_ERR_ARG, "fe_gemm_schedule_query", "null or zero argument");
    // a stand-in workspace: nonzero addresses that are never dereferenced here
    const FeGemmSchedule s = fe_gemm_schedule(tiles, ktiles, cus, 1, (size_t)cus * kFeGemmSlotsPerCu * kFeGemmPartBytes, 1,
                                              (size_t)tiles, 8, mode, small_b != 0);
    *stream_k = s.stream_k ? 1 : 0, *programs = s.programs, *whole = s.args.full_tiles;
    *splits = s.stream_k ? 1 : s.split.splits, *run = s.args.sk_base, *run_rem = s.args.sk_rem;
    return 0;
}

static int check_shape(const char *name, uint32_t n, uint32_t k) {
    if (!n || !k || n % kTile || k % 128) {
        char msg[160];
        snprintf(msg, sizeof msg, "%s: nvfp4 linear n %u k %u (multiples of 128)", name ? name : "?", n, k);
        return fe_set_error(FE_ERR_SHAPE, "fe_fp4_linear", msg);
    }
    return 0;
}

int fe_fp4_linear_upload(fe_fp4_linear **out, const char *name, uint32_t n, uint32_t k, const uint8_t *codes,
                         const uint8_t *scales, const float *alpha, float g) {
    if (!out || !codes || !scales || !alpha) return fe_set_error(FE_ERR_ARG, "fe_fp4_linear_upload", "null argument");
    FE_TRY(check_shape(name, n, k));
    if (!(g > 0.0f)) return fe_set_error(FE_ERR_ARG, "fe_fp4_linear_upload", "input_scale 0");  // lib.rs:345
    auto *l = new fe_fp4_linear;
    l->name = name ? name : "";
    l->n = n, l->k = k, l->g = g;
    // k-tile-major device layout: the 128 rows of a tile contribute 32 bytes of codes (4 scales) each to one k tile,
    // stored contiguously, so a program's weight read for a k tile is one 4 KB (512 byte) run
    const uint32_t kts = k / 64, nts = n / kTile;
    std::vector<uint8_t> wt((size_t)n * k / 2), st((size_t)n * k / 16);
    for (uint32_t nt = 0; nt < nts; nt++)
        for (uint32_t r = 0; r < kTile; r++) {
            const uint8_t *wrow = codes + (size_t)(nt * kTile + r) * (k / 2), *srow = scales + (size_t)(nt * kTile + r) * (k / 16);
            for (uint32_t kt = 0; kt < kts; kt++) {
                memcpy(&wt[(((size_t)nt * kts + kt) * kTile + r) * 32], wrow + kt * 32, 32);
                memcpy(&st[(((size_t)nt * kts + kt) * kTile + r) * 4], srow + kt * 4, 4);
            }
        }
    l->w_snt = kts * kTile * 32, l->w_skt = kTile * 32, l->w_sr = 32;
    l->s_snt = kts * kTile * 4, l->s_skt = kTile * 4, l->s_sr = 4;
    int c = l->w.from_host(wt.data(), wt.size());
    if (!c) c = l->sw.from_host(st.data(), st.size());
    if (!c) c = l->alpha.from_host(alpha, (size_t)n * 4);
    if (c) {
        delete l;
        return c;
    }
    *out = l;
    return 0;
}

int fe_fp4_linear_from_view(fe_fp4_linear **out, const char *name, uint32_t n, uint32_t k, fe_devptr_t codes,
                            fe_devptr_t scales, fe_devptr_t alpha, float g) {
    if (!out || !codes || !scales || !alpha) return fe_set_error(FE_ERR_ARG, "fe_fp4_linear_from_view", "null argument");
    FE_TRY(check_shape(name, n, k));
    auto *l = new fe_fp4_linear;
    l->name = name ? name : "";
    l->n = n, l->k = k, l->g = g;
    l->w.view(codes, (size_t)n * k / 2);
    l->sw.view(scales, (size_t)n * k / 16);
    l->alpha.view(alpha, (size_t)n * 4);
    // the format's row-major layout, read in place
    l->w_snt = kTile * (k / 2), l->w_skt = 32, l->w_sr = k / 2;
    l->s_snt = kTile * (k / 16), l->s_skt = 4, l->s_sr = k / 16;
    *out = l;
    return 0;
}

int fe_fp8_linear_upload(fe_fp4_linear **out, const char *name, uint32_t n, uint32_t k, const uint8_t *codes,
                         const float *alpha, float g) {
    if (!out || !codes || !alpha) return fe_set_error(FE_ERR_ARG, "fe_fp8_linear_upload", "null argument");
    FE_TRY(check_shape(name, n, k));
    if (!(g > 0.0f)) return fe_set_error(FE_ERR_ARG, "fe_fp8_linear_upload", "input_scale 0");
    auto *l = new fe_fp4_linear;
    l->name = name ? name : "";
    l->n = n, l->k = k, l->g = g, l->fp8 = true;
    // k-tile-major like the NVFP4 codes: [n / 128][k / 64][128 rows][64 bytes]
    const uint32_t kts = k / 64, nts = n / kTile;
    std::vector<uint8_t> wt((size_t)n * k);
    for (uint32_t nt = 0; nt < nts; nt++)
        for (uint32_t r = 0; r < kTile; r++) {
            const uint8_t *wrow = codes + (size_t)(nt * kTile + r) * k;
            for (uint32_t kt = 0; kt < kts; kt++) memcpy(&wt[(((size_t)nt * kts + kt) * kTile + r) * 64], wrow + kt * 64, 64);
        }
    l->w_snt = kts * kTile * 64, l->w_skt = kTile * 64, l->w_sr = 64;
    int c = l->w.from_host(wt.data(), wt.size());
    if (!c) c = l->alpha.from_host(alpha, (size_t)n * 4);
    if (c) {
        delete l;
        return c;
    }
    *out = l;
    return 0;
}

int fe_fp8_linear_from_view(fe_fp4_linear **out, const char *name, uint32_t n, uint32_t k, fe_devptr_t codes,
                            fe_devptr_t alpha, float g) {
    if (!out || !codes || !alpha) return fe_set_error(FE_ERR_ARG, "fe_fp8_linear_from_view", "null argument");
    FE_TRY(check_shape(name, n, k));
    auto *l = new fe_fp4_linear;
    l->name = name ? name : "";
    l->n = n, l->k = k, l->g = g, l->fp8 = true;
    l->w.view(codes, (size_t)n * k);
    l->alpha.view(alpha, (size_t)n * 4);
    l->w_snt = kTile * k, l->w_skt = 64, l->w_sr = k;
    *out = l;
    return 0;
}

int fe_fp4_linear_destroy(fe_fp4_linear *l) {
    delete l;
    return 0;
}

int fe_fp4_linear_shape(const fe_fp4_linear *l, uint32_t *n, uint32_t *k, float *g) {
    if (!l) return fe_set_error(FE_ERR_ARG, "fe_fp4_linear_shape", "null linear");
    if (n) *n = l->n;
    if (k) *k = l->k;
    if (g) *g = l->g;
    return 0;
}

int fe_fp4_workspace_create(fe_fp4_workspace **out, uint32_t max_rows, uint32_t max_k) {
    if (!out || !max_rows || !max_k || max_k % 128) return fe_set_error(FE_ERR_ARG, "fe_fp4_workspace_create", "bad size");
    auto *ws = new fe_fp4_workspace;
    ws->max_rows = max_rows, ws->max_k = max_k;
    const size_t rp = (size_t)(max_rows + kTile - 1) / kTile * kTile;
    // codes sized for one byte an element like the reference's (lib.rs:213-225: enough for FP8, NVFP4 uses half)
    int c = ws->codes.alloc(rp * max_k);
    if (!c) c = ws->sf.zeroed(rp * max_k / 16);
    if (!c) c = ws->aq.alloc(rp * max_k * 2);
    int cus = 0;
    if (!c) c = fe_hip_cu_count(&cus);
    if (!c && cus > 0) c = ws->part.alloc((size_t)cus * kFeGemmSlotsPerCu * kFeGemmPartBytes);
    if (!c) c = ws->counters.zeroed(kGemvCounters * 4);
    if (c) {
        delete ws;
        return c;
    }
    *out = ws;
    return 0;
}

int fe_fp4_workspace_destroy(fe_fp4_workspace *ws) {
    delete ws;
    return 0;
}

int fe_fp4_workspace_buffers(const fe_fp4_workspace *ws, fe_devptr_t *codes, fe_devptr_t *sf, uint32_t *max_rows,
                             uint32_t *max_k) {
    if (!ws) return fe_set_error(FE_ERR_ARG, "fe_fp4_workspace_buffers", "null workspace");
    if (codes) *codes = ws->codes.p;
    if (sf) *sf = ws->sf.p;
    if (max_rows) *max_rows = ws->max_rows;
    if (max_k) *max_k = ws->max_k;
    return 0;
}

int fe_fp4_workspace_operand(const fe_fp4_workspace *ws, fe_devptr_t *aq) {
    if (!ws || !aq) return fe_set_error(FE_ERR_ARG, "fe_fp4_workspace_operand", "null argument");
    *aq = ws->aq.p;
    return 0;
}

static int check_quantize(const fe_fp4_linear *l, const fe_fp4_kernels *kern, const fe_fp4_workspace *ws, fe_devptr_t x, uint32_t lda, uint32_t m) {
    if (!l || !kern || !ws) return fe_set_error(FE_ERR_ARG, "fe_fp4_linear_quantize", "null argument");
    if (m > ws->max_rows || l->k > ws->max_k) {  // lib.rs:521-522
        char msg[200];
        snprintf(msg, sizeof msg, "%s: workspace %ux%u < %ux%u", l->name.c_str(), ws->max_rows, ws->max_k, m, l->k);
        return fe_set_error(FE_ERR_WORKSPACE, "fe_fp4_linear_quantize", msg);
    }
    if (m && (!x || lda < l->k || lda % 8 || x % 16))
        return fe_set_error(FE_ERR_ARG, "fe_fp4_linear_quantize", "x must be 16-byte aligned rows of >= k");
    return 0;
}

int fe_fp4_linear_quantize(const fe_fp4_linear *l, const fe_fp4_kernels *kern, fe_stream_t s, const fe_fp4_workspace *ws,
                           fe_devptr_t x, uint32_t lda, uint32_t m) {
    FE_TRY(check_quantize(l, kern, ws, x, lda, m));
    if (m == 0) return 0;
    uint32_t k = l->k;
    float g = l->g;
    fe_devptr_t codes = ws->codes.p, sf = ws->sf.p, aq = ws->aq.p;
    if (l->fp8) {
        void *args8[] = {&codes, &x, &m, &k, &lda, &g};
        return fe_hip_launch(kern->quant8, (m * (k / 16) + 255) / 256, 1, 1, 256, 1, 1, 0, s, args8);
    }
    void *args[] = {&codes, &sf, &aq, &x, &m, &k, &lda, &g};
    const uint32_t blocks16 = m * (k / 16);
    return fe_hip_launch(kern->quant4, (blocks16 + 255) / 256, 1, 1, 256, 1, 1, 0, s, args);
}

// Which of kWideColForms a GEMV takes: the least of the loads of the CU with the most programs (a program's codes and activations;
// a quarter more where a CU holds one at a time and has several) and the starts of its rounds of programs. us at 1 row: 34816 columns
// of 5120 at 1, 2, .. 6 octets a program 36.9, 24.7, 24.7, 22.1, 23.3, 21.7; 17408 columns 21.8, 15.5, 15.1, 15.4, 13.7, 14.0; 5120 columns
// of 17408 21.0, 17.6, 14.3, 15.7, 18.9, 19.3. Programs of 72 columns pay where the activations weigh most: 34816 columns at 16 rows
// 28.8 us against 29.8 at 48 columns; at 1 row 25.6. Against the weight tiles (gemv_strips = 0), which are ahead at one width: 5120 columns of
// 17408 at 8 / 9 / 12 / 16 rows 19.1 / 20.0 / 20.5 / 21.3 us against 18.4 / 18.8 / 19.2 / 19.9. They are not taken there because a row's bits are to
// be the same at 1 to 16 rows, and at 1 row it is 15.4 against 18.3 (5120 columns of 8704: 1 / 12 rows 10.6 / 13.3 against 13.8 / 14.1).
static uint32_t wide_cols(uint32_t n, uint32_t xp, uint32_t cus, uint32_t forced, bool q = false, uint32_t m = 0, uint32_t k = 0) {
    uint32_t best = 0;
    uint64_t least = ~0ull;
    for (uint32_t i = 0; i < 7; i++) {
        const uint32_t co = kWideColForms[i], programs = (n / 8 + co - 1) / co, room = wide_lds(xp, co, 4, q, m, k) <= 80 * 1024 ? 2 : 1;
        if (forced) {
            best = i;
            if (8 * co >= forced) break;
            continue;
        }
        if (co == 9 && xp < 8) break;
        uint64_t cost = 4ull * ((programs + cus - 1) / cus) * (4 * co + xp);
        if (room == 1 && programs > cus) cost += cost / 4;
        cost += 32ull * ((programs + room * cus - 1) / (room * cus));
        if (cost <= least) best = i, least = cost;
    }
    return best;
}

// The kernel of the GEMV of up to 16 rows; q: the one that quantizes its activations itself.
// Linears that give no CU a second program sum eighths of K, with eight wavefronts up to 8 rows: a program's steps are a chain of LDS reads, scale
// products and matrix instructions, which two wavefronts a SIMD overlap. (By the linear's shape alone: its rows' bits are the same at 1 to 16 rows.)
// us, quarters -> eighths: 5120 x 5120 at 1 / 4 / 8 / 12 rows 7.2 -> 6.6, 8.2 -> 8.0, 9.0 -> 9.0, 9.8 -> 9.8; 5120 x 17408 15.1 -> 14.0, 14.8 ->
// 14.8, 18.3 -> 17.2, 19.7 -> 20.0; 5120 x 8704 9.9 -> 9.1, 10.3 -> 10.4, 11.9 -> 11.4, 12.8 -> 12.9; 2048 x 11008 9.3 -> 7.2, 9.3 -> 8.7, 9.4 ->
// 9.4, 12.4 -> 12.4; 10240 x 4096 at 3 9.9 -> 8.0; 7168 x 2048 at 6 6.9 -> 5.2. With more programs than CUs two of four wavefronts a CU are better
// (34816 x 5120 at 1 row 22.7 against 24.5), and of 1024 channels half of eight have no step (1024 x 1024 at 8 rows 4.3 -> 4.9). Programs of eight
// that quantize take two octets rather than one: 1024 x 5120 at 1 row 5.3 -> 4.8, 2048 x 2048 at 8 rows 5.5 -> 4.9.
struct WideForm {
    uint32_t programs, waves, lds;
    fe_function_t f;
};
static WideForm wide_form(const fe_fp4_linear *l, const fe_fp4_kernels *kern, uint32_t m, bool q) {
    const uint32_t form = m <= 2 ? 0 : m <= 4 ? 1 : m <= 8 ? 2 : 3, xp = kWideRowForms[form], cus = std::max(kern->cus, 1u);
    const bool eighths = l->k >= 2048 && l->n <= 48 * cus;
    uint32_t cols = wide_cols(l->n, xp, cus, kern->gemv_cols, q, m, l->k);
    if (cols == 6 && !wide_built(9, eighths, q)) cols = 5;  // (only where gemv_cols asks for 72)
    if (cols == 0 && !wide_built(1, eighths, q)) cols = 1;
    const uint32_t co = kWideColForms[cols], waves = wide_waves(xp, co, eighths, q);
    return {(l->n / 8 + co - 1) / co, waves, wide_lds(xp, co, waves, q, m, l->k), (q ? kern->wide_q[eighths][form] : kern->wide[eighths][form])[cols]};
}

// Whether fe_fp4_linear_gemm takes the GEMV of up to 16 rows over programs of some columns and all of K, nothing handed between them.
static bool takes_wide(const fe_fp4_linear *l, const fe_fp4_kernels *kern, uint32_t m) {
    return !l->fp8 && m <= 16 && l->n / kTile <= kGemvCounters && kern->gemv && kern->gemv_strips && !kern->gemv_sk && l->k % 256 == 0;
}
// Whether m rows go through a GEMV: all of one pass. 49..64 rows take two, which the GEMM beats (us at 64 rows, two passes -> GEMM: 34816 x 5120 83
// -> 63, 17408 x 5120 41 -> 32, 5120 x 17408 43 -> 30, 5120 x 5120 27 -> 17.5, 2048 x 6144 27 -> 14; 48 rows in one pass 51, 26, 27, 17, 17 against
// 62, 31, 30, 17, 14); they stay where the caller asked for weight tiles (gemv_strips 0: a row's bits the same at every count up to 64) or their K
// splits, with operands that the GEMM does not reach, and where K is so deep that the GEMM's eight pieces of a tile are longer than 16 splits (of
// 1907 linears of 49..64 rows the rule leaves 23 more than 3 % slower than the better one; without it 256 x 59136 at 53 45 against 57). From 33 rows
// on narrow linears of middling depth take it, too, whose tiles are cut along K either way (us at 48 rows, GEMV -> GEMM: 4096 x 4096 16.7 -> 14.1,
// 2048 x 6144 17.1 -> 13.7, 1024 x 5120 15.0 -> 11.3, 1024 x 2816 12.3 -> 10.1, 128 x 8192 14.4 -> 13.1; beyond the lines 5120 x 5120 16.8 -> 16.9,
// 7168 x 2048 13.0 -> 13.7, 1024 x 1024 9.1 -> 9.9, 512 x 14336 17.0 -> 18.9).
static bool takes_gemv(const fe_fp4_linear *l, const fe_fp4_kernels *kern, uint32_t m, bool gemm_reaches) {
    if (l->fp8 || m > kGemvMaxRows || l->n / kTile > kGemvCounters || !kern->gemv) return false;
    if (!kern->gemv_strips || kern->gemv_sk || !gemm_reaches) return true;
    return m <= 32 || (m <= kGemvRows ? l->n > 4096 || l->k < 2048 || l->k > 8192 : l->k > 28000 + 12 * l->n);
}

// K splits of the GEMV over weight tiles. Two programs fit a CU: as many programs as run at once, not more (a second round of short programs costs
// more than idle CUs in the first).
static uint32_t gemv_splits(const fe_fp4_kernels *kern, const fe_fp4_workspace *ws, uint32_t n, uint32_t k) {
    uint32_t sk = std::min({kern->gemv_sk ? kern->gemv_sk : 2 * kern->cus / (n / kTile), 16u, k / 64 / 4});
    while (sk > 1 && (size_t)sk * kGemvRows * n * 4 > ws->part.bytes) sk--;
    return std::max(sk, 1u);
}

// Whether a fused gate|up linear's rows go through the GEMV, by sk splits of K, and not through the GEMM that `plan` is of: up to 16 rows, and up to
// 48 where an estimate of both
// (us) has it ahead. The GEMV's: a start, a wavefront's k tiles (less each where a CU has two programs), the weights' way, and the splits' sums,
// written and read. The GEMM's: its plan's and what that leaves out at so few rows; pieces of K cost less than it says. Fitted to 11766 calls of
// 17..48 rows (256 .. 40960 columns, K 256 .. 19200, weight tiles and, one in five, rows as they lie): half of either within 3 %. With the lines of
// takes_gemv 0.872 of the GEMM's time in all, 1798 calls more than 3 % slower than it, at most 39 %; by this rule 0.867, 88, at most 23 % (the better
// one each time 0.856; of 3922 calls of 1..16 rows the GEMV is the slower one in 2). us, GEMM -> GEMV: 512 x 4992 at 45 rows 13.8 -> 18.4, 1536 x
// 4480 at 38 14.6 -> 19.1, 4864 x 4224 at 40 18.7 -> 23.1, 1280 x 8832 at 35 18.5 -> 20.6 (not taken); 34816 x 5120 at 17 / 48 63 -> 37, 51, 40192 x
// 512 at 46 21.6 -> 15.0, 1536 x 1152 at 28 17.8 -> 11.2.
static bool swiglu_takes_gemv(const fe_fp4_linear *l, const fe_fp4_kernels *kern, uint32_t m, uint32_t sk, const FeGemmPlan &plan) {
    if (m > kGemvRows || l->n / kTile > kGemvCounters || !kern->gemv || kern->tile.force_tile || kern->gemm_sk >= 2) return false;
    if (m <= 16 || !kern->gemv_strips || kern->gemv_sk) return true;
    const uint32_t nts = l->n / kTile, steps = (l->k / 64 + 4 * sk - 1) / (4 * sk), pieces = plan.tile == 1 || plan.tile == 2 ? plan.splits : plan.big.split.splits;
    const float groups = (float)((m + 15) / 16), weights = (float)l->n * (float)l->k, a_cu = std::max(1.0f, (float)(nts * sk) / (float)std::max(kern->cus, 1u));
    const float gemv = 3.47f + groups * (1.6f + (0.513f - 0.142f * a_cu) * (float)steps + 0.124f * (float)sk) + (l->w_sr == 32 ? 0.102e-6f : 0.207e-6f) * weights +
                       (sk > 1 ? 2.0f : 0.0f) + 0.96e-6f * (float)sk * (float)m * (float)l->n;
    return gemv <= 0.95f * (7.95f + 1.007f * plan.us - 0.0174e-6f * weights - (pieces > 1 ? 6.08f : 0.0f));
}

// x: null, or the activations (bf16 rows of lda) which that GEMV quantizes itself
static int linear_gemm(const fe_fp4_linear *l, const fe_fp4_kernels *kern, fe_stream_t s, const fe_fp4_workspace *ws, fe_devptr_t y, uint32_t ldy,
                       uint32_t m, fe_devptr_t res, fe_devptr_t x, uint32_t lda) {
    if (m == 0) return 0;  // lib.rs:535-537
    if (m > ws->max_rows || l->k > ws->max_k) return fe_set_error(FE_ERR_WORKSPACE, "fe_fp4_linear_gemm", "rows or k exceed the workspace");
    // lib.rs:156-157
    if (!y || ldy % 8 || y % 16 || (res && res % 16) || ldy < l->n)
        return fe_set_error(FE_ERR_ARG, "fe_fp4_linear_gemm", "gemm: y/res must be 16-byte aligned rows");
    uint32_t n = l->n, k = l->k;
    const bool gemm_reaches = (uint64_t)m * k * 2 < (1ull << 32) && (uint64_t)n * k < (1ull << 32);
    if (takes_gemv(l, kern, m, gemm_reaches)) {
        // decode-sized: the weight-read-bound GEMV, up to 48 rows a pass
        const uint32_t nts = n / kTile;
        if (takes_wide(l, kern, m)) {
            const WideForm wf = wide_form(l, kern, m, x != 0);
            struct {  // Fp4QuantTo
                fe_devptr_t codes, sf, aq;
                uint32_t ldx;
                float g;
            } to = {ws->codes.p, ws->sf.p, ws->aq.p, lda, l->g};
            fe_devptr_t aq = x ? x : ws->aq.p, w = l->w.p, sw = l->sw.p, alpha = l->alpha.p;
            uint32_t w_snt = l->w_snt, w_skt = l->w_skt, w_sr = l->w_sr, s_snt = l->s_snt, s_skt = l->s_skt, s_sr = l->s_sr;
            void *args[] = {&y, &aq, &w, &sw, &alpha, &res, &m, &n, &k, &ldy, &w_snt, &w_skt, &w_sr, &s_snt, &s_skt, &s_sr, &to};
            return fe_hip_launch(wf.f, wf.programs, 1, 1, 64 * wf.waves, 1, 1, wf.lds, s, args);
        }
        uint32_t sk = gemv_splits(kern, ws, n, k);
        fe_devptr_t w = l->w.p, sw = l->sw.p, alpha = l->alpha.p, z = ws->part.p, cnt = ws->counters.p;
        uint32_t w_snt = l->w_snt, w_skt = l->w_skt, w_sr = l->w_sr, s_snt = l->s_snt, s_skt = l->s_skt, s_sr = l->s_sr;
        for (uint32_t r0 = 0; r0 < m; r0 += kGemvRows) {
            uint32_t rows = m - r0 < kGemvRows ? m - r0 : kGemvRows;
            fe_devptr_t yy = y + (size_t)r0 * ldy * 2, aq = ws->aq.p + (size_t)r0 * k * 2, rr = res ? res + (size_t)r0 * ldy * 2 : 0;
            void *args[] = {&yy, &aq, &w, &sw, &alpha, &rr, &z, &cnt, &rows, &n, &k, &ldy, &sk, &w_snt, &w_skt, &w_sr, &s_snt, &s_skt, &s_sr};
            FE_TRY(fe_hip_launch(kern->gemv4[w_sr != 32][(rows + 15) / 16 - 1], nts * sk, 1, 1, 256, 1, 1, 0, s, args));
        }
        return 0;
    }
    if (!gemm_reaches) return fe_set_error(FE_ERR_UNSUPPORTED, "fe_fp4_linear_gemm", "operand of 4 GB or more");
    const uint32_t tiles_m = (m + kTileM - 1) / kTileM;
    uint32_t group = kern->group_m == 0 || kern->group_m > tiles_m ? tiles_m : kern->group_m;  // lib.rs:148-151
    // FP8 codes: the weights are the larger operand from n >= m on, and at the 8-bit instruction's rate their traffic
    // shows: column tiles are dealt to the XCDs (gemm_raster with group 0), each weight panel through one L2
    if (l->fp8 && n >= m) group = 0;
    if (kern->xcd >= 0) group = kern->xcd ? 0 : group ? group : tiles_m;
    fe_devptr_t aq = ws->aq.p, w = l->w.p, sw = l->sw.p, alpha = l->alpha.p;
    uint32_t w_snt = l->w_snt, w_skt = l->w_skt, w_sr = l->w_sr, s_snt = l->s_snt, s_skt = l->s_skt, s_sr = l->s_sr;
    // FP8 runs on the 8-bit matrix instruction over the codes of both operands, k tiles of 128 (FE_FP8_F16=1: the fp16
    // expansion on the 16-bit instruction, k tiles of 64; same products, another order of the f32 sums)
    const bool codes8 = l->fp8 && !kern->fp8_f16;
    const FeGemmTileOptions f16_form{1, 0, false};  // (the fp16 form exists for 256 x 256 tiles only)
    const bool few = codes8 && kern->gemv && !kern->tile.force_tile && kern->gemm_sk < 2 && m <= kGemvMaxRows;
    FeGemmPlan plan;
    if (!few || m > kFeGemvFp8.always)
        plan = fe_gemm_plan(m, n, codes8 ? k / 128 : k / 64, kern->cus, ws->part.p, ws->part.bytes, ws->counters.p, kGemvCounters, kern->gemm_splits, kern->gemm_sk, /*small_b=*/!l->fp8,
                            l->fp8 ? kFeCostFp8 : kFeCostNvfp4, l->fp8 && !codes8 ? f16_form : kern->tile);
    if (few && fe_gemv_ahead(kFeGemvFp8, m, n, k, k / 128, std::max(kern->cus, 1u), 4, plan)) {
        const uint32_t form = gemv_row_form(m), xo = kGemvRowForms[form], cols = gemv_cols(std::max(m, 3u), n, k, xo, std::max(kern->cus, 1u), kern->gemv_cols ? (int32_t)kern->gemv_cols : -1), co = kGemvColForms[cols];
        fe_devptr_t codes = ws->codes.p;
        uint32_t pc = gemv_even(n, 8 * co, std::max(kern->cus, 1u), 4, kern->gemv_cols != 0 || m <= 2);
        void *args[] = {&y, &codes, &w, &alpha, &res, &m, &n, &k, &ldy, &w_snt, &w_skt, &w_sr, &pc};
        return fe_hip_launch(kern->gemv8[form][cols], (n + pc - 1) / pc, 1, 1, 256, 1, 1, gemv_lds(xo, co), s, args);
    }
    if (l->fp8 && !codes8) {
        uint32_t count = m * k;
        fe_devptr_t codes = ws->codes.p;
        void *args[] = {&aq, &codes, &count};
        FE_TRY(fe_hip_launch(kern->expand8, (count / 8 + 255) / 256, 1, 1, 256, 1, 1, 0, s, args));
    }
    // stream-K programs sit at different depths of K: one row tile at a time (column tiles fastest) keeps those that are
    // in step on one panel of activations
    if (!plan.tile && plan.big.stream_k && kern->xcd < 0) group = 1;
    return fe_gemm_launch(
        plan,
        [&](uint32_t form, uint32_t programs, FeGemmSchedArgs sched) {
            if (codes8) {
                fe_devptr_t codes = ws->codes.p;
                void *args[] = {&y, &codes, &w, &alpha, &res, &m, &n, &k, &ldy, &group, &w_snt, &w_skt, &w_sr, &sched};
                return fe_hip_launch(kern->gemm8c[form], programs, 1, 1, kGemmThreads, 1, 1, kGemmLds8[form], s, args);
            }
            if (l->fp8) {
                void *args[] = {&y, &aq, &w, &alpha, &res, &m, &n, &k, &ldy, &group, &w_snt, &w_skt, &w_sr, &sched};
                return fe_hip_launch(kern->gemm8[form], programs, 1, 1, kGemmThreads, 1, 1, kGemmLds[form], s, args);
            }
            void *args[] = {&y,     &aq,    &w,     &sw,    &alpha, &res,   &m,    &n,    &k,
                            &ldy,   &group, &w_snt, &w_skt, &w_sr,  &s_snt, &s_skt, &s_sr, &sched};
            return fe_hip_launch(kern->gemm4[form], programs, 1, 1, kGemmThreads, 1, 1, kGemmLds[form], s, args);
        },
        [&](uint32_t tile, uint32_t grid, uint32_t first, uint32_t splits) {
            fe_devptr_t part = ws->part.p;
            float scale = l->fp8 ? 1.0f : 0.5f;  // 1 / what the fp16 operands carry (FP4_GEMM_SCALE)
            void *args[] = {&y, &part, &alpha, &res, &m, &n, &ldy, &group, &first, &splits, &scale};
            return fe_hip_launch(codes8 ? kern->reduce8c[tile] : kern->reduce4[tile], grid, 1, 1, fe_reduce_threads(tile), 1, 1, 0, s, args);
        });
}

int fe_fp4_linear_gemm(const fe_fp4_linear *l, const fe_fp4_kernels *kern, fe_stream_t s, const fe_fp4_workspace *ws,
                       fe_devptr_t y, uint32_t ldy, uint32_t m, fe_devptr_t res) {
    if (!l || !kern || !ws) return fe_set_error(FE_ERR_ARG, "fe_fp4_linear_gemm", "null argument");
    return linear_gemm(l, kern, s, ws, y, ldy, m, res, 0, 0);
}

// Whether the GEMV's programs each quantize all of the activations: few values, since a program waits for all of them before its first product. us, with the
// quantizer's launch -> without: 1024 x 1024 at 1 / 8 rows 6.9 -> 3.8, 7.1 -> 4.1; 5120 x 5120 at 1 / 2 rows 8.7 -> 7.3, 8.9 -> 8.0; 17408 x 5120 at
// 1 / 2 15.8 -> 14.0, 16.2 -> 14.5; 34816 x 5120 at 2 24.7 -> 23.7; 16384 x 2560 at 4 9.3 -> 8.3; 5120 x 8704 at 1 11.5 -> 10.0. Beyond 10240 values
// it turns: 34816 x 5120 at 3 rows 25.2 -> 27.0, 16384 x 2560 at 6 10.2 -> 14.3 (one program a CU). Eight wavefronts quantize twice as many in that
// time: 5120 x 17408 at 1 row 17.2 -> 15.9, 4096 x 4096 at 4 6.7 -> 5.8, 1024 x 5120 at 4 / 5 (25600 values) 6.7 -> 6.8, 7.1 -> 7.9. What it costs is
// a wavefront's turns (64 blocks each) times the rounds of programs, each of which quantizes again: of 268 shapes (1024 .. 152064 columns, 1 to 8
// rows), by values alone 0.934 of the time, 51 more than 2 % slower, at most 36 % (152064 x 1280 at 8 rows 35.7 -> 48.4, 152064 x 5120 at 1 74.6 ->
// 82.3, 16384 x 1280 at 8 7.8 -> 8.6); with at most three turns, five times the rounds, 0.918, three more than 2 %, at most 4 % (1024 columns; the
// better of both 0.916). Inputs that no cache holds or that the last call read: the same within 2 %. Up to 8 rows, what the LDS holds and 32 bits
// address. Not where the output or the workspace lies in the activations' memory: programs that have finished would write over what others have yet
// to read.
static bool fp4_quants_itself(const fe_fp4_linear *l, const fe_fp4_kernels *kern, const fe_fp4_workspace *ws, fe_devptr_t y, uint32_t ldy, fe_devptr_t x,
                              uint32_t lda, uint32_t m) {
    if (!m || m > 8 || !takes_wide(l, kern, m) || (uint64_t)m * lda >= (1u << 30)) return false;
    const WideForm f = wide_form(l, kern, m, true);
    const uint64_t most = kern->gemv_quant < 0 ? kQuantValues : (uint64_t)kern->gemv_quant;
    if ((uint64_t)m * l->k > std::min<uint64_t>(most * f.waves / 4, 32768) || f.lds > kCuLds) return false;
    if (kern->gemv_quant < 0) {
        const uint32_t turns = ((l->k / 256 + f.waves - 1) / f.waves * m + 3) / 4, at_once = (f.lds <= kCuLds / 2 ? 2 : 1) * std::max(kern->cus, 1u);
        if (turns > 3 || turns * std::max(at_once, f.programs) > 5 * at_once) return false;
    }
    const fe_devptr_t xe = x + ((size_t)(m - 1) * lda + l->k) * 2;
    auto apart = [&](fe_devptr_t p, size_t bytes) { return p + bytes <= x || p >= xe; };
    return apart(y, ((size_t)(m - 1) * ldy + l->n) * 2) && apart(ws->codes.p, ws->codes.bytes) && apart(ws->sf.p, ws->sf.bytes) && apart(ws->aq.p, ws->aq.bytes);
}

int fe_fp4_linear_forward(const fe_fp4_linear *l, const fe_fp4_kernels *kern, fe_stream_t s, const fe_fp4_workspace *ws,
                          fe_devptr_t y, uint32_t ldy, fe_devptr_t x, uint32_t lda, uint32_t m, fe_devptr_t res) {
    FE_TRY(check_quantize(l, kern, ws, x, lda, m));
    if (fp4_quants_itself(l, kern, ws, y, ldy, x, lda, m)) return linear_gemm(l, kern, s, ws, y, ldy, m, res, x, lda);
    FE_TRY(fe_fp4_linear_quantize(l, kern, s, ws, x, lda, m));
    return fe_fp4_linear_gemm(l, kern, s, ws, y, ldy, m, res);
}

int fe_fp4_linear_forward_swiglu(const fe_fp4_linear *l, const fe_fp4_kernels *kern, fe_stream_t s,
                                 const fe_fp4_workspace *ws, const fe_fp4_workspace *act, fe_devptr_t x, uint32_t lda,
                                 uint32_t m, float down_g) {
    if (!l || !kern || !ws || !act) return fe_set_error(FE_ERR_ARG, "fe_fp4_linear_forward_swiglu", "null argument");
    if (l->fp8 || l->n % 256) {  // lib.rs:388-392, 500
        char msg[200];
        snprintf(msg, sizeof msg, "%s: not an NVFP4 gate|up pair (n %u)", l->name.c_str(), l->n);
        return fe_set_error(FE_ERR_ARG, "fe_fp4_linear_forward_swiglu", msg);
    }
    if (m == 0) return 0;
    uint32_t n = l->n, k = l->k, inter = n / 2;
    if (m > act->max_rows || inter > act->max_k)
        return fe_set_error(FE_ERR_WORKSPACE, "fe_fp4_linear_forward_swiglu", "rows or n / 2 exceed the act workspace");
    if (!(down_g > 0.0f)) return fe_set_error(FE_ERR_ARG, "fe_fp4_linear_forward_swiglu", "down_g");
    FE_TRY(fe_fp4_linear_quantize(l, kern, s, ws, x, lda, m));
    if ((uint64_t)m * k * 2 >= (1ull << 32) || (uint64_t)n * k / 2 >= (1ull << 32))
        return fe_set_error(FE_ERR_UNSUPPORTED, "fe_fp4_linear_forward_swiglu", "operand of 4 GB or more");
    const uint32_t tiles_m = (m + kTileM - 1) / kTileM;
    uint32_t group = kern->group_m == 0 || kern->group_m > tiles_m ? tiles_m : kern->group_m;
    fe_devptr_t aq = ws->aq.p, w = l->w.p, sw = l->sw.p, alpha = l->alpha.p, part = ws->part.p;
    fe_devptr_t q_codes = act->codes.p, q_sf = act->sf.p, q_aq = act->aq.p;
    uint32_t w_snt = l->w_snt, w_skt = l->w_skt, w_sr = l->w_sr, s_snt = l->s_snt, s_skt = l->s_skt, s_sr = l->s_sr;
    // (stream-K only when forced: this kernel's stream-K form was slower wherever measured, 688 -> 714 us on 5120 x 34816)
    auto gemm_plan = [&](const FeGemmTileOptions &tile) {
        return fe_gemm_plan(m, n, k / 64, kern->cus, ws->part.p, ws->part.bytes, ws->counters.p, kGemvCounters, kern->gemm_splits, kern->gemm_sk >= 2 ? kern->gemm_sk : 0, true, kFeCostNvfp4, tile);
    };
    const uint32_t sk = gemv_splits(kern, ws, n, k);
    if (m <= kGemvRows && swiglu_takes_gemv(l, kern, m, sk, gemm_plan(kern->tile))) {  // (fitted to the plans of a plain launch)
        fe_devptr_t cnt = ws->counters.p;
        void *args[] = {&aq, &w, &sw, &alpha, &part, &cnt, &m, &n, &k, (void *)&sk, &w_snt, &w_skt, &w_sr, &s_snt, &s_skt, &s_sr, &q_codes, &q_sf, &q_aq, &down_g};
        return fe_hip_launch(kern->gemv_swiglu4[w_sr != 32][(m + 15) / 16 - 1], n / kTile * sk, 1, 1, 256, 1, 1, 0, s, args);
    }
    FeGemmTileOptions tile = kern->tile;
    tile.nvfp4_front = true;
    const FeGemmPlan plan = gemm_plan(tile);
    if (!plan.tile && plan.big.stream_k && kern->xcd < 0) group = 1;
    return fe_gemm_launch(
        plan,
        [&](uint32_t form, uint32_t programs, FeGemmSchedArgs sched) {
            void *args[] = {&aq,   &w,     &sw,    &alpha, &m,     &n,       &k,    &group, &w_snt, &w_skt,
                            &w_sr, &s_snt, &s_skt, &s_sr,  &sched, &q_codes, &q_sf, &q_aq,  &down_g};
            return fe_hip_launch(kern->swiglu4[form], programs, 1, 1, kGemmThreads, 1, 1, kGemmLds[form], s, args);
        },
        [&](uint32_t tile, uint32_t grid, uint32_t first, uint32_t splits) {
            void *args[] = {&part, &alpha, &m, &n, &group, &first, &splits, &q_codes, &q_sf, &q_aq, &down_g};
            return fe_hip_launch(kern->swiglu_reduce4[tile], grid, 1, 1, fe_reduce_threads(tile), 1, 1, 0, s, args);
        });
}

}  // extern "C"

// Matrix-unit peak (fe_mfma_peak_*): `launches` launches of grid x 256 threads between two events, after one warm-up.
extern "C" int fe_fp4_mfma_peak(const fe_fp4_kernels *kern, fe_stream_t s, int kind, uint32_t seed, uint32_t grid, uint32_t iters,
                                uint32_t launches, float *ms) {
    const char *fn = "fe_fp4_mfma_peak";
    if (!kern || kind < 0 || kind > 2 || !grid || !launches) return fe_set_error(FE_ERR_ARG, fn, "kind 0 (f16), 1 (bf16), 2 (f8)");
    static const char *names[] = {"fe_mfma_peak_f16", "fe_mfma_peak_bf16", "fe_mfma_peak_f8"};
    fe_function_t f = nullptr;
    FE_TRY(fe_hip_module_get_function(&f, kern->module, names[kind]));
    FeBuf out;
    FE_TRY(out.alloc((size_t)grid * 256 * 4));
    fe_devptr_t o = out.p;
    void *args[] = {&o, &iters, &seed};
    fe_event_t a = nullptr, b = nullptr;
    FE_TRY(fe_hip_event_create(&a));
    int c = fe_hip_event_create(&b);
    if (!c) c = fe_hip_launch(f, grid, 1, 1, 256, 1, 1, 0, s, args);
    if (!c) c = fe_hip_event_record(a, s);
    for (uint32_t i = 0; !c && i < launches; i++) c = fe_hip_launch(f, grid, 1, 1, 256, 1, 1, 0, s, args);
    if (!c) c = fe_hip_event_record(b, s);
    if (!c) c = fe_hip_event_sync(b);
    float t = 0;
    if (!c) c = fe_hip_event_elapsed_ms(&t, a, b);
    fe_hip_event_destroy(a);
    fe_hip_event_destroy(b);
    if (!c && ms) *ms = t / (float)launches;
    return c;
}
