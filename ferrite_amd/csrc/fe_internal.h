// Shared by the host-side sources of libferrite_amd: error plumbing, device buffers, embedded code objects.
#pragma once
#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <cstdlib>

#include "fe_hip.h"

int fe_set_error(int code, const char *call, const char *detail);
int fe_check_hip(int code, const char *call);

#define FE_TRY(x)            \
    do {                     \
        int _c = (x);        \
        if (_c) return _c;   \
    } while (0)

// gfx950 code objects linked into the library (fe_embed.S)
extern "C" const unsigned char fe_k_exl3_hsaco[];
extern "C" const unsigned char fe_k_exl3_hsaco_end[];
extern "C" const unsigned char fe_k_exl3_gemm_hsaco[];
extern "C" const unsigned char fe_k_exl3_gemm_hsaco_end[];
#define FE_RGEMM_OBJECT(B)                                             \
    extern "C" const unsigned char fe_k_exl3_rgemm_b##B##_hsaco[];     \
    extern "C" const unsigned char fe_k_exl3_rgemm_b##B##_hsaco_end[];
FE_RGEMM_OBJECT(2)
FE_RGEMM_OBJECT(3)
FE_RGEMM_OBJECT(4)
FE_RGEMM_OBJECT(5)
FE_RGEMM_OBJECT(6)
FE_RGEMM_OBJECT(8)
extern "C" const unsigned char fe_k_fp4_hsaco[];
extern "C" const unsigned char fe_k_fp4_hsaco_end[];
extern "C" const unsigned char fe_k_route_hsaco[];
extern "C" const unsigned char fe_k_route_hsaco_end[];
extern "C" const unsigned char fe_k_bf16_hsaco[];
extern "C" const unsigned char fe_k_bf16_hsaco_end[];

// The embedded image, or the file the environment variable names.
int fe_load_module(fe_module_t *out, const char *env, const unsigned char *begin, const unsigned char *end);

// Device memory owned until destruction, or a borrowed view (DeviceBuffer / DeviceBuffer::view,
// crates/fe-cuda/src/lib.rs:201-297).
struct FeBuf {
    fe_devptr_t p = 0;
    size_t bytes = 0;
    bool owned = false;
    FeBuf() = default;
    FeBuf(const FeBuf &) = delete;
    FeBuf &operator=(const FeBuf &) = delete;
    ~FeBuf() { release(); }
    int alloc(size_t n) {
        release();
        FE_TRY(fe_hip_malloc(&p, n));
        bytes = n;
        owned = true;
        return 0;
    }
    int zeroed(size_t n) {
        FE_TRY(alloc(n));
        if (fe_hip_zero_alloc_on()) return 0;  // fe_hip_malloc has cleared the block and synchronized
        FE_TRY(fe_hip_memset_d8(p, 0, n, nullptr));
        return fe_hip_synchronize();
    }
    int from_host(const void *src, size_t n) {
        FE_TRY(alloc(n));
        return fe_hip_memcpy_htod(p, src, n);
    }
    void view(fe_devptr_t q, size_t n) {
        release();
        p = q;
        bytes = n;
        owned = false;
    }
    void release() {
        if (owned && p) fe_hip_free(p);
        p = 0;
        bytes = 0;
        owned = false;
    }
};

// forward() of an EXL3 linear for at most max_rows rows over caller-provided device memory instead of a workspace object:
// arrival counters (zero at rest), rotated inputs, split partial sums. Sizes that do not fit are FE_ERR_WORKSPACE.
// Allocates nothing. (fe_exl3.cpp; used by fe_exl3_linear_forward_static.)
struct fe_exl3_linear;
struct fe_exl3_kernels;
struct fe_exl3_workspace;
int fe_exl3_forward_over(const fe_exl3_linear *l, const fe_exl3_kernels *kern, fe_stream_t s, fe_devptr_t x, int x_dtype,
                         fe_devptr_t y, int y_dtype, uint32_t rows, uint32_t max_rows, fe_devptr_t counters,
                         size_t counters_bytes, fe_devptr_t xh, size_t xh_bytes, fe_devptr_t z, size_t z_bytes, const char *fn);
// Linears of one input (bf16, rows of k) over a prompt in one launch behind one rotation, bf16 out, where the GEMM that decodes into
// registers takes all of them and the workspace holds their rotated inputs; *taken: whether it was. A member's sums may add in
// another order than its own forward's (the launch's tiles are spread as one). For the routing layer.
int fe_exl3_forward_prompt_group(const fe_exl3_linear *const *ls, size_t count, const fe_exl3_kernels *kern, fe_stream_t s, fe_devptr_t x,
                                 const fe_devptr_t *ys, uint32_t rows, const fe_exl3_workspace *ws, bool *taken);
// Looks up the static scratch array of fe_exl3_linear_forward_static on the current device and clears its counters
// (fe_exl3_static.hip); fe_hip_init calls it for the device it binds.
int fe_exl3_static_setup_current_device();

// Column blocks of upb units that the decode GEMV of `programs` runs (run q starts at unit q base + min(q, rem)), `per` of them a workgroup, cuts: those inside
// which a workgroup's run starts.
inline uint32_t fe_gemv_cut_blocks(uint32_t units, uint32_t programs, uint32_t upb, uint32_t per) {
    const uint32_t base = units / programs, rem = units % programs;
    uint32_t cut = 0, nb = 0, in = 0, last = 0xffffffffu;  // the start: unit `in` of block nb
    for (uint32_t q = per; q < programs; q += per) {
        for (in += per * base + std::min(q, rem) - std::min(q - per, rem); in >= upb; in -= upb) nb++;
        if (in && nb != last) cut++, last = nb;
    }
    return cut;
}

// How the prefill GEMM's output tiles (256 x 256) are spread over the CUs: `full` tiles are computed whole, one per
// program; the `tiles - full` tiles of a last, mostly empty round are each cut `splits` ways along K (partials in a
// workspace, then a reduce kernel). splits == 1 means nothing is cut (full == tiles).
struct FeGemmSplit {
    uint32_t tiles = 0, full = 0, splits = 1;
    uint32_t programs() const { return full + (tiles - full) * splits; }
    uint32_t cut() const { return tiles - full; }
};
constexpr size_t kFeGemmPartBytes = 256 * 256 * 4;  // one partial slot
constexpr uint32_t kFeGemmSlotsPerCu = 2;           // slots a workspace holds per CU
// The cut that finishes the last round soonest: s pieces a tile take ceil(rem s / cus) rounds of 1 / s of a tile's time;
// every piece also writes its 256 KB partial and the reduce kernel reads it back (about 2 % of a tile's time a piece).
// At most `slots` pieces in all and `cap` a tile (1: never cut).
inline FeGemmSplit fe_gemm_split(uint32_t tiles, uint32_t ktiles, uint32_t cus, uint32_t slots, uint32_t cap = 8) {
    FeGemmSplit g;
    g.tiles = g.full = tiles;
    if (!cus || !slots) return g;
    const uint32_t rem = tiles % cus;
    if (rem == 0) return g;
    cap = std::min(cap, ktiles / 4);                                        // at least 4 k tiles a program
    cap = std::min(cap, slots / rem);
    uint32_t best = 1;
    float best_cost = 1.0f;
    for (uint32_t sp = 2; sp <= cap; sp++) {
        const float cost = (float)((rem * sp + cus - 1) / cus) / (float)sp + 0.02f * (float)sp;
        if (cost < best_cost - 1e-6f) best = sp, best_cost = cost;
    }
    if (best < 2) return g;
    g.full = tiles - rem;
    g.splits = best;
    return g;
}

// The schedule argument of the GEMM kernels (GemmSched of kernels/gemm_core.h) and what to launch with it.
struct FeGemmSchedArgs {
    uint32_t full_tiles, splits, sk_base, sk_rem;
    fe_devptr_t part;
    uint32_t part_bytes, pad_;
    fe_devptr_t counters;
};
struct FeGemmSchedule {
    FeGemmSplit split;     // the one-piece schedule (when !stream_k): its cut tiles need the reduce launch
    FeGemmSchedArgs args;
    uint32_t programs = 0;
    bool stream_k = false;
};
// mode 0: always one piece a program. mode 2: runs over all tiles wherever the workspace allows, mode 3: as many whole
// rounds as leave runs that are in step (both for tests). mode 1: stream-K where it is the faster schedule, as measured
// (MI355X, NVFP4, FP8 and EXL3, 20..1088 tiles). It pays where the one-piece schedule cannot fill its last round: the
// tiles of that round (all tiles when there are fewer than CUs) then run as runs over all CUs, behind the whole rounds.
// Taken when the one-piece schedule cuts those tiles (tiles that run whole in one partly filled round are left alone:
// 192 or 224 tiles on as many CUs clock higher under the power limit, stream-K loses 1..12 % there), a tile has at most
// three pieces (runs of at least half a tile: the piece that arrives last adds the others alone, about 5 us a piece; 32
// tiles of 8 pieces: 74 against 39 us), and either
//  (a) the cut leaves a partly filled round and the runs are equal and in step, programs 8 apart (the same XCD) at the same
//      depth of K at the same time, so that they share panels in their L2 (160 tiles on 256 CUs, 2048 rows x 5120
//      columns: NVFP4 300 -> 284 us, FP8 166 -> 154, EXL3 over kept tiles 358 -> 352, decoding 393 -> 363), or
//  (b) small weight operand only (small_b: packed weights of a few KB a k tile; NVFP4, the decoding EXL3 GEMM): the cut
//      loses 12 % or more to its rounds, whether or not the runs are in step (129..160 tiles: three pieces a tile, a
//      second round half empty; NVFP4 +14..27 %, EXL3 +11..15 %; 1536 rows x 17408 columns = 256 whole + 152: 241 -> 227
//      us). Where it loses 7 % (120 or 240 tiles) stream-K loses 9..20 %: programs that are not in step stream their
//      operands past the L2.
// With a whole number of rounds stream-K and the one-piece schedule are within 1 % of each other: one piece a program.
// Whole rounds and runs that are in step over more than the last round (576 tiles as 256 + runs of 100 k tiles) spare the
// reduce launch and are 1..3 % faster: taken for a small weight operand, (c) below; (d) and (e) below are two more cases
// of a small weight operand, runs over all tiles behind no whole round.
// With decoded fp16 tiles or FP8 codes as the weight operand (32 KB a k tile) runs behind whole rounds lose 4..9 %.
// (NVFP4 up to 2048 rows with more tiles than CUs asks with mode 0: fe_gemm_mode. Of what is said here about more tiles than CUs, the NVFP4 figures
// up to 2048 rows were taken against a one-piece schedule without lower tiles and with rows that do not exist read again; the rules stand for NVFP4
// over 2048 rows and for the trellis GEMM that decodes into LDS.) Needs two partial slots a program and a zeroed counter a tile.
constexpr uint32_t kFeXcds = 8;
inline FeGemmSchedule fe_gemm_schedule(uint32_t tiles, uint32_t ktiles, uint32_t cus, fe_devptr_t part, size_t part_bytes,
                                       fe_devptr_t counters, size_t counters_len, uint32_t cap, int mode, bool small_b) {
    FeGemmSchedule r;
    const uint32_t slots = (uint32_t)(part_bytes / kFeGemmPartBytes);
    r.split = fe_gemm_split(tiles, ktiles, cus, slots, cap);
    r.programs = r.split.programs();
    r.args = {r.split.full, r.split.splits, 0, 0, part, (uint32_t)std::min<size_t>(part_bytes, 0xffffffffu), 0, counters};
    const uint32_t programs = std::min<uint32_t>({cus, tiles * ktiles, slots / 2});
    if (!mode || !programs || !counters || tiles > counters_len || (uint64_t)tiles * ktiles >= (1ull << 31) ||
        (size_t)programs * 2 * kFeGemmPartBytes > 0xffffffffu)
        return r;
    // whole rounds first (mode 3, and mode 1 where it pays), the runs over the tiles after them
    uint32_t whole = 0, base = 0, rem = 0;
    auto runs = [&](uint32_t rounds) {
        whole = rounds * programs;
        const uint32_t units = (tiles - whole) * ktiles;
        base = units / programs, rem = units % programs;
    };
    auto good = [&]() { return rem == 0 && 2 * base >= ktiles && (kFeXcds * base) % ktiles == 0; };
    auto most_whole_rounds = [&](uint32_t at_least) {
        for (uint32_t rounds = tiles / programs + 1; rounds-- > at_least;) {
            runs(rounds);
            if (base > 0 && good()) return true;
        }
        return false;
    };
    runs(0);
    if (mode == 1) {
        // the tiles of the last, partly filled round (all tiles when there are fewer than CUs): are runs over them worth it?
        const uint32_t last = tiles % cus;
        bool take = false;
        // (e) small weight operand, short K (up to 128 k tiles), between one and 2 1/8 rounds with a cut last round of at
        // most 5/8 of the CUs: equal runs over all tiles, in step, instead of whole rounds with runs behind them or a cut
        // (every tile then has two pieces, but the programs reach their tile ends at different times; behind a whole round
        // all of them meet at once). 5120-wide K, NVFP4 / decoding EXL3, us: 320 tiles 184.5 -> 181 / 235.5 -> 230; 384:
        // 213 -> 204.5 / 265.5 -> 263; 416: 238 -> 232 / 302 -> 292.5; 544: 286 -> 284.7 / 364 -> 356.5. With a fuller last
        // round (448 tiles: 248 -> 250 / 315 -> 320), from 2 1/4 rounds on (576, 640, 1088 tiles) and with 272 k tiles a tile
        // (320 tiles: 675 -> 728) it loses 1..8 %: not taken.
        if (small_b && last && 8 * last <= 5 * cus && tiles > cus && 8 * tiles <= 17 * cus && ktiles <= 128 &&
            r.split.splits > 1 && programs == cus) {
            runs(0);
            take = good() && base >= 64;
        }
        if (!take && last && (tiles < cus || small_b)) {
            runs(tiles / cus);
            // what the one-piece schedule loses to its partly filled rounds, as a fraction of the balanced time
            const uint32_t sp = r.split.splits;
            const float one_piece = (float)((last * sp + cus - 1) / cus) / (float)sp, balanced = (float)last / (float)cus;
            const float gain = one_piece / balanced - 1.0f;
            take = programs == cus && 2 * base >= ktiles && sp > 1 && ((good() && gain > 0.0f) || (small_b && gain >= 0.12f));
        }
        // (c) small weight operand, a cut last round of too many pieces a tile: one whole round fewer, so that the runs are
        // longer, if they are then in step (576 tiles = 256 whole + runs of 100 k tiles over 320: no reduce launch, NVFP4
        // 312 -> 309 us, EXL3 404 -> 392). A last round that runs whole (480 tiles: 224 on as many CUs) is left alone: runs
        // of 70 behind a whole round are 2..4.5 % slower there.
        if (!take && small_b && last && tiles > cus && r.split.splits > 1) take = most_whole_rounds(1);
        // (d) small weight operand, one whole round and a last round of few tiles (an eighth of the CUs or fewer), which (c)
        // cannot turn into runs in step: runs over all tiles, if they are equal, at least a tile long (two pieces a tile)
        // and keep the programs of an XCD at no more than two depths of K at a time. 272 tiles of 80 k tiles (1024 rows x
        // 17408 columns; the one-piece schedule cuts the 16 tiles 7 ways and adds a reduce launch), runs of 85: EXL3
        // 199.5 -> 190.8 us, NVFP4 155.0 -> 154.3; 288 tiles, runs of 90: EXL3 211 -> 201, NVFP4 165 -> 162. Behind a
        // second whole round (528 tiles as 256 + runs of 85) nothing is gained: not taken.
        if (!take && small_b && last && tiles > cus && tiles < 2 * cus && 8 * last <= cus && r.split.splits > 1 &&
            programs == cus) {
            runs(0);
            const uint32_t step = (kFeXcds * base) % ktiles;
            take = rem == 0 && base >= ktiles && base >= 64 && (step == 0 || 2 * step == ktiles);
        }
        if (!take) return r;
    } else if (mode >= 3 && !most_whole_rounds(0)) {
        return r;
    }
    if (base == 0 || (base >= ktiles && rem == 0 && base % ktiles == 0 && whole == 0)) return r;  // whole tiles only: nothing to gain
    r.stream_k = true;
    r.programs = programs;
    r.args.full_tiles = whole;
    r.args.sk_base = base, r.args.sk_rem = rem;
    return r;
}

// ---- which tiles a GEMM launch takes -------------------------------------------------------------------------------------------
// Tile 0: 256 x 256, on one of the two schedules above. Tiles 1 (128 x 256) and 2 (128 x 128): a launch of small tiles, each cut
// `splits` ways along K. Tiles 3, 4, 5 (224, 192, 160 x 256): as tile 0, one piece a program.
constexpr uint32_t kFeGemmTiles = 6, kFeGemmTileM[kFeGemmTiles] = {256, 128, 128, 224, 192, 160}, kFeGemmTileN[kFeGemmTiles] = {256, 256, 128, 256, 256, 256};
constexpr uint32_t kFeGemmForms = kFeGemmTiles + 1;  // kernels: tile 0 one piece a program and stream-K, then the other tiles

struct FeGemmPlan {
    FeGemmSchedule big;  // tiles 0 and 3..5
    uint32_t tile = 0, tiles = 0, splits = 1;
    float us = 0;  // the estimate (0: a tile was forced)
};
// Switches of the plan (options of the three kernels handles): force_tile 0 = by the rule, 1 = 256 x 256, 2, 3 = small tile 1, 2
// with force_pieces pieces of K (0: one).
struct FeGemmTileOptions {
    uint32_t force_tile = 0, force_pieces = 0;
    bool low = false;  // the handle has kernels of tiles 3..5 (force_tile 4, 5, 6)
    bool nvfp4_front = false;  // an NVFP4 launch with SwiGLU and the quantizer behind it
    // option "gemm_tile": refused past the tiles that the handle has kernels of (fe_gemm_plan and the tables of kernels are indexed by it)
    bool set(int64_t value) {
        if (value < 0 || value > (low ? kFeGemmTiles : 3u)) return false;
        force_tile = (uint32_t)value;
        return true;
    }
};

// What a program of each tile takes on one weight form: us a k tile (64; FP8: 128), `full` more of it when all CUs are busy (clock and
// memory), us a program besides, and how much slower two programs that share a CU (tile 2) are than one alone. Fitted to 770
// timings a form (MI355X, 80..1536 rows, 2048 x 2048 .. 17408 x 5120, 1..8 pieces; most of them within 6 % for trellis and NVFP4 weights,
// 10..13 % for bf16 and FP8, whose panels compete for memory). stream_k: what meeting through the workspace adds. again: what small
// tiles in more than one round take more than their rounds add up to (trellis: the programs that come second decode alone; 528 tiles 128 x 128 of
// 32 k tiles 80 us where the rounds add up to 67).
// short_k: how much of the small tiles' estimate a lower tile may take with more tiles than CUs and fewer than 24 k tiles (fe_gemm_plan).
// high: us a k tile of tiles of 256, 224, 192, 160 rows, and how much more of it when all CUs are busy, for the choice among them (fe_gemm_height):
// fitted to 112 timings a form and height (128..1900 rows, 2048 x 4096 .. 17408 x 5120) without a fixed part, half of them within 5 % (FP8: to 60,
// half within 5 %, nine tenths within 11..15 %; 962 launches against the tree before its lower tiles' loop of today, 647 of them with another tile:
// those 0.910 of the time, one more than 3 % slower, 1792 x 19072 at 1263 rows 69.0 -> 73.3; the others 0.985, 8704 x 5120 at 129 rows 20.5 -> 21.1).
// f8: FP8 weights, for two lines of fe_gemm_plan.
struct FeGemmCost {
    float ktile[3], full[3], fixed[3], shared, stream_k, again, high[4][2], short_k;
    bool f8 = false;
};
constexpr FeGemmCost kFeCostTrellis = {{1.38f, 1.02f, 0.71f}, {0.12f, 0.07f, 0.08f}, {1.0f, 3.0f, 1.9f}, 1.63f, 48.7f, 1.12f, {}, 0.0f};
constexpr FeGemmCost kFeCostNvfp4 = {{1.32f, 0.73f, 0.44f}, {-0.07f, 0.05f, 0.09f}, {0.0f, 2.2f, 2.3f}, 1.59f, 44.0f, 1.0f, {{1.11f, 0.29f}, {1.16f, 0.16f}, {0.90f, 0.36f}, {0.57f, 1.03f}}, 0.97f};
constexpr FeGemmCost kFeCostFp8 = {{1.20f, 0.58f, 0.66f}, {0.09f, 0.46f, 0.21f}, {0.0f, 2.5f, 0.4f}, 1.21f, 36.4f, 1.0f, {{1.04f, 0.13f}, {1.07f, 0.03f}, {0.93f, 0.10f}, {0.88f, 0.05f}}, 0.77f, true};
constexpr FeGemmCost kFeCostBf16 = {{1.10f, 0.64f, 0.45f}, {0.22f, 0.43f, 0.41f}, {0.0f, 1.5f, 0.3f}, 1.53f, 53.2f, 1.0f, {{1.26f, 0.04f}, {1.24f, 0.01f}, {0.92f, 0.20f}, {0.77f, 0.34f}}, 0.9f};

// `programs` programs of `ktiles` k tiles each, in rounds of all CUs (tile 2: two a CU).
inline float fe_gemm_cost(const FeGemmCost &c, uint32_t tile, uint32_t programs, uint32_t ktiles, uint32_t cus) {
    const uint32_t round = tile == 2 ? 2 * cus : cus, last = programs % round;
    const float whole = (float)ktiles * c.ktile[tile] * (1.0f + c.full[tile]) * (tile == 2 ? c.shared : 1.0f) + c.fixed[tile];
    const float part = (float)ktiles * c.ktile[tile] * (1.0f + c.full[tile] * (float)last / (float)cus) + c.fixed[tile];
    return (float)(programs / round) * whole + (last > cus ? whole : last ? part : 0.0f);
}
// The reduce launch: its start, and the partials written and read once.
inline float fe_gemm_reduce_cost(uint32_t programs, uint32_t tile) {
    return 4.0f + (float)programs * (float)(kFeGemmTileM[tile] * kFeGemmTileN[tile]) * 8.0f / 5e6f;
}

// What a launch of tiles of one height (256, 224, 192, 160 rows: h 0..3) takes, for the choice among them: rounds of one program a CU, and the
// pieces' sums, which travel twice.
inline float fe_gemm_height(const FeGemmCost &c, uint32_t h, const FeGemmSplit &g, uint32_t ktiles, uint32_t cus, uint32_t rows_a_tile) {
    auto rounds = [&](uint32_t programs, uint32_t k) {
        const uint32_t last = programs % cus;
        return (float)k * c.high[h][0] * ((float)(programs / cus) * (1.0f + c.high[h][1]) + (last ? 1.0f + c.high[h][1] * (float)last / (float)cus : 0.0f));
    };
    float t = rounds(g.full, ktiles);
    if (g.cut()) t += rounds(g.cut() * g.splits, (ktiles + g.splits - 1) / g.splits) + 2.5f + (float)(g.cut() * g.splits * rows_a_tile) * 2048.0f / 5e6f;
    return t;
}

// Stream-K of the forms that have lower tiles, up to 2048 rows: only with fewer tiles than CUs. Behind or over whole rounds, rows that do not exist,
// the reduce launch and lower tiles cost the one-piece schedule less than the runs' meetings cost (NVFP4, us, stream-K -> one piece: 34816 x 5120 at
// 400 / 777 / 2048 rows 144 -> 130, 267 -> 242, 531 -> 521; 17408 x 5120 at 777 / 1800 138 -> 130, 273 -> 257; 16384 x 4096 at 1500 182 -> 154; at
// most 2 % the other way: 12288 x 2048 at 1500 69.0 -> 70.6). With
// fewer: 34816 x 5120 at 200 rows 94 against 102, 5120 x 17408 at 2048 265 against 277.
inline int fe_gemm_mode(int mode, uint32_t m, uint32_t tiles256, uint32_t cus, const FeGemmTileOptions &opt) {
    return mode == 1 && opt.low && m <= 2048 && tiles256 > cus ? 0 : mode;
}

// The rule: with fewer than a few rounds of 256 x 256 tiles, most of the time is CUs without a tile or pieces of K that meet;
// tiles of half and a quarter the size fill the chip with fewer pieces. They read more operand bytes and run fewer matrix
// instructions between two barriers (a k tile of them costs more than its share), so they pay only where the fill gains more:
// the estimate above decides, with 6 % against a small tile. The margin is the one that loses least over the estimate's errors, not a bound
// of them: of 14 row counts on 10 layers in each form the rule took a tile more than 3 % slower than 256 x 256 once (NVFP4, 1536 rows of 8704 x 5120:
// 133 us against 126); with the errors' 10..13 % as the margin bf16 and FP8 miss a dozen gains (bf16 192 rows of 17408 x 5120 59 -> 67, FP8 777 rows
// of 5120 x 17408 80 -> 88) and avoid no loss. Pieces of at least 8 k tiles, at most as many
// programs as run at once when K is cut. Up to 2048 rows, what the estimate was fitted on: beyond, whole rounds of 256 x 256
// prevail. 5120 x 5120, us, before -> with small tiles: NVFP4 100 rows 31 -> 21, bf16 1000 rows 58 -> 56, FP8 1000 rows 42 -> 30.
inline FeGemmPlan fe_gemm_plan(uint32_t m, uint32_t n, uint32_t ktiles, uint32_t cus, fe_devptr_t part, size_t part_bytes,
                               fe_devptr_t counters, size_t counters_len, uint32_t cap, int mode, bool small_b,
                               const FeGemmCost &cost, const FeGemmTileOptions &opt) {
    FeGemmPlan p;
    const uint32_t tiles256 = ((m + 255) / 256) * ((n + 255) / 256);
    mode = fe_gemm_mode(mode, m, tiles256, cus, opt);
    p.big = fe_gemm_schedule(tiles256, ktiles, cus, part, part_bytes, counters, counters_len, cap, mode, small_b);
    auto take = [&](uint32_t tile, uint32_t tiles, uint32_t pieces) { p.tile = tile, p.tiles = tiles, p.splits = pieces, p.big.stream_k = false; };
    auto tiles_of = [&](uint32_t tile) {
        return ((m + kFeGemmTileM[tile] - 1) / kFeGemmTileM[tile]) * ((n + kFeGemmTileN[tile] - 1) / kFeGemmTileN[tile]);
    };
    auto most_pieces = [&](uint32_t tile, uint32_t want) {
        const size_t slots = part_bytes / (kFeGemmTileM[tile] * kFeGemmTileN[tile] * 4);
        return (uint32_t)std::max<size_t>(1, std::min<size_t>({want, ktiles, slots / tiles_of(tile)}));
    };
    auto low = [&](uint32_t tile) {  // the one-piece schedule of tiles as high as kFeGemmTileM[tile]
        return fe_gemm_schedule(tiles_of(tile), ktiles, cus, part, part_bytes, 0, 0, cap, 0, small_b);
    };
    if (opt.force_tile >= 4 && opt.low) {
        p.tile = opt.force_tile - 1, p.big = low(p.tile);
        return p;
    }
    if (opt.force_tile == 2 || opt.force_tile == 3) {
        take(opt.force_tile - 1, tiles_of(opt.force_tile - 1), most_pieces(opt.force_tile - 1, std::max(1u, opt.force_pieces)));
        return p;
    }
    if (opt.force_tile || mode >= 2 || !cus) return p;
    float best;
    if (p.big.stream_k) {
        const FeGemmSchedArgs &a = p.big.args;
        best = fe_gemm_cost(cost, 0, p.big.programs, a.full_tiles / p.big.programs * ktiles + a.sk_base + 1, cus) + cost.stream_k;
    } else {
        const FeGemmSplit &g = p.big.split;
        best = fe_gemm_cost(cost, 0, g.full, ktiles, cus);
        if (g.cut())
            best += fe_gemm_cost(cost, 0, g.cut() * g.splits, (ktiles + g.splits - 1) / g.splits, cus) + fe_gemm_reduce_cost(g.cut() * g.splits, 0);
    }
    // Lower tiles: as many row tiles of less waste, or another count of them that fills the rounds of the CUs better (rows that do not exist cost
    // little power, but their time). By the ratio of the two estimates, which share most of their errors. Of 336 launches (8 layers, 14 row counts,
    // NVFP4, FP8 and bf16) against 256 rows: 0.925, 0.93, 0.905 of the time (the best height each time: 0.92, 0.92, 0.90), four more than 2 % slower,
    // at most 7 %. With the small tiles in the choice, 12 other layers of 144 launches a form against the rule without lower tiles: 0.93, 0.97, 0.93;
    // 8 of 432 more than 3 % slower, at most 7 %. (With FP8's loop and heights, the reduce launches and the epilogues of before; FP8's figures since
    // are at FeGemmCost.)
    uint32_t pick = 0;
    float ratio = p.big.stream_k ? 0.9f : 0.97f;
    if (opt.low && m <= 2048) {
        const uint32_t tiles_n = (n + 255) / 256;
        auto height = [&](uint32_t tile, uint32_t h, const FeGemmSplit &g) { return fe_gemm_height(cost, h, g, ktiles, cus, m / (tiles_of(tile) / tiles_n)); };
        const float high = height(0, 0, p.big.split);
        for (uint32_t tile = 3; tile < kFeGemmTiles; tile++) {
            const FeGemmSplit g = low(tile).split;
            float r = height(tile, tile - 2, g) / high;
            if (2 * g.programs() < cus) r = std::max(r, 0.85f);  // (mostly idle CUs: a k tile takes the trip of its loads, at any height)
            if (r < ratio) ratio = r, pick = tile;
        }
    }
    const float whole = best;
    p.us = best;
    for (uint32_t tile = 1; tile <= 2 && m <= 2048; tile++) {
        const uint32_t tiles = tiles_of(tile), most = most_pieces(tile, std::min(cap, ktiles / 8));
        for (uint32_t pieces = 1; pieces <= most; pieces++) {
            if (pieces > 1 && tiles * pieces > cus * tile) break;
            float c = fe_gemm_cost(cost, tile, tiles * pieces, (ktiles + pieces - 1) / pieces, cus);
            if (pieces > 1) c += fe_gemm_reduce_cost(tiles * pieces, tile);
            if (tiles * pieces > cus * tile) c *= cost.again;
            if (1.06f * c < best) take(tile, tiles, pieces), p.us = c, best = 1.06f * c;
        }
    }
    if (!pick) return p;
    // In the place of a small tile a lower one is taken only with at least 12 k tiles and half of the CUs: the heights' estimate has no fixed part
    // and was fitted on launches that fill the chip. Of 1499 launches (128 .. 40000 columns, K 256 .. 20000, 65 .. 2048 rows; NVFP4, its SwiGLU
    // front, FP8, bf16) against the rule without lower tiles: with them wherever the estimate says so 68 more than 3 % slower (5248 x 256 at 636 rows
    // 9.2 -> 13.1 us, 7168 x 256 SwiGLU at 140 13.4 -> 25.6, 256 x 1536 bf16 at 210 7.8 -> 10.3, 11136 x 256 FP8 at 315 9.1 -> 11.6) and 0.986 /
    // 0.983 / 0.998 / 0.993 of the time in all; so 11, at most 6 %, and 0.980 / 0.979 / 0.991 / 0.989. Of 52360 launches, deep narrow and wide
    // shallow ones among them, 807 were more than 3 % slower (bf16 1792 x 16384 at 864 rows 56.8 -> 89.7, 768 x 15104 at 1303 41.9 -> 52.6; at most
    // 1.8 times); with the lines below 139 (41 of them bf16 in the place of 256 rows, at most 1.5 times: 35 and 49 tiles cut seven and five ways),
    // 0.957 / 0.959 / 0.986 / 0.960 / 0.964 of the time (bf16, its SwiGLU front, FP8, NVFP4, its front; the best each time 0.949 / 0.950 / 0.982 /
    // 0.953 / 0.952). All of these with FP8's loop and heights, the reduce launches and the epilogues of before, and FP8 with a margin of 0.9 for
    // short K.
    const FeGemmSchedule lower = low(pick);
    if (p.tile) {
        // (Of an NVFP4 SwiGLU front with 16..23 k tiles, which small tiles may cut in two only, lower ones also with fewer programs: 45 launches of
        // up to 16 tiles 0.82 of the small tiles' time; with 24..31, three pieces, 1.15, and of plain linears of 20..23 1.14.)
        if (ktiles < 12 || (2 * lower.split.programs() < cus && !(opt.nvfp4_front && ktiles >= 16 && ktiles < 24))) return p;
        // Dense weights (bf16, FP8) in fewer lower tiles than a quarter of the CUs: deep narrow linears, which small tiles cut finer than eight
        // pieces of a lower one (bf16: 826 launches 1.16 times the small tiles' time, from there on 0.90). More lower tiles than CUs and short K:
        // rounds of them want a clearer gain (48 of FP8 1.01, bf16 past 0.9 level; not so from 24 k tiles on: 5120 x 17408 at 559 rows, NVFP4 block
        // 290 us with them, 305 without).
        const uint32_t tiles = tiles_of(pick);
        if (!small_b && 4 * tiles < cus) return p;
        // FP8, whose heights leave out what a cut and short K cost: not where every lower tile is cut, unless one is as high as the rows (small
        // tiles, us -> lower ones: 5120 x 17408 at 1100 / 1216 rows 88.6 -> 91.7, 92.7 -> 103.6, 5120 x 6144 at 512 25.0 -> 28.5, 2048 x 8192 at 1536
        // 32.9 -> 35.4; 70 launches 0.95 to 1.14 of the small tiles' time; one row tile: 18944 x 8448 at 155 53.5 -> 45.9). A few cut tiles behind a
        // whole round are ahead (34816 x 5120 at 250 82.8 -> 66.5). And the clearer gain for short K at any count: with fewer tiles than CUs 8192 x
        // 2048 at 1024 rows takes 19.7 -> 20.7 where the ratio is 0.99, at 1100 rows 23.7 -> 20.9 where it is 0.46 (ten launches between 0.46 and
        // 0.77: 0.71 to 0.96).
        if (cost.f8 && !lower.split.full && m > kFeGemmTileM[pick]) return p;
        const float margin = ktiles < 24 && (tiles > cus || cost.f8) ? cost.short_k : small_b ? 1.06f : 1.0f;  // (bf16 and FP8: what a lower tile gained is part of that margin)
        if (margin * p.us < whole * ratio) return p;
    }
    p.tile = pick, p.tiles = 0, p.splits = 1, p.big = lower, p.us = whole * ratio;
    return p;
}

// ---- the GEMM that decodes a trellis into registers (k_exl3_rgemm.hip): how a launch is spread --------------------------------
// A program takes `blocks` column blocks of 128 and 16 rg rows. The first `full` tiles are computed whole, the others by `runs` programs: as many a tile, each
// an equal part of its steps, where that comes out even, else the tiles' steps laid end to end and dealt in equal runs. Pieces of a tile meet through the
// workspace and a reduce launch.
struct FeRgemmPlan {
    uint32_t blocks = 1, rg = 16, tiles_m = 0, tiles_n = 0, full = 0, runs = 0, k = 0;
    float us = 0;
    uint32_t steps() const { return k / (blocks == 1 ? 128 : 64); }  // of a tile
    bool reduce() const { return runs && runs != tiles_m * tiles_n - full; }
};
// The rule: the cheapest by an estimate among one or two column blocks a program, the fewest row tiles of 256 rows at most or one more,
// all tiles whole, or whole rounds of the CUs (or one round fewer) and the rest in one run a CU or in 2, 3, .. runs a tile. Fitted to 10600 timings
// of 589 single linears (2 to 8 bits, 65..2303 rows, every plan that looked near the best; launches replayed from a graph, without the rotation): half of them
// within 7 %, nine tenths within 19 %. The plan it picks takes 1.2 % more than the fastest one timed (geometric mean; 5 of 589 more than 10 %, at most 17 %).
// Its terms: a step's matrix instructions and decode; a program's start, and its output rotation or piece by the tile's size; runs that end inside a tile,
// which meet their neighbours' inputs at another depth of K, so that with several row tiles each reads them past L2, the more the larger they are; the
// reduce launch by the pieces' bytes (more a byte where short runs leave them all at once) and by its rounds of eight. Forced block counts and pieces: for
// tests.
inline FeRgemmPlan fe_rgemm_plan(uint32_t rows, uint32_t k, const uint32_t *n, uint32_t count, uint32_t cus, size_t part_bytes, uint32_t force_blocks,
                                 uint32_t force_pieces) {
    FeRgemmPlan best;
    best.us = 1e30f;
    for (uint32_t blocks = 1; blocks <= 2; blocks++) {
        // Two column blocks from 129 rows on: their lowest tile is 160 rows, whose last pieces lie, by the scalar offset alone, past the end of fewer
        // rows, and the range check is only stated for scalar offsets inside the buffer. (Every other tile has more than rg - 2 row groups.)
        if (blocks != (rows <= 128 ? 1 : force_blocks ? force_blocks : blocks)) continue;
        for (uint32_t cut_m = (rows + 255) / 256; cut_m <= (rows + 255) / 256 + 1; cut_m++) {
            FeRgemmPlan p;
            p.k = k, p.blocks = blocks, p.rg = std::max(((rows + cut_m - 1) / cut_m + 31) / 32 * 2, blocks == 1 ? 6u : 10u);
            p.tiles_m = (rows + 16 * p.rg - 1) / (16 * p.rg);
            for (uint32_t i = 0; i < count; i++) p.tiles_n += (n[i] / 128 + blocks - 1) / blocks;
            const size_t slot = (size_t)blocks * p.rg * 16 * 512;
            const uint32_t tiles = p.tiles_m * p.tiles_n, all = p.steps(), slots = (uint32_t)(part_bytes / slot);
            const float step = (0.63f + 0.06f * (float)p.rg) * (blocks == 2 ? 0.91f : 1.0f), ends = 0.24f * (float)(p.rg * blocks);
            const float apart = p.tiles_m > 1 ? 0.35f * (0.3f + std::min(1.0f, (float)rows * (float)k * 2.0f / 32e6f)) : 0.0f;
            auto consider = [&](uint32_t full, uint32_t runs) {
                const uint32_t rest = tiles - full, rounds = (full + cus - 1) / cus;
                if (rest && (!runs || runs > rest * all || runs + rest > slots)) return;
                float t = full ? 2.7f + 12.0f * (float)(rounds - 1) + (float)rounds * (ends + (float)all * step) : -2.6f;
                if (rest) {
                    const uint32_t len = (rest * all + runs - 1) / runs, pieces = (runs + rest - 1) / rest;
                    const bool even = runs % rest == 0;
                    t += 5.3f + ends + (float)len * step;
                    if (!even) t += 6.3f * (float)((len + all - 2) / all) + (float)len * step * apart;
                    if (runs != rest)
                        t += 1e-6f * (float)slot * (float)(even ? runs : runs + rest) * (0.2f + 0.45f / (1.0f + (float)len / 3.0f)) + 2.2f * (float)((pieces + 6) / 8);
                }
                if (t < best.us) best = p, best.full = full, best.runs = rest ? runs : 0, best.us = t;
            };
            const uint32_t forced = std::min(tiles * std::min(force_pieces, all), slots > tiles ? slots - tiles : 0);
            if (force_pieces > 1 && forced > tiles) {
                consider(0, forced);
                continue;
            }
            consider(tiles, 0);
            for (uint32_t back = 0; back <= 1 && back <= tiles / cus && !force_pieces; back++) {
                const uint32_t full = (tiles / cus - back) * cus, rest = tiles - full;
                if (!rest) continue;
                consider(full, cus);
                for (uint32_t s = 2; s * rest <= cus; s++) consider(full, s * rest);
            }
        }
    }
    return best;
}

// Of the two GEMMs that decode a trellis, whether the one that decodes into registers takes `count` linears in one launch: both estimates, the other GEMM's
// (its launches together) with what the comparison of 589 single linears showed it to leave out, 12 us a round of programs after the first, and to count twice,
// 3 us of the reduce launch of cut small tiles. On those linears the rule's pick takes 0.3 % more than the faster of the two (geometric mean); 6 of them take
// more than 5 % longer than through the other GEMM (at most 15 %), 7 more than 5 % longer than through this one (at most 13 %).
inline float fe_rgemm_other_us(const FeGemmPlan &p, uint32_t cus) {
    const uint32_t programs = p.tile ? p.tiles * p.splits : p.big.programs, round = p.tile == 2 ? 2 * cus : cus;
    return p.us + 12.0f * (float)((std::max(programs, 1u) - 1) / round) - (p.tile && p.splits > 1 ? 3.0f : 0.0f);
}
inline bool fe_rgemm_takes(const FeRgemmPlan &p, float other_us, uint32_t count) { return p.us <= other_us + 3.0f * (float)count; }

constexpr uint32_t fe_reduce_threads(uint32_t tile) { return tile == 2 ? 256 : 512; }  // of the reduce kernels, half a wavefront a row (g8_reduce_rows of gemm8.h)
// Launches a plan. gemm(form, programs, sched): form 0 = 256 x 256 one piece a program, 1 = stream-K, 2, 3 = tile 1, 2;
// 4, 5, 6 = tile 3, 4, 5; reduce(tile, grid, first, splits): the reduce kernel of a tile, for the tiles from `first` on.
template <class Gemm, class Reduce>
int fe_gemm_launch(const FeGemmPlan &p, Gemm gemm, Reduce reduce) {
    const uint32_t reduce_grid = kFeGemmTileM[p.tile] / (fe_reduce_threads(p.tile) / 32) * (kFeGemmTileN[p.tile] / 128);  // workgroups a tile
    if (p.tile == 1 || p.tile == 2) {
        FeGemmSchedArgs a = p.big.args;
        a.full_tiles = 0, a.splits = p.splits, a.sk_base = a.sk_rem = 0;
        FE_TRY(gemm(p.tile + 1, p.tiles * p.splits, a));
        if (p.splits > 1) FE_TRY(reduce(p.tile, p.tiles * reduce_grid, 0u, p.splits));
        return 0;
    }
    FE_TRY(gemm(p.big.stream_k ? 1u : p.tile ? p.tile + 1 : 0u, p.big.programs, p.big.args));
    if (!p.big.stream_k && p.big.split.cut())
        FE_TRY(reduce(p.tile, p.big.split.cut() * reduce_grid, p.big.split.full, p.big.split.splits));
    return 0;
}

// ---- gate, up and SwiGLU of decode rows over plain bf16 weights (fe_bf16.cpp) ---------------------------------------------------
// Whether fe_bf16_gemv_swiglu does what two fe_bf16_linear_forward into big ([m][inter] each) and fe_route_silu_mul into act do: all rows go through
// the GEMV in one pass, the operands are what those take, and act lies apart from what other programs still read. (Two launches less: see
// gemv_bf16_body for both sides.) over_gemm: the call would otherwise take the GEMM with SwiGLU in its epilogue over interleaved weights, which is
// ahead of it at some row counts where gate, up and SwiGLU in three launches are not.
struct fe_bf16_kernels;
bool fe_bf16_gemv_swiglu_takes(const fe_bf16_kernels *kern, fe_devptr_t big, fe_devptr_t act, fe_devptr_t x, fe_devptr_t gate, fe_devptr_t up, uint32_t m, uint32_t inter,
                               uint32_t k, uint32_t dec, bool over_gemm);
int fe_bf16_gemv_swiglu(const fe_bf16_kernels *kern, fe_stream_t s, fe_devptr_t act, fe_devptr_t x, fe_devptr_t gate, fe_devptr_t up, uint32_t m, uint32_t inter, uint32_t k);

// ---- the GEMVs over programs of 8 CO columns and all of K, bf16 and FP8 ---------------------------------------------------------
// Their forms: rows / 8, and columns / 8 of a program (those whose stages fit LDS)
constexpr uint32_t kGemvRowForms[5] = {1, 2, 4, 6, 8}, kGemvColForms[7] = {1, 2, 3, 4, 5, 6, 9};
constexpr bool gemv_form(uint32_t xo, uint32_t co) { return 12 * (co + xo) <= 160; }
constexpr uint32_t gemv_row_form(uint32_t m) { return m <= 8 ? 0 : (m + 15) / 16; }
// Bf16Gemv<XO, CO>::LDS of k_bf16.hip, and what Fp8Gemv of k_fp4.hip takes
inline uint32_t gemv_lds(uint32_t xo, uint32_t co) { return 4 * std::max(3u, std::min(20 / (co + xo), 8u)) * (co + xo) * 1024; }
// The columns that each program of a form of `most` columns takes (`whole`: those): as even as whole rounds of one program a CU allow, in steps of
// `step`; rows of a load past them repeat the last one, which a cache holds. 5120 columns are 256 programs of 20 instead of 214 of 24, 17408 of 68
// instead of 242 of 72. us, bf16 blocks (gate, up, down) of 5120 x 17408 at 8 / 12 / 48 rows 83.9 -> 82.5, 87.5 -> 85.7, 142 -> 135, of 5120 x 8704
// at 12 49.7 -> 47.1, of 1536 x 5120 at 12 15.2 -> 14.2; FP8 5120 x 17408 at 16 rows 17.3 -> 16.2, 5120 x 5120 7.6 -> 7.1. One and two rows, which
// are bound by the weights' way alone, gain nothing (bf16 3072 x 8192 27.7 -> 28.1: whole octets there), nor does NVFP4, whose octets are pieces of
// 256 bytes (5120 x 17408 at 4 rows 14.6 -> 14.9: not done there).
inline uint32_t gemv_even(uint32_t n, uint32_t most, uint32_t cus, uint32_t step, bool whole) {
    const uint32_t programs = (n + most - 1) / most;
    if (whole || 2 * programs <= cus) return most;
    const uint32_t slots = (programs + cus - 1) / cus * cus;
    return std::min(most, ((n + slots - 1) / slots + step - 1) / step * step);
}

// Which of kGemvColForms a GEMV takes. Time goes by the CU with the most columns, so the form is the one with the least of
// rounds of one program a CU times a program's loads (columns, and half the weight for the x rows, which come from L2). us, 5120
// columns of 17408 at 1 / 16 rows (640 octets of columns on 256 CUs): 2 octets 33.8 / 47.9, 3 octets 27.1 / 33.7, 4 octets
// 30.0 / 39.4; 8704 columns of 5120 at 1 / 64 rows: 4 octets 20.9 / 43, 5 octets 15.2 / 27. With one or two rows a linear
// of several octets a CU is better off with programs that start while others run: 17408 columns 27.1 us at 3 octets, 27.7 at 9.
// (One and two rows as dot products on the vector ALUs would be up to 0.4 us faster at some widths: 5120 columns of 5120 9.7 / 10.1 us against
// 10.0 / 10.2, 1024 of 5120 3.9 / 4.1 against 4.3 / 4.5; but a row's bits may not depend on the batch, and from three rows on the matrix
// instruction is far ahead.)
inline uint32_t gemv_cols(uint32_t m, uint32_t n, uint32_t k, uint32_t xo, uint32_t cus, int32_t nc) {
    const uint32_t octets = n / 8;
    uint32_t best = 0;
    uint64_t least = ~0ull;
    for (uint32_t i = 0; i < 7; i++) {
        const uint32_t co = kGemvColForms[i];
        if (i && (!gemv_form(xo, co) || 16ull * co * k >= (1ull << 32))) break;
        if (nc > 0) {
            best = i;
            if (8 * co >= (uint32_t)nc) break;
            continue;
        }
        const uint64_t rounds = (octets + co * cus - 1) / (co * cus), cost = rounds * (2 * co + xo);
        if (cost <= least) best = i, least = cost;
    }
    if (nc <= 0 && m <= 2 && best > 4) best = 2;
    return best;
}

// Whether a GEMV over programs of columns is ahead of the GEMM that would run in its place, by an estimate of both (us). The GEMV's: a start, rounds
// of programs, the weights' way from HBM, the activations' way from L2 once a program (the CU with the most; x: the form's rows, x_row: those that
// exist) and the outputs. The GEMM's: its plan's estimate and what that leaves out at so few rows, the weights' way, of bytes past what the chip's
// last cache holds once more (far: us a byte), and the outputs; pieces of K cost less than it says. margin: on what the GEMM takes. Up to `always`
// rows the GEMV in any case. beside: decode rows, which a GEMV of their own would take beside the GEMM.
struct FeGemvLine {
    uint32_t always;
    float start, round, w, x, x_row, out, gemm_start, gemm_us, gemm_w, gemm_cut, gemm_pieces, gemm_far, gemm_out, margin;
};
inline float fe_gemv_us(const FeGemvLine &c, uint32_t m, uint32_t n, uint32_t k, uint32_t steps, uint32_t cus, uint32_t even_step) {
    const uint32_t xo = kGemvRowForms[gemv_row_form(m)], co = kGemvColForms[gemv_cols(m, n, k, xo, cus, -1)], pc = gemv_even(n, 8 * co, cus, even_step, false);
    const uint32_t programs = (n + pc - 1) / pc, at_once = (gemv_lds(xo, co) <= 80 * 1024 ? 2 : 1) * cus, a_cu = (programs + cus - 1) / cus;
    return c.start + c.round * (float)((programs + at_once - 1) / at_once) + c.w * (float)n * (float)steps + (float)a_cu * (c.x * (float)(8 * xo) + c.x_row * (float)m) * (float)steps + c.out * (float)m * (float)n;
}
inline bool fe_gemv_ahead(const FeGemvLine &c, uint32_t m, uint32_t n, uint32_t k, uint32_t steps, uint32_t cus, uint32_t even_step, const FeGemmPlan &gemm, float bytes = 0.0f,
                          uint32_t beside = 0) {
    if (m <= c.always) return true;
    const uint32_t pieces = gemm.tile == 1 || gemm.tile == 2 ? gemm.splits : gemm.big.split.splits;
    const float weights = (float)n * (float)steps;
    const float t = c.gemm_start + c.gemm_us * gemm.us + c.gemm_w * weights + c.gemm_far * std::max(bytes - 250e6f, 0.0f) + c.gemm_out * (float)m * (float)n -
                    (pieces > 1 ? c.gemm_cut : 0.0f) - c.gemm_pieces * (float)pieces * (float)n;
    return fe_gemv_us(c, m, n, k, steps, cus, even_step) <= c.margin * t + (beside ? fe_gemv_us(c, beside, n, k, steps, cus, even_step) : 0.0f);
}
// FP8 (steps of 128 codes), up to 64 rows. Fitted to 17236 calls of 9..64 rows (128 .. 153600 columns, K 128 .. 76800, half of them past 40960
// columns or K 20480), half of either estimate within 5 %. Of the GEMM's time in all 0.824, 180 calls more than 3 % slower than it, at most 21 %, 30
// of them among the 11408 of up to 40960 columns and K 20480, at most 15 % (the better one each time 0.818). Fitted to those alone the rule took
// 0.829, 650 calls slower, at most 41 % (3328 x 49664 at 27 rows 32.7 -> 42.3 us, 46336 x 5376 at 28 39.5 -> 47.1); by K alone (64 rows, 40 where K
// is past 14336) wide linears of short K took up to 62 % more. us, GEMM -> GEMV at 1 / 17 / 32 / 64 rows: 17408 x 5120 24.4 -> 15.1, 25.2 -> 16.1,
// 25.8 -> 17.4, 27.7 -> 27.1; 5120 x 5120 12.0 -> 6.1, 12.5 -> 8.3, 12.7 -> 8.5, 13.3 -> 11.0; 1024 x 2816 9.7 -> 3.9, 10.2 -> 3.8, 10.2 -> 4.2, 10.7
// -> 5.7; not taken: 38784 x 384 at 56 10.4 -> 16.5, 28672 x 640 at 60 10.6 -> 15.4, 11136 x 13952 at 61 40 -> 49.
constexpr FeGemvLine kFeGemvFp8{8, 3.47f, 0.835f, 14.4e-6f, 1.544e-3f, 0.0f, 2.39e-6f, 5.01f, 0.768f, 0.68e-6f, 1.64f, -17.5e-6f, 0.0f, 1.11e-6f, 0.95f};
// bf16 (steps of 64), up to 32 rows that are no decode rows. Fitted to 21244 linears of 17..32 rows (64 .. 96000 columns, K 256 .. 19456), half of
// either estimate within 5 %. By this rule 0.832 of the GEMM's time in all, 194 more than 3 % slower than it, at most 25 % (the better one each time
// 0.824); with lines by rows times K alone (350000 up to 24 rows, 180000 up to 32) 0.862 of 18642, 2207 slower, at most 2.1 times. us, GEMM -> GEMV
// at 17 / 24 / 32 rows: 17408 x 5120 40 -> 31, 31, 32; 34816 x 5120 77 -> 58, 79 -> 60, 81 -> 62; 5120 x 5120 17 -> 13, 15, 16; 1024 x 2816 8.7 ->
// 5.4, 5.7, 6.1; not taken: 61728 x 256 at 31 7.6 -> 15.8, 55304 x 256 at 27 7.2 -> 14.5. From 33 rows on (three groups of 16) the GEMM is ahead
// wherever K is 5120 and more.
constexpr FeGemvLine kFeGemvBf16{16, 0.91f, 1.236f, 15.0e-6f, 0.962e-3f, 0.894e-3f, 1.63e-6f, 3.05f, 0.681f, 4.69e-6f, 1.084f, -5.1e-6f, 0.0987e-6f, 0.0f, 0.97f};
// bf16 gate and up (n each) in one launch against the GEMM with SwiGLU over their interleaved weights (its plan's): of 10529 calls 0.906 of the
// GEMM's time in all, 179 more than 3 % slower, at most 28 % (the better one each time 0.901); by rows times K and inter 0.942 of 2284, 410 slower,
// at most 2.4 times. us, GEMM -> GEMV: 8512 x 3584 at 21 rows 29.2 -> 21.9, 1280 x 2560 at 20 9.5 -> 7.0; not taken: 28480 x 256 at 22 7.8 -> 18.8,
// 15168 x 256 at 21 5.6 -> 9.8, 320 x 10752 at 20 12.9 -> 22.4.
constexpr FeGemvLine kFeGemvBf16Pair{16, 2.19f, 0.371f, 28.7e-6f, 2.041e-3f, 1.674e-3f, 9.58e-6f, 3.55f, 0.689f, 11.0e-6f, 1.264f, 155e-6f, 0.0639e-6f, 5.86e-6f, 0.97f};
