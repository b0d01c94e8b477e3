// What the GEMM kernels share besides the tile loop (gemm8.h): the raster of output tiles, the two schedules that spread tiles
// over programs, the layout of decoded weights in memory.
#pragma once
#include "kcommon.h"

// Decoded fp16 weights in memory: blocks of 256 rows (columns of the output) x 64 k, 32 KB, 128 bytes a row; 16-byte chunk c of
// row r at position c ^ (r & 7) ^ ((r >> 3) & 1).
#define GM_BK 64
#define GM_B_BYTES (256 * GM_BK * 2)
__device__ __forceinline__ uint32_t gm_swz(uint32_t r, uint32_t c) {
    return r * 128 + ((c ^ (r & 7) ^ ((r >> 3) & 1)) << 4);
}

// Grouped raster: `group` row tiles (fastest) sweep all column tiles before the next group, so programs that run
// together share weight panels in L2 (kernels/k-fp4/src/lib.rs:298-308). Workgroups go to the 8 XCDs round-robin, so
// with a group of 8 row tiles each XCD's L2 keeps one 256-row panel of activations.
//
// group == 0 is the raster for weights that are large in memory (decoded fp16 tiles): column tiles are dealt to the XCDs
// instead, tile tn of a band of 8 to XCD tn % 8, all row tiles of it in turn, so that each weight panel is fetched into
// one L2 only and the (smaller) activations into all of them. A last band of fewer than 8 column tiles is swept column
// tile fastest.
__device__ __forceinline__ void gemm_raster(uint32_t pid, uint32_t tiles_m, uint32_t tiles_n, uint32_t group, uint32_t& tm,
                                            uint32_t& tn) {
    if (group == 0) {
        uint32_t bands = tiles_n / 8, in_bands = bands * 8 * tiles_m;
        if (pid < in_bands) {
            uint32_t q = pid / 8;
            tn = (q / tiles_m) * 8 + pid % 8;
            tm = q % tiles_m;
        } else {
            uint32_t r = tiles_n - bands * 8, idx = pid - in_bands;
            tn = bands * 8 + idx % r;
            tm = idx / r;
        }
        return;
    }
    uint32_t per_group = group * tiles_n;
    uint32_t first_m = (pid / per_group) * group;
    uint32_t gsize = tiles_m - first_m < group ? tiles_m - first_m : group;
    uint32_t r = pid % per_group;
    tm = first_m + r % gsize;
    tn = r / gsize;
}

// What a program computes on the one-piece schedule (the stream-K schedule is further down). Programs 0 .. full_tiles - 1
// take one output tile each over all of K. The remaining tiles
// (a last round that would leave most CUs idle) are cut `splits` ways along K: program full_tiles + i takes k tiles
// [kt0, kt0 + ktn) of tile full_tiles + i / splits and leaves its 256 x 256 f32 partial in slot i of the workspace; a
// reduce kernel adds the slots of a tile in split order and finishes it, so results do not depend on timing.
struct GemmWork {
    uint32_t tm, tn, kt0, ktn, slot;
    bool partial;
};

__device__ __forceinline__ GemmWork gemm_work(uint32_t pid, uint32_t tiles_m, uint32_t tiles_n, uint32_t group,
                                              uint32_t ktiles, uint32_t full_tiles, uint32_t splits) {
    GemmWork w;
    uint32_t tile = pid, split = 0, ns = 1;
    w.partial = pid >= full_tiles;
    w.slot = 0;
    if (w.partial) {
        w.slot = pid - full_tiles;
        tile = full_tiles + w.slot / splits;
        split = w.slot % splits;
        ns = splits;
    }
    gemm_raster(tile, tiles_m, tiles_n, group, w.tm, w.tn);
    w.kt0 = split * ktiles / ns;
    w.ktn = (split + 1) * ktiles / ns - w.kt0;
    return w;
}

// Orders the wavefront's own LDS writes before its own LDS reads (and the other way round): the lanes of a wavefront
// issue their LDS instructions together and the LDS executes them in order, so only the compiler has to be kept from
// moving accesses across this point. (A workgroup-scope fence would also wait for the global stores in flight, once
// per 32 rows.)
__device__ __forceinline__ void gm_slab_sync() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// ---- Stream-K schedule -------------------------------------------------------------------------------------------------
// The tiles' k tiles, laid end to end in raster order (tile-major, K ascending), are one sequence of units; program p of P
// takes the contiguous run of base = units / P of them (+ 1 for the first units % P programs), so every program does the
// same work to within one k tile whatever the tile count, and there is no mostly empty last round and no reduce launch.
// A run crosses tile boundaries: each piece of a tile (segment) is one pass of the main loop. A tile that lies in one
// run is finished there. Otherwise its pieces meet through the workspace: a piece that is not the last to arrive leaves
// its accumulators in a slot (two slots a program: one for a run's first segment, one for its last) and bumps the tile's
// arrival counter; the piece whose arrival completes the count adds the pieces in piece order, starting from zero, with
// its own accumulators in their place, and finishes the tile: the sums do not depend on which piece came last. The
// hand-off is the decode GEMV's: write-through stores, acknowledged, then a relaxed agent-scope atomic; the reader's loads
// bypass its L2; counters return to zero.
__device__ __forceinline__ uint32_t sk_start(uint32_t p, uint32_t base, uint32_t rem) { return p * base + (p < rem ? p : rem); }
// the program whose run holds unit u
__device__ __forceinline__ uint32_t sk_owner(uint32_t u, uint32_t base, uint32_t rem) {
    const uint32_t big = rem * (base + 1);
    return u < big ? u / (base + 1) : rem + (u - big) / base;
}

// How a GEMM launch is spread over its programs. Small tiles (128 x 256, 128 x 128): every tile is cut `splits` ways along K
// (g8_small_work of gemm8.h). 256 x 256 tiles, sk_base == 0: one piece a program (gemm_work: whole tiles, then the cut
// tiles, whose partials a reduce kernel adds). Otherwise stream-K: grid = the programs; the first full_tiles tiles (a
// multiple of the grid) are computed whole, round-robin, and the tiles after them are shared as runs of sk_base (+ 1 for
// the first sk_rem) k tiles; part holds two slots a program, counters one word a tile, zero at rest.
struct GemmSched {
    uint32_t full_tiles, splits, sk_base, sk_rem;
    float* part;
    uint32_t part_bytes;
    uint32_t* counters;
};
// A schedule's words as inputs of an empty statement at a kernel's start, with its other arguments: all asked for at once (a launch's arguments come
// from memory that no cache holds: left where they are first used, three to five trips one behind the other).
#define GEMM_SCHED_WORDS(s) "s"((s).full_tiles), "s"((s).splits), "s"((s).sk_base), "s"((s).sk_rem), "s"((s).part), "s"((s).part_bytes), "s"((s).counters)
