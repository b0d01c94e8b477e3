// MFMA GEMM core for prefill-sized M: C[BM x BN tile] = A[M][K] (16-bit, row-major, from global) times a weight tile W[N][K].
//
// 512 threads = 8 wavefronts, two a SIMD, in a WM x WN grid; a wavefront owns 16 TM rows x 16 TN columns as TM x TN
// v_mfma_f32_16x16x32 accumulators (128 registers a lane at 256 x 256). Both operands go from global memory straight into
// LDS (buffer_load ... lds, 16 bytes a lane): no staging registers and no LDS write instructions, which cost the LDS pipe
// about 17 cycles a kilobyte where the direct path costs 8. The loads of a k tile are spread evenly over the tile's MFMAs:
// the address unit takes 16 cycles for each, and a burst of them holds the wavefront's next MFMA back.
//
// What the tile loop is bound by is the board's power: the matrix pipe is busy 70 % of a bf16 launch of 2048 rows by the
// counters (first loads, last tiles and the epilogue included) and the clock settles where the power limit puts it
// (1.75..1.95 GHz on random operands). So the choices are those that take the least energy a flop:
// the 16x16x32 instruction (half the accumulator traffic a flop of 32x32x16: at the same schedule 98 against 104 us for
// 4096^3), every operand byte once through LDS. 2048 x 16384 x 5120 bf16: 225 us (1526 TFLOP/s) against 266 us for four
// wavefronts of 128 x 128 with 32x32x16 and operands staged through registers.
//
// LDS: NA stages of A (BM rows of 128 bytes) and NW stages of the weight operand; the loads run NA - 1 and NW - 1 k tiles
// ahead. A row of 128 bytes is 8 chunks of 16; chunk c of row r lies at position perm(c) ^ (r & 7). A fragment read takes
// row lane & 15, one chunk per group of 16 lanes; a 16-byte read serves the lanes {0-3, 12-15, 20-27} or {4-11, 16-19,
// 28-31} of a half wavefront in a cycle (64 banks), and those 16 need 16 different (r & 1, position) pairs: with neighbouring
// chunks in neighbouring lane groups (perm = identity) the XOR gives them; where lane group g takes chunks 2 g and 2 g + 1
// (weights expanded from packed codes, 16 codes a lane), perm swaps the two low bits of c.
#pragma once
#include <type_traits>
#include <utility>

#include "gemm_core.h"

#define G8_BK GM_BK

template <int WM_, int WN_, int TM_, int TN_>
struct G8Tile {
    static constexpr int WM = WM_, WN = WN_, TM = TM_, TN = TN_, NW = WM * WN, THREADS = 64 * NW;
    static constexpr int BM = 16 * TM * WM, BN = 16 * TN * WN;
    static constexpr int PART_FLOATS = BM * BN;
    static constexpr int PARTS = 256 * 256 / (BM * BN);  // of a tile of 256 x 256: 1 (also 224, 192, 160 x 256); 2, 4: the small tiles
    static constexpr int LA = (BM + 63) / 64, A_STAGE = LA * 64 * 128;  // loads a wavefront, LDS bytes of a k tile of A (whole loads)
    static_assert(NW == 8, "eight wavefronts");
};

// One wavefront moves 64 x 16 (4) bytes, lane l's from rs + voff + soff to LDS byte dst + 16 (4) l; dst and soff are uniform.
// Not counted by the compiler's own waits: callers wait with g8_loads_wait. What the compiler does not see inside such a statement is
// its hazards: a buffer load needs five wait states after a vector instruction (a v_readfirstlane) has written a scalar register
// that it reads, and one after m0. So the offset passes through a scalar move, which waits for it and is m0's wait state, and the
// LDS byte goes into m0 as an operand: the compiler writes that register and knows what it holds. (The resource comes from scalar code
// or stands long before the load; tests/test_code_objects.py checks the built code.)
__device__ __forceinline__ void g8_load_lds16(u32x4 rs, uint32_t dst, uint32_t voff, uint32_t soff) {
    uint32_t at;
    asm volatile("s_mov_b32 %0, %4\n\tbuffer_load_dwordx4 %2, %3, %0 offen lds"
                 : "=&s"(at)
                 : "{m0}"(__builtin_amdgcn_readfirstlane(dst)), "v"(voff), "s"(rs), "s"(__builtin_amdgcn_readfirstlane(soff))
                 : "memory");
}
__device__ __forceinline__ void g8_load_lds16_nt(u32x4 rs, uint32_t dst, uint32_t voff, uint32_t soff) {
    uint32_t at;
    asm volatile("s_mov_b32 %0, %4\n\tbuffer_load_dwordx4 %2, %3, %0 offen nt lds"
                 : "=&s"(at)
                 : "{m0}"(__builtin_amdgcn_readfirstlane(dst)), "v"(voff), "s"(rs), "s"(__builtin_amdgcn_readfirstlane(soff))
                 : "memory");
}
__device__ __forceinline__ void g8_load_lds4(u32x4 rs, uint32_t dst, uint32_t voff, uint32_t soff) {
    uint32_t at;
    asm volatile("s_mov_b32 %0, %4\n\tbuffer_load_dword %2, %3, %0 offen lds"
                 : "=&s"(at)
                 : "{m0}"(__builtin_amdgcn_readfirstlane(dst)), "v"(voff), "s"(rs), "s"(__builtin_amdgcn_readfirstlane(soff))
                 : "memory");
}
// All but the N youngest of the wavefront's vector memory operations are done, and its LDS operations are.
template <int N>
__device__ __forceinline__ void g8_loads_wait() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory");
}
// Workgroup barrier without the compiler's wait for every load in flight.
__device__ __forceinline__ void g8_barrier() {
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}
__device__ __forceinline__ u32x4 g8_rsrc(const void* p, uint32_t bytes) {
    const uint64_t a = (uint64_t)p;
    return (u32x4){(uint32_t)a, (uint32_t)(a >> 32) & 0xffffu, bytes, 0x00020000u};
}
__device__ __forceinline__ uint32_t g8_lds_addr(const void* p) {
    return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)p;
}
// Byte offset of row `row` of an operand of m rows of `pitch` bytes. Rows past m lie out of the resource's range and read zero: what they would
// multiply is never stored, and zeros take less of the board's power, which is what bounds the loop. (Operands of 2 GB and more, whose range such an
// offset could meet: row m - 1 again.) ZERO false: row m - 1 again in any case (the stream-K forms, which meet few such rows: with the other offsets
// their loops of 256 registers are 1 % slower). at: byte of the lane's piece in the row.
template <bool ZERO>
__device__ __forceinline__ uint32_t g8_row(uint32_t row, uint32_t m, uint32_t pitch, uint32_t at) {
    const uint32_t off = (row < m ? row : m - 1) * pitch + at;
    return ZERO && row >= m && m * pitch <= 0x7fff0000u ? 0x80000000u : off;
}
// chunk position <-> chunk (its own inverse): identity, or the two low bits swapped
template <bool PERM>
__device__ __forceinline__ constexpr uint32_t g8_perm(uint32_t c) {
    return PERM ? (c & 4) | ((c & 1) << 1) | ((c >> 1) & 1) : c;
}

// Where the q-th of n side operations goes among the matrix instructions x0 .. x1 - 1 of a slice: spread evenly. What is issued
// between two matrix instructions of a wavefront runs in the pipe's shadow; in a lump it does not (both wavefronts of a SIMD pass the
// same barrier and would reach the lump together).
__device__ __forceinline__ constexpr int g8_at(int q, int n, int x0, int x1) { return x0 + q * (x1 - x0) / n; }

// f(0) .. f(N - 1) with constant arguments (the compiler gives up unrolling the largest of these loops by itself)
template <class F, int... I>
__device__ __forceinline__ void g8_for_(F f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void g8_for(F f) {
    g8_for_(f, std::make_integer_sequence<int, N>{});
}

// Loads that may still be in flight at the barrier of a tile, with LA loads of A (NA stages) issued behind the barrier and LB of W
// (NW stages) in front of it each tile: those issued after the later one of the next tile's A and W. And at the start of the
// loop, where the first tile's have to be there.
constexpr int g8_flight(int LA, int NA, int LB, int NW) { return NW > NA ? (NA - 1) * LB + (NA - 2) * LA : (NW - 2) * (LA + LB); }
constexpr int g8_flight0(int LA, int NA, int LB, int NW) { return NW > NA ? (NA - 1) * (LA + LB) : (NW - 1) * LA + (NW - 2) * LB; }

// Weight operand already in 16-bit form: rows of 64 values a k tile. voff[j]: byte offset of the lane's 16-byte piece j (row
// 8 (wave + 8 j) + lane / 8, position lane & 7) at k tile 0; k tiles are kstep bytes apart. (dense_setup_rows / _image.)
template <class T>
struct G8Dense {
    static constexpr bool kRaw = false, kPerm = false;
    static constexpr int STAGE = T::BN * 128, LOADS = T::BN / 64;
    u32x4 rs;
    uint32_t voff[LOADS], kstep;
    // row-major weights [n][k]: rows past n repeat row n - 1 (their columns are never stored)
    __device__ __forceinline__ void rows(const void* w, uint32_t n, uint32_t k, uint32_t n0) {
        const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
        rs = g8_rsrc(w, n * k * 2);
        kstep = 128;
#pragma unroll
        for (int j = 0; j < LOADS; j++) {
            const uint32_t r = 8 * (wave + 8 * j) + (lane >> 3), g = n0 + r < n ? n0 + r : n - 1;
            voff[j] = (g * k + ((lane & 7) ^ (r & 7)) * 8) * 2;
        }
    }
    __device__ __forceinline__ void issue(uint32_t kt, uint32_t dst, int j) const { g8_load_lds16(rs, dst + j * 8192, voff[j], kt * kstep); }
};

// acc[i][j]: weight rows (output columns) 16 (wn TN + j) + 4 (lane >> 4) + e, activation row 16 (wm TM + i) + (lane & 15).
// k tiles kt0 .. kt0 + ktiles - 1. a: 16-bit values [m][lda]; rows past m read zero (ZERO) or
// repeat row m - 1 (g8_row). lds: the start of the dynamic LDS.
//
// One k tile is two slices of 32 k. A slice walks the TN columns of fragments (outer), TM MFMAs each; the outer fragment's
// register is refilled for the next slice as soon as its MFMAs are issued, the TM inner fragments are double-buffered. The
// barrier sits between the slices: by then every wavefront has this tile's fragments in registers (this tile's LDS stages
// are free for the k tiles NA / NW ahead) and the loads of tile kt + 1 have been waited for. Slice 0 issues the weight loads,
// slice 1 those of A.
template <class T, int NA, int NW, bool BF16, bool ZERO, class W>
__device__ __forceinline__ void g8_mainloop(const void* a, uint32_t lda, uint32_t m, uint32_t kt0, uint32_t ktiles, uint32_t m0,
                                            const W& wo, unsigned char* lds, f32x4 (&acc)[T::TM][T::TN]) {
    constexpr int TM = T::TM, TN = T::TN, LA = T::LA, LB = W::LOADS, A_STAGE = T::A_STAGE, W_AT = NA * A_STAGE;
    static_assert(NA >= 2 && NW >= 2 && g8_flight0(LA, NA, LB, NW) < 64, "loads in flight");
    static_assert(W_AT + NW * W::STAGE <= 160 * 1024, "LDS");
    const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t wm = wave / T::WN, wn = wave % T::WN;
    const u32x4 ra = g8_rsrc(a, m * lda * 2);
    uint32_t va[LA];
#pragma unroll
    for (int j = 0; j < LA; j++) {
        const uint32_t r = 8 * (wave + 8 * j) + (lane >> 3);
        va[j] = g8_row<ZERO>(r < T::BM ? m0 + r : m, m, lda * 2, (g8_perm<W::kPerm>((lane & 7) ^ (r & 7))) * 16);
    }
    const uint32_t base = g8_lds_addr(lds) + wave * 1024;
    auto ktc = [&](uint32_t kt) { return kt0 + (kt < ktiles ? kt : ktiles - 1); };  // past the end: the last tile again, never used
    auto load_a = [&](uint32_t kt, uint32_t st, int j) { g8_load_lds16(ra, base + st * A_STAGE + j * 8192, va[j], ktc(kt) * 128); };
    auto load_w = [&](uint32_t kt, uint32_t st, int j) { wo.issue(ktc(kt), base + W_AT + st * W::STAGE, j); };
    auto next = [](uint32_t st, uint32_t n) { return st + 1 == n ? 0u : st + 1; };

    const uint32_t fr = lane & 15, fc = lane >> 4;
    uint32_t foff[2];
#pragma unroll
    for (int kk = 0; kk < 2; kk++) foff[kk] = fr * 128 + (((4 * kk + fc) ^ (fr & 7)) << 4);
    const unsigned char* pa = lds + wm * TM * 2048;
    const unsigned char* pw = lds + W_AT + wn * TN * 2048;
    f16x8 fa[2][TM], fw[TN];
    auto rd_a = [&](int set, uint32_t st, int kk, int i) { fa[set][i] = *(const f16x8*)(pa + st * A_STAGE + 2048 * i + foff[kk]); };
    auto rd_w = [&](uint32_t st, int kk, int j) { fw[j] = *(const f16x8*)(pw + st * W::STAGE + 2048 * j + foff[kk]); };
    auto mfma = [&](int set, int i, int j) {
        if constexpr (BF16)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, fw[j]), __builtin_bit_cast(bf16x8, fa[set][i]),
                                                                 acc[i][j], 0, 0, 0);
        else
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fw[j], fa[set][i], acc[i][j], 0, 0, 0);
    };
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};

    // prologue: the loads in the order of the loop's own ([W in slice 0, A in slice 1] a tile), as of tiles before the first
#pragma unroll
    for (int t = -(NA > NW - 1 ? NA : NW - 1); t < 0; t++) {
        if (t - 1 + NW >= 0) {
#pragma unroll
            for (int j = 0; j < LB; j++) load_w(t - 1 + NW, t - 1 + NW, j);
        }
        if (t + NA >= 0) {
#pragma unroll
            for (int j = 0; j < LA; j++) load_a(t + NA, t + NA, j);
        }
    }
    g8_loads_wait<g8_flight0(LA, NA, LB, NW)>();
    g8_barrier();
#pragma unroll
    for (int i = 0; i < TM; i++) rd_a(0, 0, 0, i);
#pragma unroll
    for (int j = 0; j < TN; j++) rd_w(0, 0, j);

    uint32_t sa = 0, sw = 0, sw_in = NW - 1;  // stages of tile kt; the weight stage that slice 0 of tile kt fills
    for (uint32_t kt = 0; kt < ktiles; kt++) {
        const uint32_t sa1 = next(sa, NA), sw1 = next(sw, NW);
#pragma unroll
        for (int kk = 0; kk < 2; kk++) {
            if (kk == 1) {
                g8_loads_wait<g8_flight(LA, NA, LB, NW)>();
                g8_barrier();
            }
            const uint32_t ra_st = kk ? sa1 : sa, rw_st = kk ? sw1 : sw;
            constexpr int MF = TM * TN;
#pragma unroll
            for (int x = 0; x < MF; x++) {
                const int j = x / TM, i = j & 1 ? TM - 1 - x % TM : x % TM;
                mfma(kk, i, j);
                bool side = x % TM == TM - 1;
                if (side) rd_w(rw_st, kk ^ 1, j);
#pragma unroll
                for (int q = 0; q < TM; q++)
                    if (g8_at(q, TM, 0, MF / 2) == x) rd_a(kk ^ 1, ra_st, kk ^ 1, q), side = true;
                const int n = kk ? LA : LB;
#pragma unroll
                for (int q = 0; q < n; q++)
                    if (g8_at(q, n, 1, MF) == x) {
                        side = true;
                        if (kk == 0)
                            load_w(kt + NW - 1, sw_in, q);
                        else
                            load_a(kt + NA, sa, q);
                    }
                if (side) __builtin_amdgcn_sched_barrier(0);
            }
        }
        sa = sa1, sw_in = sw, sw = sw1;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();  // the stages are free for the epilogue
}

// Hands the wavefront's accumulators out row by row: 16 rows at a time pass through the wavefront's own LDS slab so that
// LPR = 4 TN consecutive lanes hold the wavefront's 16 TN columns of one row, 4 a lane. U passes of 64 / LPR rows are in
// flight together: transform(v[U][4], lane in row) works on all of them at once (no branches), then
// store(row in 0 .. 16 TM - 1, lane in row, v[4], what ahead(row, lane in row) returned) is called for each. ahead: what store needs of memory, asked
// for 16 rows at a time in front of the first of them: behind a store the next load waits for it (NVFP4 stream-K, 2048 rows of 5120 x 17408 with a
// residual 310 -> 300 us, FP8 185 -> 177.5). No workgroup barrier: a slab belongs to its wavefront.
template <class T, class Transform, class Ahead, class Store>
__device__ __forceinline__ void g8_epilogue(f32x4 (&acc)[T::TM][T::TN], unsigned char* lds, Transform transform, Ahead ahead, Store store) {
    constexpr int LPR = 4 * T::TN, RP = 64 / LPR, PITCH = 16 * T::TN + 4, U = 16 / RP < 4 ? 16 / RP : 4, PASSES = 16 / RP;
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6, fr = lane & 15, fc = lane >> 4;
    float* slab = (float*)(lds + wave * (16 * PITCH * 4));
    const uint32_t lr = lane / LPR, lc = lane % LPR;
    typedef decltype(ahead(0u, 0u)) Old;
    Old old[PASSES];
#pragma unroll
    for (int i = 0; i < T::TM; i++) {
#pragma unroll
        for (int q = 0; q < PASSES; q++) old[q] = ahead(16 * i + RP * q + lr, lc);
#pragma unroll
        for (int j = 0; j < T::TN; j++) *(f32x4*)(slab + fr * PITCH + 16 * j + 4 * fc) = acc[i][j];
        gm_slab_sync();
#pragma unroll
        for (int q0 = 0; q0 < PASSES; q0 += U) {
            float v[U][4];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const f32x4 t = *(const f32x4*)(slab + (RP * (q0 + u) + lr) * PITCH + 4 * lc);
                v[u][0] = t[0], v[u][1] = t[1], v[u][2] = t[2], v[u][3] = t[3];
            }
            transform(v, lc);
            // All of them have arrived from here on, also those of rows that are not stored: a load left in flight would have the next segment of a
            // stream-K form wait for everything at its start, its own first k tiles too (FP8, 2048 rows of 5120 x 17408 without a residual 169 ->
            // 172.5 us).
            if constexpr (!std::is_empty<Old>::value) {
#pragma unroll
                for (int u = 0; u < U; u++) asm volatile("" : "+v"(old[q0 + u]));
            }
#pragma unroll
            for (int u = 0; u < U; u++) store(16 * i + RP * (q0 + u) + lr, lc, v[u], old[q0 + u]);
        }
        gm_slab_sync();
    }
}
struct G8Nothing {};  // for epilogues that ask for nothing ahead
__device__ __forceinline__ auto g8_ask_nothing() {
    return [](uint32_t, uint32_t) { return G8Nothing{}; };
}

// a: its rows of 16 lanes 0, 2 and those of b, alternating; b: rows 1, 3 likewise. And the same with halves of the wavefront.
__device__ __forceinline__ void g8_swap16(uint32_t& a, uint32_t& b) {
    const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    a = r[0], b = r[1];
}
__device__ __forceinline__ void g8_swap32(uint32_t& a, uint32_t& b) {
    const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = r[0], b = r[1];
}
typedef uint32_t u32x4_a8 __attribute__((ext_vector_type(4), aligned(8)));

// The wavefront's accumulators as bf16 rows added to a residual: c = bf16(bf16(sum) + res), row stride ldc, both pointers at its first row and
// column; pack(sums, column tile) -> two words of bf16. A lane holds 4 columns of a row in every column tile and trades the half of two tiles with
// the lane 16 away: 8 neighbouring columns a lane, without LDS. rows, cols: those that exist from there on (cols a multiple of 8). What a residual costs is the trip to memory: asked
// for where it is added, row piece by row piece, each load waits behind the store before it, 10 us a launch. Asked for 16 rows ahead, us, launches
// without / with one before -> now: bf16, 2048 rows of 8192 x 256 15.0 / 25.3 -> 14.5 / 19.8, of 8192 x 4096 95 / 105 -> 95 / 99.5; FP8, 1000 rows of
// 5120 x 5120 34.2 / 40.9 -> 33.9 / 34.4, 512 of 17408 x 5120 55 / 65 -> 55 / 56; NVFP4, 2048 of 8192 x 512 23.6 / 33.1 -> 23.4 / 27.5. Through the
// slab (g8_epilogue, asked for ahead as well) the first takes 21.8; without a residual the slab's whole lines are ahead (14.5 against 15.2).
template <class T, class Pack>
__device__ __forceinline__ void g8_add_bf16(f32x4 (&acc)[T::TM][T::TN], uint16_t* c, const uint16_t* res, uint32_t ldc, uint32_t rows, uint32_t cols, Pack pack) {
    constexpr int TM = T::TM, TN = T::TN, P = TN / 2;
    const uint32_t lane = threadIdx.x & 63, fr = lane & 15, fc = lane >> 4, cc = 16 * (fc & 1) + 8 * (fc >> 1);
    auto run = [&](auto whole_tag) {
        constexpr bool WHOLE = decltype(whole_tag)::value;
        uint16_t* p = c + (size_t)fr * ldc + cc;
        const uint16_t* r = res + (size_t)fr * ldc + cc;
        auto in = [&](int i, int j) { return WHOLE || (16 * i + fr < rows && 32 * j + cc < cols); };
        u32x4 old[2][P];
        auto ask = [&](int i) {
#pragma unroll
            for (int j = 0; j < P; j++)
                if (in(i, j)) old[i & 1][j] = *(const u32x4_a8*)(r + 32 * j);
            r += (size_t)16 * ldc;
        };
        ask(0);
#pragma unroll
        for (int i = 0; i < TM; i++) {
            if (!WHOLE && 16 * i >= rows) break;
            if (i + 1 < TM) ask(i + 1);
#pragma unroll
            for (int j = 0; j < P; j++) {
                const u32x2 a = pack(acc[i][2 * j], 2 * j), b = pack(acc[i][2 * j + 1], 2 * j + 1);
                uint32_t a0 = a[0], a1 = a[1], b0 = b[0], b1 = b[1];
                g8_swap16(a0, b0), g8_swap16(a1, b1);
                if (in(i, j)) *(u32x4_a8*)(p + 32 * j) = add_bf16x8((u32x4){a0, a1, b0, b1}, old[i & 1][j]);
            }
            p += (size_t)16 * ldc;
        }
    };
    if (rows >= 16 * TM && cols >= 16 * TN)
        run(std::true_type{});
    else
        run(std::false_type{});
}

// A program's accumulators in its partial slot, as the lanes hold them: piece (i, j) of thread t at ((i TN + j) 512 + t) 16. rows: those of the tile that
// exist; groups of 16 past them are left out.
template <class T>
__device__ __forceinline__ void g8_store_partial(f32x4 (&acc)[T::TM][T::TN], float* slot, uint32_t rows) {
    const uint32_t row0 = (threadIdx.x >> 6) / T::WN * (16 * T::TM), tid = threadIdx.x;
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)slot, 0, T::PART_FLOATS * 4, 0x00020000);  // (pieces by a scalar offset)
#pragma unroll
    for (int i = 0; i < T::TM; i++)
        if (row0 + 16 * i < rows)
#pragma unroll
            for (int j = 0; j < T::TN; j++)
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, acc[i][j]), rs, tid * 16, (i * T::TN + j) * T::THREADS * 16, 0);
}

// Body of a reduce kernel: grid = cut tiles * (BM / 16) * (BN / 128), 512 threads for 16 rows x 128 columns. A wavefront sums the `splits` slots of 16 of
// the columns as g8_store_partial left them, 1 KB a slot, in split order; the sums change hands through LDS, and each half wavefront passes one row,
// 4 columns a lane, to fn(row, first column of the block, l32, v[4], ahead(row, first column, l32)); blocks outside n are left out, rows are not.
// `ahead` reads what fn needs besides the sums. What it costs is trips to memory, not bytes: so every load of a workgroup is asked for before the
// first is waited for (up to eight slots, and what `ahead` reads). Tiles of 128 x 128: 8 rows and 256 threads a workgroup, a half wavefront reads its
// row's pieces, the first slot, then four, two, one. Their launches are small (64 tiles for 215 rows of 4096 columns), and more and smaller
// workgroups are ahead there (all slots at once are not: 5120 x 5120 at 300 rows 22.1 -> 23.5): us, GEMM and reduce, 16 -> 8 rows: FP8 4096 x 4096 at
// 130 / 215 rows 16.7 / 18.1 -> 14.9 / 15.7, 2048 x 8192 at 130 17.0 -> 14.2, 1024 x 5120 at 512 15.4 -> 13.8, NVFP4 4096 x 4096 at 215 21.9 -> 19.7;
// bf16 level (1024 x 5120 at 512 17.4 -> 18.5).
template <class T, class Ahead, class RowFn>
__device__ __forceinline__ void g8_reduce_rows(const float* __restrict__ part, uint32_t m, uint32_t n, uint32_t group, uint32_t first,
                                               uint32_t splits, Ahead ahead, RowFn fn) {
    constexpr bool WHOLE = T::PARTS < 4;  // 1 KB of a slot a wavefront
    constexpr uint32_t ROWS = WHOLE ? 16 : 8, CB = T::BN / 128, PER_TILE = T::BM / ROWS * CB, PITCH = 132;
    const uint32_t t = blockIdx.x / PER_TILE, b = blockIdx.x % PER_TILE, cb = b % CB;
    const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l32 = threadIdx.x & 31, hw = threadIdx.x >> 5;
    uint32_t tm, tn;
    if constexpr (T::PARTS > 1) {
        const uint32_t tiles_m = (m + T::BM - 1) / T::BM;
        tm = t % tiles_m, tn = t / tiles_m;
    } else {
        gemm_raster(first + t, (m + T::BM - 1) / T::BM, (n + T::BN - 1) / T::BN, group, tm, tn);
    }
    const uint32_t in = b / CB * ROWS, row0 = tm * T::BM + in, n0 = tn * T::BN + cb * 128;  // in: the workgroup's first row of the tile
    if (row0 >= m || n0 >= n) return;
    if constexpr (WHOLE) {
        __shared__ __attribute__((aligned(16))) float red[16 * PITCH];
        const uint32_t rg = in / 16, c16 = 8 * cb + wave, piece = (rg % T::TM * T::TN + c16 % T::TN) * T::THREADS + (rg / T::TM * T::WN + c16 / T::TN) * 64 + lane;
        const float* p = part + (size_t)t * splits * T::PART_FLOATS + piece * 4;
        auto slot = [&](uint32_t sp) { return *(const f32x4*)(p + (size_t)(sp < splits ? sp : splits - 1) * T::PART_FLOATS); };  // (past the last: that one again, not added)
        f32x4 q[8];
#pragma unroll
        for (uint32_t i = 0; i < 4; i++) q[i] = slot(i);
        if (splits > 4) {
#pragma unroll
            for (uint32_t i = 4; i < 8; i++) q[i] = slot(i);
        }
        const auto st = ahead(row0 + hw, n0, l32);
        f32x4 sum = q[0];
#pragma unroll
        for (uint32_t i = 1; i < 8; i++)
            if (i < splits) sum += q[i];
        for (uint32_t sp = 8; sp < splits; sp++) sum += slot(sp);
        *(f32x4*)(red + (lane & 15) * PITCH + 16 * wave + 4 * (lane >> 4)) = sum;
        __syncthreads();
        const f32x4 r = *(const f32x4*)(red + hw * PITCH + 4 * l32);
        float v[4] = {r[0], r[1], r[2], r[3]};
        fn(row0 + hw, n0, l32, v, st);
    } else {
        const uint32_t row = in + hw, c4 = cb * 32 + l32, wn = c4 / (4 * T::TN), j = (c4 / 4) % T::TN, fc = c4 % 4;
        const uint32_t wm = row / (16 * T::TM), i = (row / 16) % T::TM, fr = row % 16;
        const float* p = part + (size_t)t * splits * T::PART_FLOATS + ((i * T::TN + j) * T::THREADS + (wm * T::WN + wn) * 64 + fc * 16 + fr) * 4;
        const auto st = ahead(row0 + hw, n0, l32);
        f32x4 sum = *(const f32x4*)p;
        auto add = [&](auto n_tag, uint32_t sp) {  // so many pieces in flight a lane
            constexpr uint32_t N = decltype(n_tag)::value;
            f32x4 piece[N];
#pragma unroll
            for (uint32_t q = 0; q < N; q++) piece[q] = *(const f32x4*)(p + (size_t)(sp + q) * T::PART_FLOATS);
#pragma unroll
            for (uint32_t q = 0; q < N; q++) sum += piece[q];
        };
        uint32_t sp = 1;
        for (; sp + 4 <= splits; sp += 4) add(std::integral_constant<uint32_t, 4>{}, sp);
        if (sp + 2 <= splits) add(std::integral_constant<uint32_t, 2>{}, sp), sp += 2;
        if (sp < splits) add(std::integral_constant<uint32_t, 1>{}, sp);
        float v[4] = {sum[0], sum[1], sum[2], sum[3]};
        fn(row0 + hw, n0, l32, v, st);
    }
}

// The same loop for a weight operand that is packed in memory and expanded to 16-bit values as it becomes a fragment: the
// packed k tile goes into LDS as it is (a fraction of the 16-bit form: less LDS traffic, and three stages of it are small),
// a wavefront reads its TN fragments' codes once a k tile and expands each slice's half while the matrix instructions of
// the slice before run. Lane group g = lane >> 4 expands the 16 consecutive k 16 g .. 16 g + 15 of its row: slice kk multiplies k
// 16 g + 8 kk .. + 7, so A's fragments take chunk 2 g + kk (kPerm). Outer loop: A's fragments, in place; inner: the expanded
// weights, double-buffered.
// W: kPerm = true, STAGE bytes and LOADS loads a stage, issue(kt, dst of the stage, j, wave), Raw, read(stage in LDS, row of
// the tile, lane group) -> Raw, expand(Raw, kk) -> values 8 kk .. + 7.
template <class T, int NA, int NW, bool ZERO, class W>
__device__ __forceinline__ void g8_mainloop_packed(const _Float16* a, uint32_t lda, uint32_t m, uint32_t kt0, uint32_t ktiles, uint32_t m0,
                                                   const W& wo, unsigned char* lds, f32x4 (&acc)[T::TM][T::TN]) {
    constexpr int TM = T::TM, TN = T::TN, LA = T::LA, LB = W::LOADS, A_STAGE = T::A_STAGE, W_AT = NA * A_STAGE;
    static_assert(NA >= 2 && NW >= 2 && g8_flight0(LA, NA, LB, NW) < 64, "loads in flight");
    static_assert(W_AT + NW * W::STAGE <= 160 * 1024, "LDS");
    static_assert(W::kPerm, "A's chunks");
    const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t wm = wave / T::WN, wn = wave % T::WN;
    const u32x4 ra = g8_rsrc(a, m * lda * 2);
    uint32_t va[LA];
#pragma unroll
    for (int j = 0; j < LA; j++) {
        const uint32_t r = 8 * (wave + 8 * j) + (lane >> 3);
        va[j] = g8_row<ZERO>(r < T::BM ? m0 + r : m, m, lda * 2, (g8_perm<true>((lane & 7) ^ (r & 7))) * 16);
    }
    const uint32_t base = g8_lds_addr(lds);
    auto ktc = [&](uint32_t kt) { return kt0 + (kt < ktiles ? kt : ktiles - 1); };
    auto load_a = [&](uint32_t kt, uint32_t st, int j) {
        g8_load_lds16(ra, base + wave * 1024 + st * A_STAGE + j * 8192, va[j], ktc(kt) * 128);
    };
    auto load_w = [&](uint32_t kt, uint32_t st, int j) { wo.issue(ktc(kt), base + W_AT + st * W::STAGE, j, wave); };
    auto next = [](uint32_t st, uint32_t n) { return st + 1 == n ? 0u : st + 1; };

    const uint32_t fr = lane & 15, fc = lane >> 4;
    uint32_t foff[2];
#pragma unroll
    for (int kk = 0; kk < 2; kk++) foff[kk] = fr * 128 + ((g8_perm<true>(2 * fc + kk) ^ (fr & 7)) << 4);
    const unsigned char* pa = lds + wm * TM * 2048;
    f16x8 fa[TM], fw[2][TN];
    typename W::Raw raw[TN];
    auto rd_a = [&](uint32_t st, int kk, int i) { fa[i] = *(const f16x8*)(pa + st * A_STAGE + 2048 * i + foff[kk]); };
    auto rd_raw = [&](uint32_t st, int j) { raw[j] = wo.read(lds + W_AT + st * W::STAGE, (wn * TN + j) * 16 + fr, fc); };
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = -(NA > NW - 1 ? NA : NW - 1); t < 0; t++) {
        if (t - 1 + NW >= 0) {
#pragma unroll
            for (int j = 0; j < LB; j++) load_w(t - 1 + NW, t - 1 + NW, j);
        }
        if (t + NA >= 0) {
#pragma unroll
            for (int j = 0; j < LA; j++) load_a(t + NA, t + NA, j);
        }
    }
    g8_loads_wait<g8_flight0(LA, NA, LB, NW)>();
    g8_barrier();
#pragma unroll
    for (int j = 0; j < TN; j++) rd_raw(0, j);
#pragma unroll
    for (int i = 0; i < TM; i++) rd_a(0, 0, i);
#pragma unroll
    for (int j = 0; j < TN; j++) fw[0][j] = wo.expand(raw[j], 0);

    uint32_t sa = 0, sw = 0, sw_in = NW - 1;
    for (uint32_t kt = 0; kt < ktiles; kt++) {
        const uint32_t sa1 = next(sa, NA), sw1 = next(sw, NW);
#pragma unroll
        for (int kk = 0; kk < 2; kk++) {
            if (kk == 1) {
                g8_loads_wait<g8_flight(LA, NA, LB, NW)>();
                g8_barrier();
            }
            const uint32_t ra_st = kk ? sa1 : sa;
            constexpr int MF = TM * TN;
#pragma unroll
            for (int x = 0; x < MF; x++) {
                const int i = x / TN, j = i & 1 ? TN - 1 - x % TN : x % TN;
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fw[kk][j], fa[i], acc[i][j], 0, 0, 0);
                bool side = x % TN == TN - 1;
                if (side) rd_a(ra_st, kk ^ 1, i);
                // slice 0: the second half of this tile's codes; slice 1: the next tile's codes, then their first half
                if (kk == 1) {
#pragma unroll
                    for (int q = 0; q < TN; q++)
                        if (g8_at(q, TN, 0, MF / 4) == x) rd_raw(sw1, q), side = true;
                }
#pragma unroll
                for (int q = 0; q < TN; q++)
                    if (g8_at(q, TN, kk ? MF / 2 : 1, MF) == x) fw[kk ^ 1][q] = wo.expand(raw[q], kk ^ 1), side = true;
                const int n = kk ? LA : LB;
#pragma unroll
                for (int q = 0; q < n; q++)
                    if (g8_at(q, n, 1, MF) == x) {
                        side = true;
                        if (kk == 0)
                            load_w(kt + NW - 1, sw_in, q);
                        else
                            load_a(kt + NA, sa, q);
                    }
                if (side) __builtin_amdgcn_sched_barrier(0);
            }
        }
        sa = sa1, sw_in = sw, sw = sw1;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
}

// The loop for a weight operand that is decoded by more arithmetic than a wavefront should repeat: every weight of the tile is
// decoded once, by the thread that has its words, and written into LDS as 16-bit rows (as G8Dense's). The packed words of a k tile go
// into LDS as they are (NR stages); a thread reads its words of tile t + 2 in slice 1 of tile t, decodes and writes their
// first half there and their second half in slice 0 of tile t + 1, always into the weight stage the barrier before has freed.
// NA stages of A, two of decoded weights.
// W: RAW_STAGE bytes and LOADS loads a packed stage, issue(kt, dst of the stage, j, wave), Words, read(stage in LDS) -> Words,
// prepare(words), OPS 8-value chunks a thread, pair(words, chunk, p) -> values 2 p, 2 p + 1 of a chunk as packed fp16,
// put(weight stage, chunk, 4 pairs).
template <class T, int NA, int NR, bool ZERO, class W>
__device__ __forceinline__ void g8_mainloop_decode(const _Float16* a, uint32_t lda, uint32_t m, uint32_t kt0, uint32_t ktiles, uint32_t m0,
                                                   const W& wo, unsigned char* lds, f32x4 (&acc)[T::TM][T::TN]) {
    constexpr int TM = T::TM, TN = T::TN, LA = T::LA, LR = W::LOADS, A_STAGE = T::A_STAGE, W_STAGE = T::BN * 128;
    constexpr int W_AT = NA * A_STAGE, R_AT = W_AT + 2 * W_STAGE;
    static_assert(R_AT + NR * W::RAW_STAGE <= 160 * 1024, "LDS");
    static_assert(NA >= 2 && NR >= 2 && NA <= NR + 1, "stages");
    // In slice 1 of tile t the loads of A of tile t + NA, then the packed ones of tile t + 1 + NR. At the barrier of tile t A of tile
    // t + 1 and the packed tile t + 2 have to be there: issued in tiles t + 1 - NA and t + 1 - NR.
    constexpr int FLIGHT = NR >= NA ? (NA - 2) * (LA + LR) + (NR > NA ? LR : 0) : (NR - 2) * (LA + LR);
    const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t wm = wave / T::WN, wn = wave % T::WN;
    const u32x4 ra = g8_rsrc(a, m * lda * 2);
    uint32_t va[LA];
#pragma unroll
    for (int j = 0; j < LA; j++) {
        const uint32_t r = 8 * (wave + 8 * j) + (lane >> 3);
        va[j] = g8_row<ZERO>(r < T::BM ? m0 + r : m, m, lda * 2, ((lane & 7) ^ (r & 7)) * 16);
    }
    const uint32_t base = g8_lds_addr(lds);
    auto ktc = [&](uint32_t kt) { return kt0 + (kt < ktiles ? kt : ktiles - 1); };
    auto load_a = [&](uint32_t kt, uint32_t st, int j) { g8_load_lds16(ra, base + wave * 1024 + st * A_STAGE + j * 8192, va[j], ktc(kt) * 128); };
    auto load_r = [&](uint32_t kt, uint32_t st, int j) { wo.issue(ktc(kt), base + R_AT + st * W::RAW_STAGE, j, wave); };
    auto next = [](uint32_t st, uint32_t n) { return st + 1 == n ? 0u : st + 1; };

    const uint32_t fr = lane & 15, fc = lane >> 4;
    uint32_t foff[2];
#pragma unroll
    for (int kk = 0; kk < 2; kk++) foff[kk] = fr * 128 + (((4 * kk + fc) ^ (fr & 7)) << 4);
    const unsigned char* pa = lds + wm * TM * 2048;
    const unsigned char* pw = lds + W_AT + wn * TN * 2048;
    f16x8 fa[2][TM], fw[TN];
    auto rd_a = [&](int set, uint32_t st, int kk, int i) { fa[set][i] = *(const f16x8*)(pa + st * A_STAGE + 2048 * i + foff[kk]); };
    auto rd_w = [&](uint32_t st, int kk, int j) { fw[j] = *(const f16x8*)(pw + st * W_STAGE + 2048 * j + foff[kk]); };
    auto words = [&](uint32_t st) { return wo.read(lds + R_AT + st * W::RAW_STAGE); };
    constexpr int OPS = W::OPS;
    typename W::Words w;
    u32x4 chunk;
    // pair p of the thread's share of a tile; behind the last of a chunk the chunk goes to weight stage st
    auto decode = [&](int p, uint32_t st) {
        chunk[p % 4] = wo.pair(w, p / 4, p % 4);
        if (p % 4 == 3) wo.put(lds + W_AT + st * W_STAGE, p / 4, chunk);
    };
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};

    // prologue: the loads in the order of the loop's own, as of tiles before the first, but for packed tile NR, whose stage is not free yet
#pragma unroll
    for (int t = -(NR + 1); t < 0; t++) {
        if (t + NA >= 0) {
#pragma unroll
            for (int j = 0; j < LA; j++) load_a(t + NA, t + NA, j);
        }
        if (t < -1) {
#pragma unroll
            for (int j = 0; j < LR; j++) load_r(t + 1 + NR, t + 1 + NR, j);
        }
    }
    g8_loads_wait<(NR - 2) * LR + (NR - 1 < NA ? NR - 1 : NA) * LA>();  // packed tiles 0 and 1
    g8_barrier();
    w = words(0);
    wo.prepare(w);
#pragma unroll
    for (int p = 0; p < 4 * OPS; p++) decode(p, 0);
    w = words(1);
    wo.prepare(w);
#pragma unroll
    for (int p = 0; p < 2 * OPS; p++) decode(p, 1);
    g8_loads_wait<(NA - 1) * LA + (NA - 1 < NR ? NA - 1 : NR) * LR>();  // A of tile 0
    g8_barrier();
#pragma unroll
    for (int j = 0; j < LR; j++) load_r(NR, 0, j);
#pragma unroll
    for (int i = 0; i < TM; i++) rd_a(0, 0, 0, i);
#pragma unroll
    for (int j = 0; j < TN; j++) rd_w(0, 0, j);

    uint32_t sa = 0, sr = 2 % NR, sr_in = 1;  // stage of A of tile kt; the packed stage of tile kt + 2; the one that slice 1 of tile kt fills (tile kt + 1 + NR)
    for (uint32_t kt = 0; kt < ktiles; kt++) {
        const uint32_t s = kt & 1, sa1 = next(sa, NA);  // (decoded weights: two stages)
#pragma unroll
        for (int kk = 0; kk < 2; kk++) {
            if (kk == 1) {
                g8_loads_wait<FLIGHT>();
                g8_barrier();
            }
            const uint32_t st = kk ? s ^ 1 : s;
            constexpr int MF = TM * TN;
#pragma unroll
            for (int x = 0; x < MF; x++) {
                const int j = x / TM, i = j & 1 ? TM - 1 - x % TM : x % TM;
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fw[j], fa[kk][i], acc[i][j], 0, 0, 0);
                bool side = x % TM == TM - 1;
                if (side) rd_w(st, kk ^ 1, j);
#pragma unroll
                for (int q = 0; q < TM; q++)
                    if (g8_at(q, TM, 0, MF / 2) == x) rd_a(kk ^ 1, kk ? sa1 : sa, kk ^ 1, q), side = true;
                // slice 0: the second half of tile kt + 1; slice 1: the words of tile kt + 2, then their first half
                if (kk == 1) {
                    if (x == 0) w = words(sr), side = true;
                    if (x == MF / 4) wo.prepare(w), side = true;
                }
#pragma unroll
                for (int q = 0; q < 2 * OPS; q++)
                    if (g8_at(q, 2 * OPS, kk ? MF / 4 : 0, kk ? MF : MF * 7 / 8) == x) decode(kk ? q : 2 * OPS + q, kk ? s : s ^ 1), side = true;
                if (kk == 1) {
#pragma unroll
                    for (int q = 0; q < LA + LR; q++)
                        if (g8_at(q, LA + LR, 1, MF) == x) {
                            side = true;
                            if (q < LA)
                                load_a(kt + NA, sa, q);
                            else
                                load_r(kt + 1 + NR, sr_in, q - LA);
                        }
                }
                if (side) __builtin_amdgcn_sched_barrier(0);
            }
        }
        sa = sa1, sr = next(sr, NR), sr_in = next(sr_in, NR);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
}

// The loop for 8-bit operands (e4m3 codes on both sides) on v_mfma_f32_16x16x128_f8f6f4: a k tile is 128 codes, so rows are again
// 128 bytes and stages, chunk positions and loads are those of g8_mainloop; a lane's operand of the one MFMA step of a k
// tile is chunks fc and 4 + fc of its row (both operands alike: k is a summation index only). A fragment takes 8 registers,
// so the weight fragments pass through a ring of half the columns, each refilled as many ahead, and the A fragments are refilled in
// place behind the last column. The barrier comes after the first column of the second half, the first that makes room for the next tile's. (The
// lower tiles' four columns with a ring of four, the barrier behind the first and the weights' loads in a lump in front of it: a k tile of 160 rows
// took as long as one of 256. Ring of four -> of two, us: 380 rows of 17408 x 5120 in tiles of 160 rows 46.5 -> 40.0, 777 in tiles of 224 77.9 ->
// 71.5, 600 of 5120 x 17408 in tiles of 160 62.0 -> 56.0. 128 x 128, two programs a CU: level, kept at four.)
// a: codes [m][lda] (bytes).
typedef int g8_i32x8 __attribute__((ext_vector_type(8)));
template <class T, int NA, int NW, bool ZERO>
__device__ __forceinline__ void g8_mainloop_f8(const uint8_t* a, uint32_t lda, uint32_t m, uint32_t kt0, uint32_t ktiles, uint32_t m0,
                                               const G8Dense<T>& wo, unsigned char* lds, f32x4 (&acc)[T::TM][T::TN]) {
    constexpr int TM = T::TM, TN = T::TN, R = T::PARTS == 1 ? TN / 2 : 4, LA = T::LA, LB = G8Dense<T>::LOADS, A_STAGE = T::A_STAGE, W_AT = NA * A_STAGE;
    constexpr int W_STAGE = G8Dense<T>::STAGE, BAR = TN - R;  // the barrier follows column BAR
    static_assert(TN == 2 * R || TN == R, "a ring of half or of all the columns");
    static_assert(NA >= 2 && NW >= 2 && g8_flight0(LA, NA, LB, NW) < 64, "loads in flight");
    static_assert(W_AT + NW * W_STAGE <= 160 * 1024, "LDS");
    const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t wm = wave / T::WN, wn = wave % T::WN;
    const u32x4 ra = g8_rsrc(a, m * lda);
    uint32_t va[LA];
#pragma unroll
    for (int j = 0; j < LA; j++) {
        const uint32_t r = 8 * (wave + 8 * j) + (lane >> 3);
        va[j] = g8_row<ZERO>(r < T::BM ? m0 + r : m, m, lda, ((lane & 7) ^ (r & 7)) * 16);
    }
    const uint32_t base = g8_lds_addr(lds) + wave * 1024;
    auto ktc = [&](uint32_t kt) { return kt0 + (kt < ktiles ? kt : ktiles - 1); };
    auto load_a = [&](uint32_t kt, uint32_t st, int j) { g8_load_lds16(ra, base + st * A_STAGE + j * 8192, va[j], ktc(kt) * 128); };
    auto load_w = [&](uint32_t kt, uint32_t st, int j) { wo.issue(ktc(kt), base + W_AT + st * W_STAGE, j); };
    auto next = [](uint32_t st, uint32_t n) { return st + 1 == n ? 0u : st + 1; };
    const uint32_t fr = lane & 15, fc = lane >> 4;
    uint32_t foff[2];
#pragma unroll
    for (int h = 0; h < 2; h++) foff[h] = fr * 128 + (((4 * h + fc) ^ (fr & 7)) << 4);
    const unsigned char* pa = lds + wm * TM * 2048;
    const unsigned char* pw = lds + W_AT + wn * TN * 2048;
    auto read = [&](const unsigned char* p) {
        const u32x4 lo = *(const u32x4*)(p + foff[0]), hi = *(const u32x4*)(p + foff[1]);
        return (g8_i32x8){(int)lo[0], (int)lo[1], (int)lo[2], (int)lo[3], (int)hi[0], (int)hi[1], (int)hi[2], (int)hi[3]};
    };
    g8_i32x8 fa[TM], fw[R];
    auto rd_a = [&](uint32_t st, int i) { fa[i] = read(pa + st * A_STAGE + 2048 * i); };
    auto rd_w = [&](uint32_t st, int j) { fw[j % R] = read(pw + st * W_STAGE + 2048 * j); };
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = -(NA > NW - 1 ? NA : NW - 1); t < 0; t++) {
        if (t - 1 + NW >= 0) {
#pragma unroll
            for (int j = 0; j < LB; j++) load_w(t - 1 + NW, t - 1 + NW, j);
        }
        if (t + NA >= 0) {
#pragma unroll
            for (int j = 0; j < LA; j++) load_a(t + NA, t + NA, j);
        }
    }
    g8_loads_wait<g8_flight0(LA, NA, LB, NW)>();
    g8_barrier();
#pragma unroll
    for (int i = 0; i < TM; i++) rd_a(0, i);
#pragma unroll
    for (int j = 0; j < R; j++) rd_w(0, j);
    uint32_t sa = 0, sw = 0, sw_in = NW - 1;
    for (uint32_t kt = 0; kt < ktiles; kt++) {
        const uint32_t sa1 = next(sa, NA), sw1 = next(sw, NW);
#pragma unroll
        for (int j = 0; j < TN; j++) {
#pragma unroll
            for (int x = 0; x < TM; x++) {
                const int i = j & 1 ? TM - 1 - x : x;  // formats 0, 0: e4m3 x e4m3; zero scale operands select the unscaled instruction
                acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(fw[j % R], fa[i], acc[i][j], 0, 0, 0, 0, 0, 0);
            }
            if (j == BAR) {
                if (BAR == 0) {  // no column before it: the weight loads come here
#pragma unroll
                    for (int q = 0; q < LB; q++) load_w(kt + NW - 1, sw_in, q);
                }
                g8_loads_wait<g8_flight(LA, NA, LB, NW)>();
                g8_barrier();
            }
            rd_w(j < BAR ? sw : sw1, (j + R) % TN);
            if (j == TN - 1) {
#pragma unroll
                for (int x = 0; x < TM; x++) rd_a(sa1, j & 1 ? TM - 1 - x : x);
            }
            // loads: W in the columns before the barrier, A after it
            if (j < BAR) {
#pragma unroll
                for (int q = j * LB / (BAR > 0 ? BAR : 1); q < (j + 1) * LB / (BAR > 0 ? BAR : 1); q++) load_w(kt + NW - 1, sw_in, q);
            } else {
#pragma unroll
                for (int q = (j - BAR) * LA / R; q < (j - BAR + 1) * LA / R; q++) load_a(kt + NA, sa, q);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        sa = sa1, sw_in = sw, sw = sw1;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
}

// ---- schedules -------------------------------------------------------------------------------------------------------------
// (stream-K: see gemm_core.h's account of the runs, the slots and the arrival counters; here a piece is stored and read as the
// lanes hold it, 512 threads x 16 bytes at a time)

template <class T>
__device__ __forceinline__ bool g8_sk_meet(f32x4 (&acc)[T::TM][T::TN], uint32_t p, uint32_t tile, uint32_t t0, uint32_t ktiles,
                                           uint32_t base, uint32_t rem, float* part, uint32_t part_bytes, uint32_t* counters,
                                           unsigned char* lds) {
    constexpr int TM = T::TM, TN = T::TN;
    constexpr uint32_t PIECE = T::THREADS * 16, SLOT = T::PART_FLOATS * 4;
    const uint32_t tid = threadIdx.x;
    const uint32_t first = sk_owner(t0, base, rem), last = sk_owner(t0 + ktiles - 1, base, rem);
    const uint32_t n = last - first + 1, me = p - first;
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)part, 0, part_bytes, 0x00020000);
    volatile uint32_t* flag = (volatile uint32_t*)lds;
    uint32_t* cnt = counters + tile;
    // a run's piece of a tile in which the run does not begin is the run's last segment
    auto slot_of = [&](uint32_t q) { return 2 * q + (sk_start(q, base, rem) < t0 ? 1u : 0u); };
    // (a read-modify-write, which is performed where all XCDs meet: no stale copy of the counter can answer it)
    if (tid == 0) *flag = __hip_atomic_fetch_add(cnt, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    uint32_t seen = *flag;
    __syncthreads();
    if (seen != n - 1) {  // someone is still at work: leave the piece
        const uint32_t so = slot_of(p) * SLOT;
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++)
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, acc[i][j]), rs, tid * 16, so + (i * TN + j) * PIECE, 16);
        agent_stores_wait();
        __syncthreads();
        if (tid == 0) *flag = __hip_atomic_fetch_add(cnt, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        seen = *flag;
        __syncthreads();
        if (seen != n - 1) return false;
    }
    // the pieces in piece order, starting from zero, this program's accumulators in their place
#pragma unroll
    for (int i = 0; i < TM; i++) {
        f32x4 t[TN];
#pragma unroll
        for (int j = 0; j < TN; j++) t[j] = (f32x4){0.f, 0.f, 0.f, 0.f};
        for (uint32_t q = 0; q < n; q++) {
            if (q == me) {
#pragma unroll
                for (int j = 0; j < TN; j++) t[j] += acc[i][j];
            } else {
                const uint32_t so = slot_of(first + q) * SLOT + i * TN * PIECE;
                f32x4 ld[TN];
#pragma unroll
                for (int j = 0; j < TN; j++) ld[j] = load_agent_f32x4(rs, tid * 16, so + j * PIECE);
#pragma unroll
                for (int j = 0; j < TN; j++) t[j] += ld[j];
            }
        }
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] = t[j];
    }
    if (tid == 0) __hip_atomic_store(cnt, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return true;
}

// The small tiles of a launch: tile t = column tile * row tiles + row tile, piece `piece` of its K, for the program `pid` of
// `grid` = tiles * splits. Workgroups go to the 8 XCDs round-robin; the grid is dealt so that an XCD takes a contiguous range
// of (column tile, piece, row tile), row tiles fastest: those of one column tile and piece read the same weights through one
// L2, and no XCD has more than one program more than another.
struct G8SmallWork {
    uint32_t tm, tn, tile, piece;
};
__device__ __forceinline__ G8SmallWork g8_small_work(uint32_t pid, uint32_t grid, uint32_t tiles_m, uint32_t splits) {
    const uint32_t x = pid % 8, per = grid / 8, rem = grid % 8;
    const uint32_t l = x * per + (x < rem ? x : rem) + pid / 8;
    const uint32_t tm = l % tiles_m, q = l / tiles_m;
    return G8SmallWork{tm, q / splits, q / splits * tiles_m + tm, q % splits};
}

// Runs the program's share of the schedule: main(m0, n0, kt0, ktn, acc) is one pass of the main loop over k tiles
// kt0 .. kt0 + ktn - 1 of the tile at row m0, column n0, finish(m0, n0, acc) the tile's epilogue. sc.sk_base is nonzero exactly
// when SK.
template <class T, bool SK, class Main, class Finish>
__device__ __forceinline__ void g8_schedule(const GemmSched& sc, uint32_t m, uint32_t n, uint32_t group, uint32_t ktiles,
                                            unsigned char* lds, Main main, Finish finish) {
    const uint32_t p = blockIdx.x, tiles_m = (m + T::BM - 1) / T::BM, tiles_n = (n + T::BN - 1) / T::BN;
    f32x4 acc[T::TM][T::TN];
    if constexpr (T::PARTS > 1) {
        const G8SmallWork wk = g8_small_work(p, gridDim.x, (m + T::BM - 1) / T::BM, sc.splits);
        const uint32_t kt0 = wk.piece * ktiles / sc.splits;
        main(wk.tm * T::BM, wk.tn * T::BN, kt0, (wk.piece + 1) * ktiles / sc.splits - kt0, acc);
        if (sc.splits > 1)
            g8_store_partial<T>(acc, sc.part + (size_t)(wk.tile * sc.splits + wk.piece) * T::PART_FLOATS, m - wk.tm * T::BM);
        else
            finish(wk.tm * T::BM, wk.tn * T::BN, acc);
    } else if constexpr (!SK) {
        const GemmWork wk = gemm_work(p, tiles_m, tiles_n, group, ktiles, sc.full_tiles, sc.splits);
        main(wk.tm * T::BM, wk.tn * T::BN, wk.kt0, wk.ktn, acc);
        if (wk.partial)
            g8_store_partial<T>(acc, sc.part + (size_t)wk.slot * T::PART_FLOATS, m - wk.tm * T::BM);
        else
            finish(wk.tm * T::BM, wk.tn * T::BN, acc);
    } else {
        const uint32_t whole = sc.full_tiles;  // taken whole, program p those p, p + grid, ...; the runs lie over the tiles after them
        uint32_t next_whole = p;
        uint32_t u = sk_start(p, sc.sk_base, sc.sk_rem);
        const uint32_t uend = sk_start(p + 1, sc.sk_base, sc.sk_rem);
        while (next_whole < whole || u < uend) {
            uint32_t tile, t0 = 0, kt0 = 0, ktn = ktiles;
            if (next_whole < whole) {
                tile = next_whole;
                next_whole += gridDim.x;
            } else {
                const uint32_t rel = u / ktiles;
                t0 = rel * ktiles, kt0 = u - t0;
                ktn = ktiles - kt0 < uend - u ? ktiles - kt0 : uend - u;
                tile = whole + rel;
                u += ktn;
            }
            uint32_t tm, tn;
            gemm_raster(tile, tiles_m, tiles_n, group, tm, tn);
            __syncthreads();  // the epilogue of the segment before is done with the LDS
            main(tm * T::BM, tn * T::BN, kt0, ktn, acc);
            bool fin = true;
            if (ktn != ktiles)
                fin = g8_sk_meet<T>(acc, p, tile, t0, ktiles, sc.sk_base, sc.sk_rem, sc.part, sc.part_bytes, sc.counters, lds);
            if (fin) finish(tm * T::BM, tn * T::BN, acc);
        }
    }
}
