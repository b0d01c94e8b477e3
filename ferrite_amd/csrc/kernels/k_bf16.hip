// The plain bf16 weight form of the caller's linear: y[M][N] = x[M][K] . W[N][K]^T (+ residual), W row-major bf16, f32
// sums, bf16 out. A GEMM on the shared MFMA tile loop and a decode-sized GEMV (kernels/k-core/src/gemm.rs).
#include <type_traits>

#include "gemm8.h"

// 4 sums of columns at.. of one row -> bf16; where a residual is added: bf16(bf16(sum) + old) (gemm.rs:152-158).
__device__ __forceinline__ void bf16_store4(uint16_t* c, bool adds, u32x2 old, size_t at, const float (&v)[4]) {
    u32x2 o = {pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
    if (adds) {
#pragma unroll
        for (int e = 0; e < 2; e++)
            o[e] = pack_bf16x2(bf16_bits_to_f32(o[e] & 0xffff) + bf16_bits_to_f32(old[e] & 0xffff),
                               bf16_bits_to_f32(o[e] >> 16) + bf16_bits_to_f32(old[e] >> 16));
    }
    *(u32x2*)(c + at) = o;
}

// ---- GEMM ------------------------------------------------------------------------------------------------------------

typedef G8Tile<4, 2, 4, 8> Bf16Tile;    // 256 x 256
typedef G8Tile<4, 2, 2, 8> Bf16TileS1;  // 128 x 256
typedef G8Tile<4, 2, 2, 4> Bf16TileS2;  // 128 x 128, two programs a CU
typedef G8Tile<2, 4, 7, 4> Bf16TileH7;  // 224 x 256
typedef G8Tile<2, 4, 6, 4> Bf16TileH6;  // 192 x 256
typedef G8Tile<2, 4, 5, 4> Bf16TileH5;  // 160 x 256
// k tiles of A and of W in LDS: as many as the tile leaves room for
template <class T>
struct Bf16Stages {
    static constexpr int NA = T::PARTS == 2 ? 3 : 2, NW = 3, MIN_WAVES = T::PARTS == 4 ? 4 : 2;
};

// One program's share of A . W^T: main loop, then the partial slot (a tile cut along K) or finish(acc, lds, the wavefront's first row and column).
template <class T, class Finish>
__device__ __forceinline__ void bf16_gemm_program(const uint16_t* a, const uint16_t* w, uint32_t m, uint32_t n, uint32_t k, uint32_t lda,
                                                  uint32_t group_m, const GemmSched& sc, Finish finish) {
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wm = wave / T::WN, wn = wave % T::WN;
    g8_schedule<T, false>(
        sc, m, n, group_m, k / G8_BK, lds,
        [&](uint32_t m0, uint32_t n0, uint32_t kt0, uint32_t ktn, f32x4(&acc)[T::TM][T::TN]) {
            G8Dense<T> wo;
            wo.rows(w, n, k, n0);
            g8_mainloop<T, Bf16Stages<T>::NA, Bf16Stages<T>::NW, true, true>(a, lda, m, kt0, ktn, m0, wo, lds, acc);
        },
        [&](uint32_t m0, uint32_t n0, f32x4(&acc)[T::TM][T::TN]) {
            finish(acc, lds, m0 + wm * 16 * T::TM, n0 + wn * 16 * T::TN);
        });
}

// The wavefront's rows of a finished tile, from row0, col0 on.
template <class T>
__device__ __forceinline__ void bf16_tile_store(f32x4 (&acc)[T::TM][T::TN], unsigned char* lds, uint16_t* c, const uint16_t* res, uint32_t m, uint32_t n, uint32_t ldc,
                                                uint32_t row0, uint32_t col0) {
    if (row0 >= m || col0 >= n) return;
    const size_t first = (size_t)row0 * ldc + col0;
    if (res)
        g8_add_bf16<T>(acc, c + first, res + first, ldc, m - row0, n - col0, [](f32x4 v, int) { return (u32x2){pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])}; });
    else
        g8_epilogue<T>(acc, lds, [](auto&, uint32_t) {}, g8_ask_nothing(), [&](uint32_t row, uint32_t lc, float (&v)[4], G8Nothing) {
            if (row < m - row0 && 4 * lc < n - col0) bf16_store4(c, false, (u32x2){0, 0}, first + (size_t)row * ldc + 4 * lc, v);
        });
}

// C[M][ldc] = bf16(A . W^T) (+ res); A bf16 [M][lda], W bf16 [N][K]. The grid's programs share the tiles as sc says (g8_schedule);
// 512 threads, dynamic LDS as the stages of the tile take; tiles cut along K leave partials for the reduce kernel.
// K % 64 == 0, N % 8 == 0, lda % 8 == 0, ldc % 4 == 0, operands under 4 GB. NAME: 256 x 256 tiles; NAME_s1: 128 x 256;
// NAME_s2: 128 x 128. (kernels/k-core/src/gemm.rs:128-167: fe_gemm_bf16, tile 128 x 128 x 32 on mma.m16n8k16 there)
#define BF16_GEMM_KERNELS(SUFFIX, TILE)                                                                                    \
    extern "C" __global__ __launch_bounds__(512, Bf16Stages<TILE>::MIN_WAVES) void fe_gemm_bf16##SUFFIX(                   \
        uint16_t* c, const uint16_t* a, const uint16_t* w, const uint16_t* res, uint32_t m, uint32_t n, uint32_t k,        \
        uint32_t lda, uint32_t ldc, uint32_t group_m, GemmSched sc) {                                                      \
        bf16_gemm_program<TILE>(a, w, m, n, k, lda, group_m, sc, [&](auto& acc, unsigned char* lds, uint32_t row0, uint32_t col0) { \
            bf16_tile_store<TILE>(acc, lds, c, res, m, n, ldc, row0, col0);                                                \
        });                                                                                                                \
    }                                                                                                                      \
    extern "C" __global__ __launch_bounds__(512) void fe_gemm_bf16_reduce##SUFFIX(                                         \
        uint16_t* c, const float* part, const uint16_t* res, uint32_t m, uint32_t n, uint32_t ldc, uint32_t group_m,       \
        uint32_t first, uint32_t splits) {                                                                                 \
        g8_reduce_rows<TILE>(                                                                                              \
            part, m, n, group_m, first, splits,                                                                            \
            [&](uint32_t row, uint32_t n0, uint32_t l32) {                                                                 \
                const uint32_t col = n0 + 4 * l32;                                                                         \
                return res && row < m && col < n ? *(const u32x2*)(res + (size_t)row * ldc + col) : (u32x2){0, 0};         \
            },                                                                                                             \
            [&](uint32_t row, uint32_t n0, uint32_t l32, float (&v)[4], u32x2 old) {                                       \
                const uint32_t col = n0 + 4 * l32;                                                                         \
                if (row < m && col < n) bf16_store4(c, res != nullptr, old, (size_t)row * ldc + col, v);                   \
            });                                                                                                            \
    }
BF16_GEMM_KERNELS(, Bf16Tile)
BF16_GEMM_KERNELS(_s1, Bf16TileS1)
BF16_GEMM_KERNELS(_s2, Bf16TileS2)
BF16_GEMM_KERNELS(_h7, Bf16TileH7)
BF16_GEMM_KERNELS(_h6, Bf16TileH6)
BF16_GEMM_KERNELS(_h5, Bf16TileH5)

// SwiGLU over a gate|up linear whose weight rows are interleaved in blocks of 8 ([gate 0..8, up 0..8, gate 8..16, ...],
// fe_interleave_gu): of the 4 lanes that hold one 16-column block of a row, lanes 0, 1 have the 8 gate sums and lanes 2, 3
// the matching up sums. Every lane takes part (a quad exchange); lanes 0, 1 store
// act[row][8 blk + 4 (lane & 1) ..] = bf16(bf16(silu(bf16(gate))) * bf16(up)), act row stride inter = n / 2.
// (kernels/k-core/src/gemm.rs:264-279)
__device__ __forceinline__ void bf16_swiglu_store4(uint16_t* act, const float (&v)[4], uint32_t l32, bool live, uint32_t grow,
                                                   uint32_t col, uint32_t n) {
    float u[4];
#pragma unroll
    for (int e = 0; e < 4; e++) u[e] = dpp_quad_xor<2>(v[e]);
    if (!live || (l32 & 2) || col >= n) return;
    const u32x2 o = {silu_mul_bf16x2(pack_bf16x2(v[0], v[1]), pack_bf16x2(u[0], u[1])),
                     silu_mul_bf16x2(pack_bf16x2(v[2], v[3]), pack_bf16x2(u[2], u[3]))};
    *(u32x2*)(act + (size_t)grow * (n >> 1) + (col >> 4) * 8 + 4 * (l32 & 1)) = o;
}

// The same for a finished tile, without LDS: the gate sums of a column tile lie in the wavefront's lower half and the up sums in its upper half, so
// two tiles trade halves, after which every lane has gate and up of 4 features; and two such pairs trade rows of 16 lanes, after which it has 8
// features of a row. (Through the slab half of the lanes computed what they did not store: an MLP block of 1000 rows of 5120 / 17408 451 -> 444 us.)
template <class T>
__device__ __forceinline__ void bf16_tile_swiglu(f32x4 (&acc)[T::TM][T::TN], uint16_t* act, uint32_t m, uint32_t n, uint32_t row0, uint32_t col0) {
    static_assert(T::TN % 4 == 0, "two pairs of column tiles");
    if (row0 >= m || col0 >= n) return;
    const uint32_t lane = threadIdx.x & 63, fr = lane & 15, fc = lane >> 4, ct = (fc >> 1) + 2 * (fc & 1);  // of four column tiles the one whose features the lane stores
    auto pair = [](f32x4 a, f32x4 b) {
        uint32_t g0 = pack_bf16x2(a[0], a[1]), g1 = pack_bf16x2(a[2], a[3]), u0 = pack_bf16x2(b[0], b[1]), u1 = pack_bf16x2(b[2], b[3]);
        g8_swap32(g0, u0), g8_swap32(g1, u1);
        return (u32x2){silu_mul_bf16x2(g0, u0), silu_mul_bf16x2(g1, u1)};
    };
    uint16_t* p = act + (size_t)(row0 + fr) * (n >> 1) + (col0 >> 1) + 8 * ct;
#pragma unroll
    for (int i = 0; i < T::TM; i++) {
        if (16 * i >= m - row0) break;
#pragma unroll
        for (int j = 0; j < T::TN; j += 4) {
            const u32x2 x = pair(acc[i][j], acc[i][j + 1]), y = pair(acc[i][j + 2], acc[i][j + 3]);
            uint32_t x0 = x[0], x1 = x[1], y0 = y[0], y1 = y[1];
            g8_swap16(x0, y0), g8_swap16(x1, y1);
            if (16 * i + fr < m - row0 && 16 * (j + ct) < n - col0) *(u32x4_a8*)(p + 8 * j) = (u32x4){x0, x1, y0, y1};
        }
        p += (size_t)8 * n;
    }
}

// act[M][N / 2] = SwiGLU(A . W^T) for interleaved gate|up weights W [N][K], N % 16 == 0: fe_gemm_bf16 with the epilogue
// above, and its reduce kernels. (kernels/k-core/src/gemm.rs:264-279: fe_gemm_swiglu)
#define BF16_SWIGLU_KERNELS(SUFFIX, TILE)                                                                                  \
    extern "C" __global__ __launch_bounds__(512, Bf16Stages<TILE>::MIN_WAVES) void fe_gemm_bf16_swiglu##SUFFIX(            \
        uint16_t* act, const uint16_t* a, const uint16_t* w, uint32_t m, uint32_t n, uint32_t k, uint32_t lda,             \
        uint32_t group_m, GemmSched sc) {                                                                                  \
        bf16_gemm_program<TILE>(a, w, m, n, k, lda, group_m, sc, [&](auto& acc, unsigned char* lds, uint32_t row0, uint32_t col0) { \
            bf16_tile_swiglu<TILE>(acc, act, m, n, row0, col0);                                                            \
        });                                                                                                                \
    }                                                                                                                      \
    extern "C" __global__ __launch_bounds__(512) void fe_gemm_bf16_swiglu_reduce##SUFFIX(                                  \
        uint16_t* act, const float* part, uint32_t m, uint32_t n, uint32_t group_m, uint32_t first, uint32_t splits) {      \
        g8_reduce_rows<TILE>(part, m, n, group_m, first, splits, [](uint32_t, uint32_t, uint32_t) { return 0u; },          \
                             [&](uint32_t row, uint32_t n0, uint32_t l32, float (&v)[4], uint32_t) {                       \
                                 bf16_swiglu_store4(act, v, l32, row < m, row, n0 + 4 * l32, n);                           \
                             });                                                                                           \
    }
BF16_SWIGLU_KERNELS(, Bf16Tile)
BF16_SWIGLU_KERNELS(_s1, Bf16TileS1)
BF16_SWIGLU_KERNELS(_s2, Bf16TileS2)
BF16_SWIGLU_KERNELS(_h7, Bf16TileH7)
BF16_SWIGLU_KERNELS(_h6, Bf16TileH6)
BF16_SWIGLU_KERNELS(_h5, Bf16TileH5)

// dst row 16 b + i = gate row 8 b + i for i < 8, up row 8 b + i - 8 otherwise: the weight layout of fe_gemm_bf16_swiglu.
// grid 2 inter, 256 threads; k % 8 == 0. (kernels/k-core/src/gemm.rs:281-296: fe_interleave_gu)
extern "C" __global__ __launch_bounds__(256) void fe_interleave_gu(uint16_t* dst, const uint16_t* gate, const uint16_t* up,
                                                                   uint32_t k) {
    const uint32_t r = blockIdx.x, b = r / 16, i = r % 16;
    const uint16_t* src = i < 8 ? gate + (size_t)(b * 8 + i) * k : up + (size_t)(b * 8 + i - 8) * k;
    uint16_t* d = dst + (size_t)r * k;
    for (uint32_t j = threadIdx.x; j < k / 8; j += 256) *((u32x4*)d + j) = *((const u32x4*)src + j);
}

// ---- GEMV (1..64 rows) -----------------------------------------------------------------------------------------------

// y[r][n] = bf16(x[r][:] . W[n][:]) (+ res) for r < m <= 8 XO. grid ceil(N / pc), 256 threads: a program takes pc <= 8 CO columns (gemv_even) over
// all of K, its four wavefronts a quarter of K's steps of 64 each; a wavefront adds its products in v_mfma_f32_16x16x32_bf16 in
// ascending k, the four sums are added in order. So a row's bits depend on K only, neither on the other rows nor on XO or
// CO: the host picks them by the row count and the shape, where the reference picks between two kernels by the shape.
// K % 64 == 0, N % 8 == 0, lda % 8 == 0. (kernels/k-core/src/gemm.rs:172-262: fe_gemv_bf16 and fe_gemv_bf16_kw)
//
// Bound by the weights' way from HBM, every row count up to 64 reading them once: the sums of dot products that this replaces
// ran out of registers at 8 rows and took another pass over the weights for every 8. Weights and x rows go straight into LDS,
// DEPTH - 1 steps ahead, 8 rows x 128 bytes a load into stages that belong to one wavefront (no barrier in the loop): whole cache
// lines, which fragments loaded straight into registers (16 rows x 64 bytes) are not, at 42 us instead of 28. The weight loads
// are non-temporal (31.5 -> 28.3 us at 1 row). x comes from L2 once a program, so wide programs (CO) matter with the rows.
// 5120 x 17408, us, before -> now: 1 row 26.6 -> 27.1, 4 rows 29.6 -> 27.8, 8 rows 40.6 -> 28.1, 16 rows 80.8 -> 29.2, 40 rows
// 202 -> 43, 64 rows 321 -> 52 (one or two rows on a few widths 2 to 5 % slower: 5120 x 5120 9.4 -> 9.8); 17408 x 5120: 27.3 -> 27.1, 32.3 -> 27.8,
// 41.7 -> 29.3, 83.3 -> 33.7, 209 -> 48, 334 -> 57. Distance of the bf16 results from 64-bit sums: 1.66e-3 of their norm, the same to seven digits
// before and now.
template <int XO, int CO>
struct Bf16Gemv {
    static constexpr int L = CO + XO, STAGE = L * 1024;  // loads of a step
    // steps in LDS: 80 KB a program, so that two share a CU, but three at least (half or twice the room: the same within 1 %)
    static constexpr int FIT = 20 * 1024 / STAGE, DEPTH = FIT < 3 ? 3 : FIT < 8 ? FIT : 8;
    static constexpr int LDS = 4 * DEPTH * STAGE;
    static_assert((DEPTH - 1) * L < 64 && LDS <= 160 * 1024, "stages");
};

// PAIR: c[r][n] = bf16(bf16(silu(bf16(x . W[n]))) * bf16(x . W2[n])), gate and up of an MLP block at once: a program runs its columns of W, then
// those of W2, in one chain of steps (the loads run across), and keeps the gate's sums in registers meanwhile. The bits of two GEMVs and fe_silu_mul
// behind them; res is not read. An MLP block
// (gate, up, SwiGLU, down) in two launches for four, us: 5120 x 17408 at 1 / 12 / 32 / 64 rows 84 -> 80, 93 -> 88, 117 -> 108, 171 -> 160; 2048 x
// 5632 19.0 -> 14.9, 21.8 -> 16.5, 27.9 -> 23.0, 39.4 -> 34.0; 1024 x 2816 12.1 -> 7.9, 13.6 -> 9.5, 17.2 -> 13.1, 23.1 -> 18.7. The columns of a
// program are those of the single linear
// (gemv_cols): within 2 % of the best width of both launches on six layers at 1 to 64 rows.
template <int XO, int CO, bool PAIR>
__device__ __forceinline__ void gemv_bf16_body(uint16_t* c, const uint16_t* a, const uint16_t* w, const uint16_t* w2, const uint16_t* res,
                                               uint32_t m, uint32_t n, uint32_t k, uint32_t lda, uint32_t ldc, uint32_t pc) {
    typedef Bf16Gemv<XO, CO> C;
    constexpr int RG = (XO + 1) / 2, CG = (CO + 1) / 2, AHEAD = C::DEPTH - 1, PITCH = 16 * CG + 4;
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r = lane & 15, g = lane >> 4;
    const uint32_t col0 = blockIdx.x * pc, cols = n - col0 < pc ? n - col0 : pc;
    const u32x4 wrs = g8_rsrc(w + (size_t)col0 * k, cols * k * 2), w2rs = PAIR ? g8_rsrc(w2 + (size_t)col0 * k, cols * k * 2) : wrs, xrs = g8_rsrc(a, ((m - 1) * lda + k) * 2);
    // a row's 16-byte chunk c of a step lies at position c ^ (row & 7); rows that do not exist repeat the last one
    const uint32_t lr = lane >> 3, lc = ((lane & 7) ^ lr) << 4;
    uint32_t vw[CO], vx[XO];
#pragma unroll
    for (int j = 0; j < CO; j++) vw[j] = (8 * j + lr < cols ? 8 * j + lr : cols - 1) * k * 2 + lc;
#pragma unroll
    for (int j = 0; j < XO; j++) vx[j] = (8 * j + lr < m ? 8 * j + lr : m - 1) * lda * 2 + lc;
    unsigned char* stages = lds + wave * (C::DEPTH * C::STAGE);
    const uint32_t stages0 = g8_lds_addr(stages);
    const uint32_t steps = k / 64, s0 = wave * steps / 4, count = (wave + 1) * steps / 4 - s0, total = PAIR ? 2 * count : count;
    auto issue = [&](uint32_t s, uint32_t slot) {
        const bool second = PAIR && s >= count;
        const uint32_t at = stages0 + slot * C::STAGE, off = (s0 + (second ? s - count : s)) * 128;
        const u32x4 rs = second ? w2rs : wrs;
#pragma unroll
        for (int j = 0; j < CO; j++) g8_load_lds16_nt(rs, at + j * 1024, vw[j], off);
#pragma unroll
        for (int j = 0; j < XO; j++) g8_load_lds16(xrs, at + (CO + j) * 1024, vx[j], off);
    };
    // where the lane's fragments lie in a stage (columns past the program's: the last one again, not stored)
    uint32_t fw[CG][2], fx[RG][2];
    auto frag = [&](uint32_t row, int h) { return row * 128 + (((4 * h + g) ^ (row & 7)) << 4); };
#pragma unroll
    for (int h = 0; h < 2; h++) {
#pragma unroll
        for (int j = 0; j < CG; j++) fw[j][h] = frag(16 * j + r < 8 * CO ? 16 * j + r : 8 * CO - 1, h);
#pragma unroll
        for (int i = 0; i < RG; i++) fx[i][h] = CO * 1024 + frag(16 * i + r < m ? 16 * i + r : m - 1, h);
    }
    f32x4 acc[RG][CG] = {}, gate[RG][CG] = {};
    auto take_gate = [&]() {
#pragma unroll
        for (int i = 0; i < RG; i++)
#pragma unroll
            for (int j = 0; j < CG; j++) gate[i][j] = acc[i][j], acc[i][j] = f32x4{};
    };
    uint32_t slot = 0;
    auto add = [&]() {
        const unsigned char* st = stages + slot * C::STAGE;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            bf16x8 wv[CG];
#pragma unroll
            for (int j = 0; j < CG; j++) wv[j] = *(const bf16x8*)(st + fw[j][h]);
#pragma unroll
            for (int i = 0; i < RG; i++) {
                const bf16x8 xv = *(const bf16x8*)(st + fx[i][h]);
#pragma unroll
                for (int j = 0; j < CG; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv[j], xv, acc[i][j], 0, 0, 0);
            }
        }
        slot = slot + 1 == C::DEPTH ? 0 : slot + 1;
    };
    if (count) {
#pragma unroll
        for (int u = 0; u < AHEAD; u++) issue((uint32_t)u < total ? u : total - 1, u);  // past the end: the last step again, not added
        uint32_t s = 0;
        auto run = [&](uint32_t end) {
            for (; s < end && s + AHEAD < total; s++) {
                g8_loads_wait<(AHEAD - 1) * C::L>();  // (the stage in front of this one has been read, too)
                issue(s + AHEAD, slot ? slot - 1 : AHEAD);
                add();
            }
        };
        if constexpr (PAIR) {
            run(count);
            if (s == count) take_gate();
        }
        run(total);
        auto tail = [&](auto u_tag) {
            constexpr int U = decltype(u_tag)::value;
            if (s + U < total) {
                if (PAIR && U > 0 && s + U == count) take_gate();  // (fewer steps than stages)
                g8_loads_wait<(AHEAD - 1 - U) * C::L>();
                add();
            }
        };
        tail(std::integral_constant<int, 0>{});
        if constexpr (AHEAD > 1) tail(std::integral_constant<int, 1>{});
        if constexpr (AHEAD > 2) tail(std::integral_constant<int, 2>{});
        if constexpr (AHEAD > 3) tail(std::integral_constant<int, 3>{});
        if constexpr (AHEAD > 4) tail(std::integral_constant<int, 4>{});
        if constexpr (AHEAD > 5) tail(std::integral_constant<int, 5>{});
        if constexpr (AHEAD > 6) tail(std::integral_constant<int, 6>{});
        g8_loads_wait<0>();
    }
    float(*red)[16][PITCH] = (float(*)[16][PITCH])lds;
#pragma unroll
    for (int i = 0; i < RG; i++) {
        auto meet = [&](f32x4(&part)[RG][CG]) {
            __syncthreads();
#pragma unroll
            for (int j = 0; j < CG; j++) *(f32x4*)&red[wave][r][16 * j + 4 * g] = part[i][j];
            __syncthreads();
        };
        auto sum = [&](uint32_t row, uint32_t j) { return ((red[0][row][j] + red[1][row][j]) + red[2][row][j]) + red[3][row][j]; };
        uint32_t gates[CG];
        if constexpr (PAIR) {
            meet(gate);
#pragma unroll
            for (int e = 0; e < CG; e++) {
                const uint32_t row = (tid + 256 * e) / (8 * CO), j = (tid + 256 * e) % (8 * CO);
                gates[e] = row < 16 ? f32_to_bf16_bits(sum(row, j)) : 0;
            }
        }
        meet(acc);
#pragma unroll
        for (int e = 0; e < CG; e++) {
            const uint32_t row = (tid + 256 * e) / (8 * CO), j = (tid + 256 * e) % (8 * CO);
            if (row < 16 && 16 * i + row < m && j < cols) {
                float y = sum(row, j);
                if constexpr (PAIR) {
                    c[(size_t)(16 * i + row) * ldc + col0 + j] = (uint16_t)silu_mul_bf16x2(gates[e], f32_to_bf16_bits(y));
                    continue;
                }
                const size_t at = (size_t)(16 * i + row) * ldc + col0 + j;
                if (res) y = bf16_bits_to_f32(f32_to_bf16_bits(y)) + bf16_bits_to_f32(res[at]);
                c[at] = (uint16_t)f32_to_bf16_bits(y);
            }
        }
    }
}

#define BF16_GEMV_KERNEL(XO, CO)                                                                                             \
    extern "C" __global__ __launch_bounds__(256) void fe_gemv_bf16_r##XO##_c##CO(                                            \
        uint16_t* c, const uint16_t* a, const uint16_t* w, const uint16_t* res, uint32_t m, uint32_t n, uint32_t k, uint32_t lda, \
        uint32_t ldc, uint32_t pc) {                                                                                       \
        gemv_bf16_body<XO, CO, false>(c, a, w, w, res, m, n, k, lda, ldc, pc);                                             \
    }                                                                                                                      \
    extern "C" __global__ __launch_bounds__(256) void fe_gemv_bf16_swiglu_r##XO##_c##CO(                                   \
        uint16_t* act, const uint16_t* a, const uint16_t* gate, const uint16_t* up, uint32_t m, uint32_t n, uint32_t k, uint32_t lda, uint32_t pc) { \
        gemv_bf16_body<XO, CO, true>(act, a, gate, up, nullptr, m, n, k, lda, n, pc);                                      \
    }
#define BF16_GEMV_ROWS(XO)                                                                                                  \
    BF16_GEMV_KERNEL(XO, 1) BF16_GEMV_KERNEL(XO, 2) BF16_GEMV_KERNEL(XO, 3) BF16_GEMV_KERNEL(XO, 4) BF16_GEMV_KERNEL(XO, 5)
BF16_GEMV_ROWS(1)
BF16_GEMV_ROWS(2)
BF16_GEMV_ROWS(4)
BF16_GEMV_ROWS(6)
BF16_GEMV_ROWS(8)
BF16_GEMV_KERNEL(1, 6) BF16_GEMV_KERNEL(2, 6) BF16_GEMV_KERNEL(4, 6) BF16_GEMV_KERNEL(6, 6)
BF16_GEMV_KERNEL(1, 9) BF16_GEMV_KERNEL(2, 9) BF16_GEMV_KERNEL(4, 9)
