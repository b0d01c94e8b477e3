// The plain bf16 weight form of the caller's linear: y[M][N] = x[M][K] . W[N][K]^T (+ residual), W row-major bf16, f32
// sums, bf16 out. A GEMM on the shared 256 x 256 MFMA tile loop and two decode-sized GEMVs (kernels/k-core/src/gemm.rs).
#include "gemm8.h"

// 4 sums of columns at.. of one row -> bf16; with res: bf16(bf16(sum) + res) (gemm.rs:152-158).
__device__ __forceinline__ void bf16_store4(uint16_t* c, const uint16_t* res, size_t at, const float (&v)[4]) {
    u32x2 o = {pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
    if (res) {
        u32x2 r = *(const u32x2*)(res + at);
#pragma unroll
        for (int e = 0; e < 2; e++)
            o[e] = pack_bf16x2(bf16_bits_to_f32(o[e] & 0xffff) + bf16_bits_to_f32(r[e] & 0xffff),
                               bf16_bits_to_f32(o[e] >> 16) + bf16_bits_to_f32(r[e] >> 16));
    }
    *(u32x2*)(c + at) = o;
}

// ---- GEMM ------------------------------------------------------------------------------------------------------------

typedef G8Tile<4, 2, 4, 8> Bf16Tile;    // 256 x 256
typedef G8Tile<4, 2, 2, 8> Bf16TileS1;  // 128 x 256
typedef G8Tile<4, 2, 2, 4> Bf16TileS2;  // 128 x 128, two programs a CU
// k tiles of A and of W in LDS: as many as the tile leaves room for
template <class T>
struct Bf16Stages {
    static constexpr int NA = T::PARTS == 2 ? 3 : 2, NW = 3, MIN_WAVES = T::PARTS == 4 ? 4 : 2;
};

// One program's share of A . W^T: main loop, then the partial slot (a tile cut along K) or done(row, col, lane in row, v[4]) for
// every row piece of the tile, all lanes of a row calling (row >= m and col >= n included).
template <class T, class Done>
__device__ __forceinline__ void bf16_gemm_program(const uint16_t* a, const uint16_t* w, uint32_t m, uint32_t n, uint32_t k, uint32_t lda,
                                                  uint32_t group_m, const GemmSched& sc, Done done) {
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
    const uint32_t wave = threadIdx.x >> 6, wm = wave / T::WN, wn = wave % T::WN;
    g8_schedule<T, false>(
        sc, m, n, group_m, k / G8_BK, lds,
        [&](uint32_t m0, uint32_t n0, uint32_t kt0, uint32_t ktn, f32x4(&acc)[T::TM][T::TN]) {
            G8Dense<T> wo;
            wo.rows(w, n, k, n0);
            g8_mainloop<T, Bf16Stages<T>::NA, Bf16Stages<T>::NW, true>(a, lda, m, kt0, ktn, m0, wo, lds, acc);
        },
        [&](uint32_t m0, uint32_t n0, f32x4(&acc)[T::TM][T::TN]) {
            const uint32_t row0 = m0 + wm * 16 * T::TM, col0 = n0 + wn * 16 * T::TN;
            g8_epilogue<T>(
                acc, lds, [](auto&, uint32_t) {},
                [&](uint32_t row, uint32_t lc, float (&v)[4]) { done(row0 + row, col0 + 4 * lc, lc, v); });
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
        bf16_gemm_program<TILE>(a, w, m, n, k, lda, group_m, sc, [&](uint32_t row, uint32_t col, uint32_t, float (&v)[4]) { \
            if (row < m && col < n) bf16_store4(c, res, (size_t)row * ldc + col, v);                                       \
        });                                                                                                                \
    }                                                                                                                      \
    extern "C" __global__ __launch_bounds__(256) void fe_gemm_bf16_reduce##SUFFIX(                                         \
        uint16_t* c, const float* part, const uint16_t* res, uint32_t m, uint32_t n, uint32_t ldc, uint32_t group_m,       \
        uint32_t first, uint32_t splits) {                                                                                 \
        g8_reduce_rows<TILE>(part, m, n, group_m, first, splits, [&](uint32_t row, uint32_t n0, uint32_t l32, float (&v)[4]) { \
            const uint32_t col = n0 + 4 * l32;                                                                             \
            if (row < m && col < n) bf16_store4(c, res, (size_t)row * ldc + col, v);                                       \
        });                                                                                                                \
    }
BF16_GEMM_KERNELS(, Bf16Tile)
BF16_GEMM_KERNELS(_s1, Bf16TileS1)
BF16_GEMM_KERNELS(_s2, Bf16TileS2)

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

// act[M][N / 2] = SwiGLU(A . W^T) for interleaved gate|up weights W [N][K], N % 16 == 0: fe_gemm_bf16 with the epilogue
// above, and its reduce kernels. (kernels/k-core/src/gemm.rs:264-279: fe_gemm_swiglu)
#define BF16_SWIGLU_KERNELS(SUFFIX, TILE)                                                                                  \
    extern "C" __global__ __launch_bounds__(512, Bf16Stages<TILE>::MIN_WAVES) void fe_gemm_bf16_swiglu##SUFFIX(            \
        uint16_t* act, const uint16_t* a, const uint16_t* w, uint32_t m, uint32_t n, uint32_t k, uint32_t lda,             \
        uint32_t group_m, GemmSched sc) {                                                                                  \
        bf16_gemm_program<TILE>(a, w, m, n, k, lda, group_m, sc, [&](uint32_t row, uint32_t col, uint32_t lc, float (&v)[4]) { \
            bf16_swiglu_store4(act, v, lc, row < m, row, col, n);                                                          \
        });                                                                                                                \
    }                                                                                                                      \
    extern "C" __global__ __launch_bounds__(256) void fe_gemm_bf16_swiglu_reduce##SUFFIX(                                  \
        uint16_t* act, const float* part, uint32_t m, uint32_t n, uint32_t group_m, uint32_t first, uint32_t splits) {      \
        g8_reduce_rows<TILE>(part, m, n, group_m, first, splits, [&](uint32_t row, uint32_t n0, uint32_t l32, float (&v)[4]) { \
            bf16_swiglu_store4(act, v, l32, row < m, row, n0 + 4 * l32, n);                                                \
        });                                                                                                                \
    }
BF16_SWIGLU_KERNELS(, Bf16Tile)
BF16_SWIGLU_KERNELS(_s1, Bf16TileS1)
BF16_SWIGLU_KERNELS(_s2, Bf16TileS2)

// dst row 16 b + i = gate row 8 b + i for i < 8, up row 8 b + i - 8 otherwise: the weight layout of fe_gemm_bf16_swiglu.
// grid 2 inter, 256 threads; k % 8 == 0. (kernels/k-core/src/gemm.rs:281-296: fe_interleave_gu)
extern "C" __global__ __launch_bounds__(256) void fe_interleave_gu(uint16_t* dst, const uint16_t* gate, const uint16_t* up,
                                                                   uint32_t k) {
    const uint32_t r = blockIdx.x, b = r / 16, i = r % 16;
    const uint16_t* src = i < 8 ? gate + (size_t)(b * 8 + i) * k : up + (size_t)(b * 8 + i - 8) * k;
    uint16_t* d = dst + (size_t)r * k;
    for (uint32_t j = threadIdx.x; j < k / 8; j += 256) *((u32x4*)d + j) = *((const u32x4*)src + j);
}

// ---- GEMV (1..8 rows) ------------------------------------------------------------------------------------------------

__device__ __forceinline__ float dot8_bf16(u32x4 w, u32x4 x, float acc) {
#pragma unroll
    for (int p = 0; p < 4; p++) {
        // the elements are copied out first: __builtin_bit_cast applied to a vector element reads element 0
        const uint32_t wp = w[p], xp = x[p];
        acc = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, wp), __builtin_bit_cast(bf16x2, xp), acc, false);
    }
    return acc;
}

// Sum over each row of 16 lanes, left in all 16 (four DPP adds: no LDS traffic, unlike a butterfly of ds_bpermute).
__device__ __forceinline__ float row16_sum(float v) {
    v += dpp_mov<DPP_QUAD_XOR1>(v);
    v += dpp_mov<DPP_QUAD_XOR2>(v);
    v += dpp_mov<DPP_HALF_MIRROR>(v);
    v += dpp_mov<DPP_ROW_MIRROR>(v);
    return v;
}

// One wavefront: the sums of x rows 0..MR-1 (rows >= m repeat row m - 1) with NC weight rows over the 16-byte chunks
// [c0, c1) of K, lane L taking chunks c0 + L, c0 + L + 64, ... in ascending order, one v_dot2 per element pair; then
// every 16 lanes add up (the sum of lanes 16 q .. 16 q + 15 is left in all of them).
template <int MR, int NC>
__device__ __forceinline__ void gemv_bf16_sums(const uint16_t* a, const uint16_t* const (&wr)[NC], uint32_t m, uint32_t lda,
                                               uint32_t c0, uint32_t c1, float (&acc)[MR][NC]) {
    const uint32_t lane = threadIdx.x & 63;
    const uint16_t* xr[MR];
#pragma unroll
    for (int r = 0; r < MR; r++) {
        xr[r] = a + (size_t)((uint32_t)r < m ? r : m - 1) * lda;
#pragma unroll
        for (int j = 0; j < NC; j++) acc[r][j] = 0.f;
    }
#pragma unroll 2
    for (uint32_t i = c0 + lane; i < c1; i += 64) {
        u32x4 wv[NC], xv[MR];
#pragma unroll
        for (int j = 0; j < NC; j++) wv[j] = __builtin_nontemporal_load((const u32x4*)wr[j] + i);
#pragma unroll
        for (int r = 0; r < MR; r++) xv[r] = *((const u32x4*)xr[r] + i);
#pragma unroll
        for (int r = 0; r < MR; r++)
#pragma unroll
            for (int j = 0; j < NC; j++) acc[r][j] = dot8_bf16(wv[j], xv[r], acc[r][j]);
    }
#pragma unroll
    for (int r = 0; r < MR; r++)
#pragma unroll
        for (int j = 0; j < NC; j++) acc[r][j] = row16_sum(acc[r][j]);
}

// y[r][n] = bf16(x[r][:] . W[n][:]) (+ res) for r < m <= MR. grid N / NC, 256 threads: a program takes NC consecutive
// columns; K is walked in steps of 64 chunks of 16 bytes (a 1 KB run of every weight row a step), wavefront w takes
// steps [w S / 4, (w + 1) S / 4) of the S steps, and the sixteen sums (4 wavefronts x 4 rows of 16 lanes) are added in order. So a row's bits depend
// on K only, neither on the other rows nor on NC: the host picks NC by the shape and the row count (more columns a program
// read x less often, fewer columns give more programs), where the reference picks between two kernels by the shape.
// K % 8 == 0, N % NC == 0, lda % 8 == 0. (kernels/k-core/src/gemm.rs:172-262: fe_gemv_bf16 and fe_gemv_bf16_kw)
template <int MR, int NC>
__device__ __forceinline__ void gemv_bf16_body(uint16_t* c, const uint16_t* a, const uint16_t* w, const uint16_t* res,
                                               uint32_t m, uint32_t n, uint32_t k, uint32_t lda, uint32_t ldc) {
    __shared__ float red[16][MR][NC];
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6, col = blockIdx.x * NC;
    const uint16_t* wr[NC];
#pragma unroll
    for (int j = 0; j < NC; j++) wr[j] = w + (size_t)(col + j) * k;
    const uint32_t chunks = k / 8, steps = (chunks + 63) / 64;
    const uint32_t c0 = (wave * steps / 4) * 64, c1 = ((wave + 1) * steps / 4) * 64;
    float acc[MR][NC];
    gemv_bf16_sums<MR, NC>(a, wr, m, lda, c0, c1 < chunks ? c1 : chunks, acc);
    if ((lane & 15) == 0) {
#pragma unroll
        for (int r = 0; r < MR; r++)
#pragma unroll
            for (int j = 0; j < NC; j++) red[threadIdx.x >> 4][r][j] = acc[r][j];
    }
    __syncthreads();
    const uint32_t r = threadIdx.x / NC, j = threadIdx.x % NC;
    if (r < m) {
        float y = red[0][r][j];
        for (int q = 1; q < 16; q++) y += red[q][r][j];
        const size_t at = (size_t)r * ldc + col + j;
        if (res) y = bf16_bits_to_f32(f32_to_bf16_bits(y)) + bf16_bits_to_f32(res[at]);
        c[at] = (uint16_t)f32_to_bf16_bits(y);
    }
}

#define BF16_GEMV_KERNEL(MR, NC)                                                                                           \
    extern "C" __global__ __launch_bounds__(256) void fe_gemv_bf16_r##MR##_c##NC(uint16_t* c, const uint16_t* a,           \
                                                                                 const uint16_t* w, const uint16_t* res,  \
                                                                                 uint32_t m, uint32_t n, uint32_t k,      \
                                                                                 uint32_t lda, uint32_t ldc) {            \
        gemv_bf16_body<MR, NC>(c, a, w, res, m, n, k, lda, ldc);                                                           \
    }
#define BF16_GEMV_ROWS(MR) BF16_GEMV_KERNEL(MR, 1) BF16_GEMV_KERNEL(MR, 2) BF16_GEMV_KERNEL(MR, 4) BF16_GEMV_KERNEL(MR, 8)
BF16_GEMV_ROWS(1)
BF16_GEMV_ROWS(2)
BF16_GEMV_ROWS(4)
BF16_GEMV_ROWS(8)
