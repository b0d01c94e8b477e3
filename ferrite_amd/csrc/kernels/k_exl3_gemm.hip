// EXL3 linear for gfx950, prefill-sized row counts: the GEMM that decodes the trellis as it goes, the pass that decodes it once
// into fp16 tiles, and the GEMM over those.
#include <type_traits>

#include "exl3_trellis.h"
#include "gemm8.h"

// ---- prefill GEMM ----------------------------------------------------------------------------------------------------

// Output tiles; a wavefront's 128 columns are one Hadamard block.
typedef G8Tile<4, 2, 4, 8> Exl3Tile;    // 256 x 256
typedef G8Tile<4, 2, 2, 8> Exl3TileS1;  // 128 x 256
typedef G8Tile<8, 1, 1, 8> Exl3TileS2;  // 128 x 128, two programs a CU

// Weight operand of the prefill GEMM: a 64-wide k tile of a 128-column block is 4 k steps x 8 tiles, and a lane of the GEMV's
// mapping decodes one run of words, 32 weights: rows n = q and q + 8 of tile L >> 3 (q = L & 7) over the 16 k of a step. At 256 columns
// wavefront w takes block w >> 2 and k step w & 3; at 128 columns k step w & 3 and row half w >> 2 (half a run a lane). A packed
// stage is [blocks][4 k steps][8 tiles][8 BITS words], pieces of 1 KB.
template <int BITS, class T>
struct Exl3Packed {
    static constexpr int BLOCKS = T::BN / 128, RAW_STAGE = 1024 * BITS * BLOCKS, PIECES = BITS * BLOCKS, LOADS = (PIECES + 7) / 8;
    static constexpr int OPS = 2 * BLOCKS;  // 8-value chunks a thread decodes a k tile
    struct Words {
        LaneWords<BITS> w;
        LaneWindows<BITS> win;
    };
    // A trellis may hold 4 GB and more (its row of tiles of a k tile or its column block is far below that): the resource starts at the
    // k tile that is loaded, with a 64-bit address, and ends where that k tile's last run of words does.
    uint64_t base;
    uint32_t voff[LOADS], step, span;
    __device__ __forceinline__ void setup(const uint32_t* trellis, uint32_t n, uint32_t k, uint32_t n0, uint32_t stride_k, uint32_t stride_nb) {
        const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
        const uint32_t nb0 = n0 / 128, blocks = n / 128 - nb0 < BLOCKS ? n / 128 - nb0 : BLOCKS;  // (an odd block count: the last tile holds one)
        const uint64_t b = (uint64_t)(trellis + (size_t)nb0 * stride_nb);
        base = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(b >> 32)) << 32 | (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)b);
        step = 16 * stride_k, span = __builtin_amdgcn_readfirstlane(4 * ((blocks - 1) * stride_nb + 3 * stride_k + 64 * BITS));
#pragma unroll
        for (int j = 0; j < LOADS; j++) {
            const uint32_t at = (wave + 8 * j) % PIECES * 1024 + lane * 16;  // (fewer pieces than wavefronts: some are moved twice)
            const uint32_t ks = at / (256 * BITS) % 4;
            uint32_t nb = at / (1024 * BITS);
            nb = nb < blocks ? nb : blocks - 1;  // the last tile of an odd block count decodes its first block twice
            voff[j] = 4 * (nb * stride_nb + ks * stride_k) + at % (256 * BITS);
        }
    }
    __device__ __forceinline__ void issue(uint32_t kt, uint32_t dst, int j, uint32_t wave) const {
        g8_load_lds16(g8_rsrc((const void*)(base + (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane(kt) * step), span), dst + (wave + 8 * j) % PIECES * 1024, voff[j], 0);
    }
    __device__ __forceinline__ Words read(const unsigned char* st) const {
        const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6, tile = (BLOCKS == 2 ? wave : wave & 3) * 8 + (lane >> 3);
        const uint32_t* p = (const uint32_t*)st + tile * (8 * BITS) + (lane & 7) * BITS;
        Words w;
        if constexpr (BITS % 4 == 0) {
#pragma unroll
            for (int i = 0; i < BITS; i += 4) {
                const u32x4 t = *(const u32x4*)(p + i);
                w.w.w[i + 1] = t[0], w.w.w[i + 2] = t[1], w.w.w[i + 3] = t[2], w.w.w[i + 4] = t[3];
            }
        } else {
#pragma unroll
            for (int i = 0; i < BITS; i++) w.w.w[i + 1] = p[i];
        }
        w.w.w[0] = 0;
        return w;
    }
    // The word before the run and the windows over the word boundaries. At 128 columns the threads of row half 1 shift their stream by
    // the 4 positions between the halves, so that both decode the same positions.
    __device__ __forceinline__ void prepare(Words& w) const {
        w.w.w[0] = lane_prev_word_halves(w.w.w[BITS]);
        if constexpr (BLOCKS == 1) {
            if (threadIdx.x >= 256) {
#pragma unroll
                for (int i = 0; i < BITS; i++)
                    w.w.w[i] = 4 * BITS == 32 ? w.w.w[i + 1] : __builtin_amdgcn_alignbit(w.w.w[i], w.w.w[i + 1], 32 - 4 * BITS % 32);
                w.w.w[BITS] = 4 * BITS == 32 ? 0u : w.w.w[BITS] << (4 * BITS % 32);
            }
        }
        w.win = lane_windows<BITS>(w.w);
    }
    // chunk o: (row half, k half) = (o >> 1, o & 1), or (the thread's, o)
    __device__ __forceinline__ uint32_t pair(const Words& w, int o, int p) const { return decode_lane_pair<BITS>(w.w, w.win, BLOCKS == 2 ? o >> 1 : 0, o & 1, p); }
    __device__ __forceinline__ void put(unsigned char* ws, int o, u32x4 v) const {
        const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
        const uint32_t r = (BLOCKS == 2 ? 128 * (wave >> 2) + 8 * (o >> 1) : 8 * (wave >> 2)) + (lane >> 3) * 16 + (lane & 7);
        *(u32x4*)(ws + r * 128 + (((2 * (wave & 3) + (o & 1)) ^ (r & 7)) << 4)) = v;
    }
};
// k tiles of A and packed k tiles in LDS, beside two of decoded weights: what 160 KB hold, or half of it for the smallest tile
template <int BITS, class T>
struct Exl3Stages {
    static constexpr int NA = T::PARTS == 2 ? 3 : 2;
    static constexpr int FREE = (T::PARTS == 4 ? 80 : 160) * 1024 - NA * T::BM * 128 - 2 * T::BN * 128, FIT = FREE / Exl3Packed<BITS, T>::RAW_STAGE;
    static constexpr int NR = FIT < 2 ? 2 : FIT > 6 ? 6 : FIT;
};
template <class T>
struct Exl3Waves {
    static constexpr int MIN = T::PARTS == 4 ? 4 : 2;
};

// y[m][n] (+)= H(xh @ W_hat) * svh / sqrt(128) for prefill-sized m: xh fp16 [m][k] (rotated inputs); a wavefront's 128
// columns are exactly one Hadamard block, so the output rotation is local to the wavefront. Tiles (grouped raster) spread
// over the grid as sched says (g8_schedule). 512 threads, dynamic LDS as the stages take (the epilogue reuses it).
// loop(m0, n0, kt0, ktn, lds, acc) is a pass of the main loop.
template <class T, bool SK, class Loop>
__device__ __forceinline__ void exl3_gemm_tile(const uint16_t* __restrict__ svh, void* y, uint32_t n, uint32_t k, uint32_t m,
                                               uint32_t y_mode, uint32_t group_m, const GemmSched& sched, Loop loop) {
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
    const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wm = wave / T::WN, wn = wave % T::WN;
    g8_schedule<T, SK>(
        sched, m, n, group_m, k / G8_BK, lds,
        [&](uint32_t m0, uint32_t n0, uint32_t kt0, uint32_t ktn, f32x4(&acc)[T::TM][T::TN]) { loop(m0, n0, kt0, ktn, lds, acc); },
        [&](uint32_t m0, uint32_t n0, f32x4(&acc)[T::TM][T::TN]) {
            const uint32_t row0 = m0 + wm * 16 * T::TM, col0 = n0 + wn * 128;
            if (col0 >= n) return;
            const uint32_t col = col0 + 4 * (lane & 31);
            const f32x4 sc = row_scales(svh, col);
            // one copy of the epilogue per output mode, so that the row loop has no mode branches
            auto run = [&](auto mode_tag) {
                constexpr uint32_t MODE = decltype(mode_tag)::value;
                g8_epilogue<T>(
                    acc, lds,
                    [&](float (&v)[4][4], uint32_t l32) {
                        fwht128_half_wave_rows(v, l32);
#pragma unroll
                        for (int u = 0; u < 4; u++)
#pragma unroll
                            for (int e = 0; e < 4; e++) v[u][e] = v[u][e] * FE_HAD_SCALE * sc[e];  // finish_row's products
                    },
                    [&](uint32_t row, uint32_t) {
                        if constexpr (MODE >= 2)
                            return row0 + row < m ? store4_old(y, MODE, (size_t)(row0 + row) * n + col) : (u32x4){0, 0, 0, 0};
                        else
                            return G8Nothing{};
                    },
                    [&](uint32_t row, uint32_t, float (&v)[4], auto old) {
                        if (row0 + row >= m) return;
                        if constexpr (MODE >= 2)
                            store4(y, MODE, (size_t)(row0 + row) * n + col, v, old);
                        else
                            store4(y, MODE, (size_t)(row0 + row) * n + col, v);
                    });
            };
            if (y_mode == 0)
                run(std::integral_constant<uint32_t, 0>{});
            else if (y_mode == 1)
                run(std::integral_constant<uint32_t, 1>{});
            else if (y_mode == 2)
                run(std::integral_constant<uint32_t, 2>{});
            else
                run(std::integral_constant<uint32_t, 3>{});
        });
}

// The GEMM decoding the trellis itself: every row tile of the output decodes its weights again.
template <int BITS, class T, bool SK>
__device__ __forceinline__ void exl3_gemm_body(const _Float16* __restrict__ xh, const uint32_t* __restrict__ trellis,
                                               const uint16_t* __restrict__ svh, void* y, uint32_t n, uint32_t k, uint32_t m,
                                               uint32_t y_mode, uint32_t stride_k, uint32_t stride_nb, uint32_t group_m,
                                               const GemmSched& sched) {
    exl3_gemm_tile<T, SK>(svh, y, n, k, m, y_mode, group_m, sched,
                          [&](uint32_t m0, uint32_t n0, uint32_t kt0, uint32_t ktn, unsigned char* lds, f32x4(&acc)[T::TM][T::TN]) {
                              Exl3Packed<BITS, T> w;
                              w.setup(trellis, n, k, n0, stride_k, stride_nb);
                              g8_mainloop_decode<T, Exl3Stages<BITS, T>::NA, Exl3Stages<BITS, T>::NR, !SK>(xh, k, m, kt0, ktn, m0, w, lds, acc);
                          });
}

// ---- prefill over decoded weights -----------------------------------------------------------------------------------
//
// For many rows the trellis is decoded once per call into `hat`, fp16, as the very images the GEMM keeps in LDS: block
// (tn, kt) of 32 KB = rows n = 256 tn .. + 255 of k tile kt, 128 bytes a row, 16-byte chunk c of row r at the position gm_swz
// gives it. The GEMM over it then copies blocks instead of decoding, with the same fragments, the same MFMA order and
// so the same bits as exl3_gemm_b*.

// grid (n / 128, gy), 256 threads; program (nb, j) decodes k tiles j, j + gy, ... of column block nb with the lane
// mapping of Exl3Producer. The 16 KB of a k tile pass through LDS (two buffers, one barrier a tile) so that they leave
// as whole 1 KB runs per wavefront instead of scattered 16-byte pieces.
template <int BITS>
__device__ __forceinline__ void exl3_hat_tiles_body(const uint32_t* __restrict__ trellis, unsigned char* __restrict__ hat,
                                                    uint32_t k, uint32_t stride_k, uint32_t stride_nb) {
    __shared__ __attribute__((aligned(16))) unsigned char img[2][GM_B_BYTES / 2];
    constexpr uint32_t tw = 8 * BITS;
    const uint32_t lane = threadIdx.x & 63, ks = threadIdx.x >> 6, tj = lane >> 3, q = lane & 7;
    const uint32_t nb = blockIdx.x, ktiles = k / GM_BK;
    const uint32_t* base = trellis + (size_t)nb * stride_nb + tj * tw;
    const uint32_t run_off = q * BITS, prev_off = (q * BITS + tw - 1) % tw;
    const uint32_t row = tj * 16 + q;
    unsigned char* out = hat + (size_t)(nb >> 1) * ktiles * GM_B_BYTES + (nb & 1) * (GM_B_BYTES / 2) + 16 * threadIdx.x;
    uint32_t kt = blockIdx.y;
    if (kt >= ktiles) return;
    const uint32_t* p = base + (size_t)(kt * 4 + ks) * stride_k;
    LaneWords<BITS> cur = load_lane_words<BITS>(p + run_off, p + prev_off);
    for (uint32_t it = 0; kt < ktiles; kt += gridDim.y, it++) {
        uint32_t nk = kt + gridDim.y < ktiles ? kt + gridDim.y : kt;
        const uint32_t* pn = base + (size_t)(nk * 4 + ks) * stride_k;
        LaneWords<BITS> nxt = load_lane_words<BITS>(pn + run_off, pn + prev_off);
        f16x8 op[2][2];
        decode_lane<BITS>(cur, op);
        unsigned char* buf = img[it & 1];
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int kh = 0; kh < 2; kh++) *(f16x8*)(buf + gm_swz(row + 8 * h, 2 * ks + kh)) = op[h][kh];
        __syncthreads();
        unsigned char* blk = out + (size_t)kt * GM_B_BYTES;
#pragma unroll
        for (int j = 0; j < 4; j++) *(u32x4*)(blk + 4096 * j) = *(const u32x4*)(buf + 16 * threadIdx.x + 4096 * j);
        cur = nxt;
    }
}

// (every GEMM kernel comes as NAME, 256 x 256 tiles one piece a program, NAME_sk, stream-K, and NAME_s1 and NAME_s2, the smaller
// tiles, with the same parameters)
#define HAT_GEMM_PARAMS                                                                                                  \
    const _Float16 *xh, const unsigned char *hat, const uint16_t *svh, void *y, uint32_t n, uint32_t k, uint32_t m, uint32_t y_mode, \
        uint32_t group_m, GemmSched sched
template <class T, bool SK>
__device__ __forceinline__ void exl3_gemm_hat_kernel(HAT_GEMM_PARAMS) {
    constexpr int NA = T::PARTS == 2 ? 3 : 2, NW = T::PARTS == 2 ? 3 : 3;
    exl3_gemm_tile<T, SK>(svh, y, n, k, m, y_mode, group_m, sched,
                          [&](uint32_t m0, uint32_t n0, uint32_t kt0, uint32_t ktn, unsigned char* lds, f32x4(&acc)[T::TM][T::TN]) {
                              // the rows' blocks of 32 KB; a row's chunks lie where gm_swz puts them: the core's position, its low
                              // bit flipped in every second group of 8 rows
                              const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6, bytes = (k / G8_BK) * GM_B_BYTES;
                              G8Dense<T> w;
                              w.rs = g8_rsrc(hat + (size_t)(n0 / 256) * bytes, bytes), w.kstep = GM_B_BYTES;
#pragma unroll
                              for (int j = 0; j < G8Dense<T>::LOADS; j++) {
                                  const uint32_t r = n0 % 256 + 8 * (wave + 8 * j) + (lane >> 3);
                                  w.voff[j] = r * 128 + (((lane & 7) ^ ((r >> 3) & 1)) << 4);
                              }
                              g8_mainloop<T, NA, NW, false, !SK>(xh, k, m, kt0, ktn, m0, w, lds, acc);
                          });
}
// Finishes the tiles that a GEMM kernel cut along K: sums their partial slots and applies the output rotation and scale.
// Grid and threads: g8_reduce_rows.
template <class T>
__device__ __forceinline__ void exl3_reduce_body(const float* part, const uint16_t* svh, void* y, uint32_t n, uint32_t m, uint32_t y_mode,
                                                 uint32_t group_m, uint32_t first, uint32_t splits) {
    struct Ahead {
        u32x2 sv;
        u32x4 old;
    };
    g8_reduce_rows<T>(
        part, m, n, group_m, first, splits,
        [&](uint32_t row, uint32_t n0, uint32_t l32) {
            const uint32_t col = n0 + 4 * l32;
            return Ahead{*(const u32x2*)(svh + col), row < m ? store4_old(y, y_mode, (size_t)row * n + col) : (u32x4){0, 0, 0, 0}};
        },
        [&](uint32_t row, uint32_t n0, uint32_t l32, float (&v)[4], Ahead a) {
            if (row < m) finish_row(v, l32, a.sv, y, y_mode, (size_t)row * n + n0 + 4 * l32, a.old);
        });
}
#define HAT_GEMM_KERNEL(SUFFIX, TILE, SK)                                                                                  \
    extern "C" __global__ __launch_bounds__(512, Exl3Waves<TILE>::MIN) void exl3_gemm_hat##SUFFIX(HAT_GEMM_PARAMS) {       \
        exl3_gemm_hat_kernel<TILE, SK>(xh, hat, svh, y, n, k, m, y_mode, group_m, sched);                                  \
    }
HAT_GEMM_KERNEL(, Exl3Tile, false)
HAT_GEMM_KERNEL(_sk, Exl3Tile, true)
HAT_GEMM_KERNEL(_s1, Exl3TileS1, false)
HAT_GEMM_KERNEL(_s2, Exl3TileS2, false)
#define REDUCE_KERNEL(SUFFIX, TILE)                                                                                        \
    extern "C" __global__ __launch_bounds__(512) void exl3_gemm_reduce##SUFFIX(                                            \
        const float* part, const uint16_t* svh, void* y, uint32_t n, uint32_t m, uint32_t y_mode, uint32_t group_m,        \
        uint32_t first, uint32_t splits) {                                                                                 \
        exl3_reduce_body<TILE>(part, svh, y, n, m, y_mode, group_m, first, splits);                                        \
    }
REDUCE_KERNEL(, Exl3Tile)
REDUCE_KERNEL(_s1, Exl3TileS1)
REDUCE_KERNEL(_s2, Exl3TileS2)

#define GEMM_KERNEL_(NAME, BITS, TILE, SK)                                                                             \
    extern "C" __global__ __launch_bounds__(512, Exl3Waves<TILE>::MIN) void NAME(                                      \
        const _Float16* xh, const uint32_t* trellis, const uint16_t* svh, void* y, uint32_t n, uint32_t k, uint32_t m,  \
        uint32_t y_mode, uint32_t stride_k, uint32_t stride_nb, uint32_t group_m, GemmSched sched) {                    \
        exl3_gemm_body<BITS, TILE, SK>(xh, trellis, svh, y, n, k, m, y_mode, stride_k, stride_nb, group_m, sched);     \
    }
#define GEMM_KERNEL(BITS)                                    \
    GEMM_KERNEL_(exl3_gemm_b##BITS, BITS, Exl3Tile, false)    \
    GEMM_KERNEL_(exl3_gemm_b##BITS##_sk, BITS, Exl3Tile, true) \
    GEMM_KERNEL_(exl3_gemm_b##BITS##_s1, BITS, Exl3TileS1, false) \
    GEMM_KERNEL_(exl3_gemm_b##BITS##_s2, BITS, Exl3TileS2, false)
#define HAT_KERNEL(BITS)                                                                                      \
    extern "C" __global__ __launch_bounds__(256) void exl3_hat_tiles_b##BITS(                                 \
        const uint32_t* trellis, unsigned char* hat, uint32_t k, uint32_t stride_k, uint32_t stride_nb) {     \
        exl3_hat_tiles_body<BITS>(trellis, hat, k, stride_k, stride_nb);                                      \
    }
HAT_KERNEL(2)
HAT_KERNEL(3)
HAT_KERNEL(4)
HAT_KERNEL(5)
HAT_KERNEL(6)
HAT_KERNEL(8)
GEMM_KERNEL(2)
GEMM_KERNEL(3)
GEMM_KERNEL(4)
GEMM_KERNEL(5)
GEMM_KERNEL(6)
GEMM_KERNEL(8)

