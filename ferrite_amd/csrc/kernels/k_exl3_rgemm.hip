// EXL3 prompt GEMM for gfx950 whose decoded weights never leave the registers: the trellis linear for 65 to 2303 rows.
//
// y[m][n] (+)= H(xh @ W_hat) * svh / sqrt(128), xh fp16 [m][k] (rotated inputs). Up to four linears of one k and width share a launch
// (gate and up), each with its own rotated inputs.
//
// A wavefront decodes the words of 32 columns x 64 k (the GEMV's mapping: one run of words a lane, decode_lane) and multiplies them with
// all rows of its tile: the eight values a lane gets are an operand of v_mfma_f32_16x16x32_f16 as they are, so there is no pass through LDS
// between decode and product (exl3_gemm_b* writes them there, 15 cycles a KB, and reads them back) and no barrier waits for a decode.
// Words come through LDS too, but each wavefront's own; A's rows are shared. The pairs of the next k tile are decoded between the matrix
// instructions of this one; both are pinned there (empty asm statements), since the compiler's scheduler moves all of the decode to the
// front of the loop, where it runs with the matrix pipe idle.
//
// What bounds it: with few rows the decode (96 rows: 156 vector instructions a wavefront and step, 24 of them products; a step of the two wavefronts of a SIMD
// takes 1980 cycles, the matrix pipe busy 38 %), from 160 rows on the board's power: 208 rows of 17408 x 5120 run at 1.76 GHz with the matrix pipe 47
// % busy, and 256 programs of whole tiles take the cycles of 130 of them (399 000) and 22 % more time, 1.73 GHz against 2.14. So what counts beside
// the balance of the programs is to move and multiply little: row tiles as even and as low as the rows need (203 rows: 224, not 256), rows that do
// not exist read as zeros, tiles whole where possible (the sums of a cut one travel twice), gate and up in one launch. Loads are issued early in a
// step (at two stages the wait at the next step's start has to find them done: 17408 x 5120, 224 rows 47.5 -> 43.0 us), words a step earlier than A.
// us, the GEMM that goes through LDS -> this one, 4 bits, with rotation and reduce
// launches: 5120 x 17408 at 203 / 512 / 2048 rows 65.8 / 112 / 350 -> 60.9 / 107 / 347, 17408 x 5120 69.5 / 110 / 370 -> 55.4 / 105 / 354, 5120 x
// 1024 at 128 rows 21.1 -> 17.3.
#include "exl3_trellis.h"
#include "gemm8.h"

#define RG_MEMBERS 4
struct RgMember {
    const uint16_t* xh;  // [m][k]
    const uint32_t* trellis;
    const uint16_t* svh;
    void* y;
    uint32_t n, stride_k, stride_nb, first;  // first: its first column tile among those of the launch
};
// The tiles: the members' column tiles, one member after the other, times tiles_m row tiles of BM rows. Programs 0 .. full - 1 take
// one tile each over all of K. The tiles after them are dealt to `runs` programs: `per` a tile, each a per-th of its steps, or (per 0) the tiles' steps laid
// end to end in equal runs (base steps, the first rem programs one more). Runs that end inside a tile start the next one's products over, and meet
// the other programs' inputs at another depth of K: where pieces come out even a tile, 3 % of the time of the best plan (589 linears). A tile that is
// cut leaves the sums of its pieces, the one of run q in slot q + (tile - full), for the reduce kernel, which adds them in the order of K.
struct RgJob {
    RgMember m[RG_MEMBERS];
    uint32_t count, k, rows, y_mode, tiles_m, tiles_n, group, full, runs, base, rem, per;
    float* part;  // [slot][column block][BM rows][128]
};

template <int BITS, int RG, int KG>
struct RgCfg {
    static constexpr int BM = 16 * RG, BLOCKS = 2 / KG, LOADERS = 8 / KG;  // LOADERS: wavefronts that move a k tile of A
    static constexpr int LA = (2 * RG + LOADERS - 1) / LOADERS, A_TILE = LA * LOADERS * 1024, A_STAGE = KG * A_TILE;
    static constexpr int LW = (BITS + 3) / 4, W_WAVE = LW * 1024, W_STAGE = 8 * W_WAVE;
    // k tiles of A in flight, and of words: one more where it fits, so that words have two k tiles' time to come at two stages of A
    static constexpr int FIT = 160 * 1024 / (A_STAGE + W_STAGE), ST = FIT < 4 ? FIT : 4;
    static constexpr int SW = ST * A_STAGE + (ST + 1) * W_STAGE <= 160 * 1024 ? ST + 1 : ST;
    static constexpr int W_AT = ST * A_STAGE, STAGES = W_AT + SW * W_STAGE;
    static constexpr int RED_ROWS = BLOCKS == 2 && BM > 128 ? 128 : BM, RED = RED_ROWS * BLOCKS * 132 * 4;
    static constexpr int LDS = STAGES > RED ? STAGES : RED;
    static constexpr int FLIGHT = (ST - 2) * (LA + LW) + (SW > ST ? LW : 0);  // loads that may be in flight at the start of a step
    static_assert(ST >= 2 && LDS <= 160 * 1024 && (SW - 1) * LW + ST * LA < 64, "stages");
};

// Steps s0 .. s0 + steps - 1 of a tile. 512 threads: wavefront w decodes and multiplies 32 columns of 128 (w & 3) over the BM rows of the
// tile. KG 2: one column block, the wavefronts w >> 2 take every other k tile and their sums meet in LDS (tiles half as wide fill the chip
// with half as many pieces of K); KG 1: two column blocks (half the bytes of A a product: from about 1000 rows on).
template <int BITS, int RG, int KG>
__device__ __forceinline__ void rgemm_segment(const RgJob& job, uint32_t tile, uint32_t s0, uint32_t steps, uint32_t slot, bool whole) {
    typedef RgCfg<BITS, RG, KG> C;
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
    const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l32 = lane & 31, hw = threadIdx.x >> 5;
    const uint32_t cg = wave & 3, kg = KG == 2 ? wave >> 2 : 0, blk = KG == 2 ? 0 : wave >> 2, r = lane & 15, g = lane >> 4;
    const uint32_t k = job.k, rows = job.rows;
    uint32_t tm, tn;
    gemm_raster(tile, job.tiles_m, job.tiles_n, job.group, tm, tn);
    uint32_t mi = 0;
    while (mi + 1 < job.count && tn >= job.m[mi + 1].first) mi++;
    const RgMember& mb = job.m[mi];
    const uint32_t n = mb.n, nbs = n / 128, nb0 = (tn - mb.first) * C::BLOCKS, nb = nb0 + blk < nbs ? nb0 + blk : nbs - 1;
    const uint32_t m0 = tm * C::BM;

    const u32x4 xrs = g8_rsrc(mb.xh, rows * k * 2), wrs = g8_rsrc(mb.trellis, (k / 16) * (n / 16) * 32 * BITS);
    const uint32_t lds0 = g8_lds_addr(lds), kt_bytes = 16 * mb.stride_k;
    constexpr uint32_t LOADERS = C::LOADERS;
    const uint32_t lw_id = wave % LOADERS;
    // A piece is 8 rows x 64 channels, chunk c of a row at position g8_perm(c) ^ (row & 7); rows that do not exist lie past the end and
    // read zero
    const uint32_t va = ((m0 + 8 * lw_id + (lane >> 3)) * k + g8_perm<true>((lane & 7) ^ (lane >> 3)) * 8) * 2, a_piece = 16 * LOADERS * k;
    uint32_t vw[C::LW];
#pragma unroll
    for (int j = 0; j < C::LW; j++) {  // the wavefront's words of a k tile: [4 k steps][2 tiles][8 BITS words]
        const uint32_t at = (j * 64 + lane) % (16 * BITS) * 16;
        vw[j] = 4 * (at / (64 * BITS) * mb.stride_k) + at % (64 * BITS);
    }
    const uint32_t w0 = 4 * (nb * mb.stride_nb + 16 * BITS * cg);
    auto ktile = [&](uint32_t t) { return (s0 + (t < steps ? t : steps - 1)) * KG + kg; };  // past the end: the last one again, never used
    auto load_a = [&](uint32_t t, uint32_t st, int j) {
        g8_load_lds16(xrs, lds0 + st * C::A_STAGE + kg * C::A_TILE + (lw_id + LOADERS * j) * 1024, va, ktile(t) * 128 + j * a_piece);
    };
    auto load_w = [&](uint32_t t, uint32_t st, int j) {
        g8_load_lds16(wrs, lds0 + C::W_AT + st * C::W_STAGE + wave * C::W_WAVE + j * 1024, vw[j], w0 + ktile(t) * kt_bytes);
    };
    const unsigned char* wp = lds + C::W_AT + wave * C::W_WAVE + (g * 2 + (r >> 3)) * (32 * BITS) + (r & 7) * (4 * BITS);
    LaneWords<BITS> lw;
    LaneWindows<BITS> win;
    auto words = [&](uint32_t st) {
        const uint32_t* p = (const uint32_t*)(wp + st * C::W_STAGE);
        if constexpr (BITS % 4 == 0) {
#pragma unroll
            for (int i = 0; i < BITS; i += 4) {
                const u32x4 t = *(const u32x4*)(p + i);
                lw.w[i + 1] = t[0], lw.w[i + 2] = t[1], lw.w[i + 3] = t[2], lw.w[i + 4] = t[3];
            }
        } else {
#pragma unroll
            for (int i = 0; i < BITS; i++) lw.w[i + 1] = p[i];
        }
    };
    auto prepare = [&]() {
        lw.w[0] = lane_prev_word_halves(lw.w[BITS]);
        win = lane_windows<BITS>(lw);
    };
    u32x4 op[2][2][2];  // decoded weights of a k tile: [set][row half][k half], 8 values each
    auto decode = [&](int set, int q) {
        uint32_t v = decode_lane_pair<BITS>(lw, win, (q >> 3) & 1, (q >> 2) & 1, q & 3);
        asm volatile("" : "+v"(v));
        op[set][(q >> 3) & 1][(q >> 2) & 1][q & 3] = v;
    };
    uint32_t foff[2];
#pragma unroll
    for (int h = 0; h < 2; h++) foff[h] = r * 128 + ((g8_perm<true>(2 * g + h) ^ (r & 7)) << 4);
    const uint32_t pa0 = lds0 + kg * C::A_TILE;

    f32x4 acc[RG][2];
#pragma unroll
    for (int i = 0; i < RG; i++) acc[i][0] = acc[i][1] = (f32x4){0.f, 0.f, 0.f, 0.f};

    // Step t issues the loads of A of tile t + ST - 1, then the words of tile t + SW + 1; at its start A of tile t and the words of
    // tile t + 2 have come.
#pragma unroll
    for (int t = -C::SW - 1; t < 0; t++) {
        if (t + C::ST - 1 >= 0) {
#pragma unroll
            for (int j = 0; j < C::LA; j++) load_a(t + C::ST - 1, t + C::ST - 1, j);
        }
        if (t < -1) {  // (the words of tile SW go where those of tile 0 lie: once these have been read)
#pragma unroll
            for (int j = 0; j < C::LW; j++) load_w(t + C::SW + 1, t + C::SW + 1, j);
        }
    }
    g8_loads_wait<(C::SW - 2) * C::LW + (C::ST - 1) * C::LA>();  // the words of tiles 0 and 1 (each wavefront reads its own)
    words(0);
    prepare();
#pragma unroll
    for (int q = 0; q < 16; q++) decode(0, q);
    words(1);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int j = 0; j < C::LW; j++) load_w(C::SW, 0, j);

    uint32_t st = 0, sw = 1;  // stages of A of tile t, of the words of tile t + 1
    auto step = [&](auto set_tag, uint32_t t) {
        constexpr int SET = decltype(set_tag)::value, MF = 4 * RG, AHEAD = 2;
        g8_loads_wait<C::FLIGHT>();
        g8_barrier();
        uint32_t at[2] = {pa0 + st * C::A_STAGE + foff[0], pa0 + st * C::A_STAGE + foff[1]};
        asm volatile("" : "+v"(at[0]), "+v"(at[1]));
        const uint32_t st_in = st ? st - 1 : C::ST - 1, sw_in = sw, sw1 = sw + 1 == C::SW ? 0u : sw + 1;
        f16x8 x[AHEAD + 1][2];
        auto rd = [&](int i) {
            for (int h = 0; h < 2; h++) x[i % (AHEAD + 1)][h] = *(const __attribute__((address_space(3))) f16x8*)(uintptr_t)(at[h] + 2048 * i);
        };
#pragma unroll
        for (int i = 0; i < AHEAD; i++) rd(i);
        prepare();
        g8_for<MF>([&](auto f_tag) {
            constexpr int f = decltype(f_tag)::value, i = f / 4, h = f & 1, kh = (f >> 1) & 1, LOADS = C::LA + C::LW;
            if constexpr (f % 4 == 0 && i + AHEAD < RG) rd(i + AHEAD);
            acc[i][h] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, op[SET][h][kh]), x[i % (AHEAD + 1)][kh], acc[i][h], 0, 0, 0);
            asm volatile("" : "+v"(acc[i][h]));
            g8_for<16>([&](auto q) {
                if constexpr (g8_at(decltype(q)::value, 16, 0, MF) == f) decode(SET ^ 1, decltype(q)::value);
            });
            g8_for<LOADS>([&](auto q_tag) {
                constexpr int q = decltype(q_tag)::value;
                if constexpr (g8_at(q, LOADS, 1, C::ST == 2 ? MF / 2 : MF) == f) {
                    if constexpr (q < C::LA)
                        load_a(t + C::ST - 1, st_in, q);
                    else
                        load_w(t + C::SW + 1, sw_in, q - C::LA);
                }
            });
        });
        words(sw1);
        st = st + 1 == C::ST ? 0u : st + 1, sw = sw1;
    };
    for (uint32_t t = 0;;) {
        step(std::integral_constant<int, 0>{}, t);
        if (++t == steps) break;
        step(std::integral_constant<int, 1>{}, t);
        if (++t == steps) break;
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");

    // The sums meet in LDS as rows: [row][column block][132]. A lane's four sums of either row half are four neighbouring columns.
    float* red = (float*)lds;
    constexpr uint32_t PITCH = 132 * C::BLOCKS;
    float* mine = red + r * PITCH + blk * 132 + 32 * cg + 16 * (g >> 1) + 4 * (g & 1);
    auto epilogue = [&](auto emit) {
#pragma unroll
        for (int i0 = 0; i0 < RG; i0 += C::RED_ROWS / 16) {
            __syncthreads();
            if (KG == 1 || kg == 1) {
#pragma unroll
                for (int i = i0; i < RG && i < i0 + C::RED_ROWS / 16; i++)
#pragma unroll
                    for (int h = 0; h < 2; h++) *(f32x4*)(mine + (i - i0) * 16 * PITCH + 8 * h) = acc[i][h];
            }
            __syncthreads();
            if constexpr (KG == 2) {
                if (kg == 0) {
#pragma unroll
                    for (int i = 0; i < RG; i++)
#pragma unroll
                        for (int h = 0; h < 2; h++) {
                            f32x4* p = (f32x4*)(mine + i * 16 * PITCH + 8 * h);
                            *p = acc[i][h] + *p;
                        }
                }
                __syncthreads();
            }
            const uint32_t left = rows - m0 - 16 * i0, most = C::BM - 16 * i0 < C::RED_ROWS ? C::BM - 16 * i0 : C::RED_ROWS, here = left < most ? left : most;
            if (m0 + 16 * i0 < rows) emit(16 * i0, here);
        }
    };
    if (!whole) {
        float* at = job.part + (size_t)slot * (C::BLOCKS * C::BM * 128);
        epilogue([&](uint32_t row0, uint32_t here) {
            for (uint32_t q = hw; q < here * C::BLOCKS; q += 16) {
                const uint32_t row = q / C::BLOCKS, b = q % C::BLOCKS;
                *(f32x4*)(at + ((size_t)b * C::BM + row0 + row) * 128 + 4 * l32) = *(const f32x4*)(red + row * PITCH + b * 132 + 4 * l32);
            }
        });
        return;
    }
    auto run = [&](auto mode_tag) {
        constexpr uint32_t MODE = decltype(mode_tag)::value;
        epilogue([&](uint32_t row0, uint32_t here) {
            // a half wavefront takes one column block's rows (KG 1: the halves of a wavefront one block each), four at a time
            const uint32_t b = C::BLOCKS == 2 ? hw & 1 : 0, h0 = C::BLOCKS == 2 ? hw >> 1 : hw, step_rows = C::BLOCKS == 2 ? 8 : 16;
            const bool live = nb0 + b < nbs;
            const uint32_t col = (live ? nb0 + b : nb0) * 128 + 4 * l32;
            const f32x4 sc = row_scales(mb.svh, col);
            for (uint32_t q0 = h0; q0 < here; q0 += 4 * step_rows) {
                float v[4][4];
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    const uint32_t row = q0 + u * step_rows < (uint32_t)C::RED_ROWS ? q0 + u * step_rows : q0;
                    const f32x4 s = *(const f32x4*)(red + row * PITCH + b * 132 + 4 * l32);
                    v[u][0] = s[0], v[u][1] = s[1], v[u][2] = s[2], v[u][3] = s[3];
                }
                // (the old outputs of all four asked for together: behind a store the next load waits for it)
                u32x4 old[4];
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    const uint32_t row = q0 + u * step_rows;
                    old[u] = live && row < here ? store4_old(mb.y, MODE, (size_t)(m0 + row0 + row) * n + col) : (u32x4){0, 0, 0, 0};
                }
                fwht128_half_wave_rows(v, l32);
#pragma unroll
                for (int u = 0; u < 4; u++) {
#pragma unroll
                    for (int e = 0; e < 4; e++) v[u][e] = v[u][e] * FE_HAD_SCALE * sc[e];
                    const uint32_t row = q0 + u * step_rows;
                    if (live && row < here) store4(mb.y, MODE, (size_t)(m0 + row0 + row) * n + col, v[u], old[u]);
                }
            }
        });
    };
    if (job.y_mode == 0)
        run(std::integral_constant<uint32_t, 0>{});
    else if (job.y_mode == 1)
        run(std::integral_constant<uint32_t, 1>{});
    else if (job.y_mode == 2)
        run(std::integral_constant<uint32_t, 2>{});
    else
        run(std::integral_constant<uint32_t, 3>{});
}

// The first step of run q, counted from the first tile that is not a program's own
__device__ __forceinline__ uint32_t rg_start(const RgJob& job, uint32_t q, uint32_t all) {
    return job.per ? q / job.per * all + q % job.per * all / job.per : sk_start(q, job.base, job.rem);
}

template <int BITS, int RG, int KG>
__device__ __forceinline__ void rgemm_body(const RgJob& job) {
    const uint32_t p = blockIdx.x, all = job.k / (64 * KG);
    // a whole tile is a run of its own
    uint32_t u = p < job.full ? p * all : job.full * all + rg_start(job, p - job.full, all);
    const uint32_t end = p < job.full ? u + all : job.full * all + rg_start(job, p - job.full + 1, all);
    while (u < end) {
        const uint32_t tile = u / all, s0 = u - tile * all, steps = all - s0 < end - u ? all - s0 : end - u;
        rgemm_segment<BITS, RG, KG>(job, tile, s0, steps, p + tile - 2 * job.full, steps == all);
        u += steps;
        if (u < end) __syncthreads();  // the segment's rows in LDS have been read
    }
}

// Every line of the launch's arguments asked for at once, in front of the first use of any (as GEMV_JOB_LINES of k_exl3.hip): a trip to memory
// instead of five, one behind the other.
#define RG_JOB_LINES(job)                                                                                                                    \
    "s"((job).m[0].first), "s"((job).m[1].first), "s"((job).m[2].first), "s"((job).m[3].first), "s"((job).count), "s"((job).k), "s"((job).rows), \
        "s"((job).y_mode), "s"((job).tiles_m), "s"((job).tiles_n), "s"((job).group), "s"((job).full), "s"((job).runs), "s"((job).base),   \
        "s"((job).rem), "s"((job).per), "s"((job).part)

// Finishes the cut tiles: sums the pieces of a row in the order of K, then the output rotation and scale. grid: tiles after the full
// ones x blocks x bm / 8, 256 threads, a half wavefront a row. all: steps of a tile.
extern "C" __global__ __launch_bounds__(256) void exl3_rgemm_reduce(RgJob job, uint32_t bm, uint32_t blocks, uint32_t all) {
    asm volatile("" ::RG_JOB_LINES(job), "s"(bm), "s"(blocks), "s"(all));
    const uint32_t per = bm / 8, l32 = threadIdx.x & 31, c = blockIdx.x / per, row = blockIdx.x % per * 8 + (threadIdx.x >> 5);
    const uint32_t t = c / blocks, b = c % blocks;
    uint32_t tm, tn;
    gemm_raster(job.full + t, job.tiles_m, job.tiles_n, job.group, tm, tn);
    uint32_t mi = 0;
    while (mi + 1 < job.count && tn >= job.m[mi + 1].first) mi++;
    const RgMember& mb = job.m[mi];
    const uint32_t nb = (tn - mb.first) * blocks + b, at = tm * bm + row;
    const uint32_t first = job.per ? t * job.per : sk_owner(t * all, job.base, job.rem);
    const uint32_t last = job.per ? first + job.per - 1 : sk_owner(t * all + all - 1, job.base, job.rem);
    if (first == last || nb >= mb.n / 128 || tm * bm + blockIdx.x % per * 8 >= job.rows) return;  // (one run's: finished there)
    const uint32_t slot = blocks * bm * 128;
    const float* p = job.part + (size_t)(first + t) * slot + ((size_t)b * bm + row) * 128 + 4 * l32;
    const uint32_t col = nb * 128 + 4 * l32;
    const size_t to = (size_t)at * mb.n + col;
    const u32x2 sv = *(const u32x2*)(mb.svh + col);  // (these two on their way beside the pieces)
    const u32x4 old = at < job.rows ? store4_old(mb.y, job.y_mode, to) : (u32x4){0, 0, 0, 0};
    constexpr uint32_t AT_ONCE = 8;  // loads in flight: one at a time the launch took 8.2 us on the 20 pieces of 5120 x 1024 at 128 rows (5.1 now)
    f32x4 sum = *(const f32x4*)p;
    for (uint32_t i0 = 1; i0 <= last - first; i0 += AT_ONCE) {
        f32x4 piece[AT_ONCE];
#pragma unroll
        for (uint32_t i = 0; i < AT_ONCE; i++) piece[i] = *(const f32x4*)(p + (size_t)(first + i0 + i <= last ? i0 + i : i0) * slot);
#pragma unroll
        for (uint32_t i = 0; i < AT_ONCE; i++)
            if (first + i0 + i <= last) sum += piece[i];
    }
    float v[4] = {sum[0], sum[1], sum[2], sum[3]};
    if (at < job.rows) finish_row(v, l32, sv, mb.y, job.y_mode, to, old);
}

#define RGEMM_KERNEL(BITS, RG, KG)                                                                                \
    extern "C" __global__ __launch_bounds__(512, 2) void exl3_rgemm_b##BITS##_r##RG##_k##KG(RgJob job) {         \
        asm volatile("" ::RG_JOB_LINES(job));                                                                     \
        rgemm_body<BITS, RG, KG>(job);                                                                            \
    }
#define RGEMM_ROWS(BITS)                                                                                          \
    RGEMM_KERNEL(BITS, 6, 2) RGEMM_KERNEL(BITS, 8, 2) RGEMM_KERNEL(BITS, 10, 2) RGEMM_KERNEL(BITS, 12, 2)         \
    RGEMM_KERNEL(BITS, 14, 2) RGEMM_KERNEL(BITS, 16, 2)                                                           \
    RGEMM_KERNEL(BITS, 10, 1) RGEMM_KERNEL(BITS, 12, 1) RGEMM_KERNEL(BITS, 14, 1) RGEMM_KERNEL(BITS, 16, 1)
// One code object a width in bits (RG_BITS): sixty unrolled kernels in one take a compiler eight times as long as the next largest source.
// Without RG_BITS the file compiles to one that holds them all.
#ifdef RG_BITS
RGEMM_ROWS(RG_BITS)
#else
RGEMM_ROWS(2)
RGEMM_ROWS(3)
RGEMM_ROWS(4)
RGEMM_ROWS(5)
RGEMM_ROWS(6)
RGEMM_ROWS(8)
#endif
