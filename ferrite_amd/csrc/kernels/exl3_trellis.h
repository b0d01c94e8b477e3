// The EXL3 trellis decode that every kernel shares: the mul1 codebook, a lane's words and states, and the output rotation's
// last step.
//
// The trellis of a 16x16 tile is a cyclic stream of 256 * BITS bits, most significant bit of each u32 first; position t
// owns the 16-bit state ending at stream bit (t + 1) * BITS (crates/fe-exl3/src/cpu.rs:12-23). Position
// t = 8 * f + i sits at row k = 2 (f & 3) + (i & 1) + 8 ((i >> 1) & 1), column n = (f >> 2) + 8 (i >> 2) of the tile
// (crates/fe-exl3/src/format.rs:146-156). A state decodes to fp16 by the mul1 codebook
// (crates/fe-exl3/src/cpu.rs:25-43, kernels/k-exl3/src/util.rs:76-85).
#pragma once
#include "kcommon.h"

// ---- the mul1 codebook ------------------------------------------------------------------------------------------

// x = state * 0x83DCD12D mod 2^32 for the 16-bit state in the low (HI = 0) or high (HI = 1) half of r; the other half
// of r may hold anything. On gfx950 v_mul_lo_u32 issues at the same rate as the other 3-operand integer instructions,
// while the shift or mask that isolates the state is one of the double-rate simple instructions.
template <int HI>
__device__ __forceinline__ uint32_t mul1_x(uint32_t r) {
    uint32_t s = HI ? (r >> 16) : (r & 0xffffu);
    return s * 0x83DCD12Du;
}

// Two codebook values as packed fp16 (x0's in the low half): 0x6400 + byte sum is fp16(1024 + sum); one fused
// fp16 multiply-add by 0x1eee with 0xc931 added, a single rounding per value.
__device__ __forceinline__ uint32_t mul1_finish2(uint32_t x0, uint32_t x1) {
    uint32_t h = __builtin_amdgcn_sad_u8(x0, 0u, 0x64006400u);
    h = __builtin_amdgcn_sad_hi_u8(x1, 0u, h);
    f16x2 v = __builtin_bit_cast(f16x2, h);
    const f16x2 c1 = __builtin_bit_cast(f16x2, 0x1eee1eeeu);
    const f16x2 c2 = __builtin_bit_cast(f16x2, 0xc931c931u);
    f16x2 o = __builtin_elementwise_fma(v, c1, c2);
    return __builtin_bit_cast(uint32_t, o);
}

__device__ __forceinline__ uint32_t decode2_mul1(uint32_t s0, uint32_t s1) {
    return mul1_finish2(mul1_x<0>(s0), mul1_x<0>(s1));
}

// ---- the lane mapping and the decode ----------------------------------------------------------------------
//
// A program works on one 128-column block at a time; 256 threads = 4 wavefronts, wavefront w owning tiles 2w, 2w + 1 of
// the block's 8. A wavefront's load step covers 4 consecutive k steps of its two tiles: lane L = 16 g + r reads k step g,
// tile r & 1, the BITS words of fragment lanes 4q .. 4q + 3 (q = r >> 1) plus the word before them, which is all its 32
// states need. (The tiles alternate over the lanes, so that the word before, the last one of lane q - 1 of the same tile, is two lanes away
// in the 16, also at q = 0: lane_prev_word, one instruction where tiles in the two halves of the 16 lanes take three. The kernels whose words come
// through LDS keep tile r >> 3, q = r & 7: alternating they read them 2 % slower, prompts of 203 rows.) Those states are rows n = q and n = q + 8 of
// the tile over all 16 k, so after decoding the lane holds, for each of the two, the 16 values as two 8-value MFMA operands (k 0..7 and k 8..15) in k
// order. v_mfma_f32_16x16x32_f16 then sums over the 4 k steps: A = decoded weights (row r), B = 16 rotated input rows (column = input row), and the
// accumulators of lane L are rows 4 g .. 4 g + 3 of A (columns q = 2 g, 2 g + 1 of both tiles), input row r; lane_cols makes four neighbouring
// columns of them.

template <int BITS>
struct LaneWords {
    uint32_t w[BITS + 1];  // w[0] = the word before the lane's run
};

template <int BITS>
__device__ __forceinline__ LaneWords<BITS> load_lane_words(const uint32_t* run, const uint32_t* prev) {
    LaneWords<BITS> r;
    r.w[0] = __builtin_nontemporal_load(prev);
    if constexpr (BITS == 1) {
        r.w[1] = __builtin_nontemporal_load(run);
    } else if constexpr (BITS == 2) {
        u32x2_a4 t = __builtin_nontemporal_load((const u32x2_a4*)run);
        r.w[1] = t[0], r.w[2] = t[1];
    } else if constexpr (BITS == 3) {
        u32x3_a4 t = __builtin_nontemporal_load((const u32x3_a4*)run);
        r.w[1] = t[0], r.w[2] = t[1], r.w[3] = t[2];
    } else {
        u32x4_a4 t = __builtin_nontemporal_load((const u32x4_a4*)run);
        r.w[1] = t[0], r.w[2] = t[1], r.w[3] = t[2], r.w[4] = t[3];
        if constexpr (BITS == 5) {
            r.w[5] = __builtin_nontemporal_load(run + 4);
        } else if constexpr (BITS == 6) {
            u32x2_a4 u = __builtin_nontemporal_load((const u32x2_a4*)(run + 4));
            r.w[5] = u[0], r.w[6] = u[1];
        } else if constexpr (BITS == 7) {
            u32x3_a4 u = __builtin_nontemporal_load((const u32x3_a4*)(run + 4));
            r.w[5] = u[0], r.w[6] = u[1], r.w[7] = u[2];
        } else if constexpr (BITS == 8) {
            u32x4_a4 u = __builtin_nontemporal_load((const u32x4_a4*)(run + 4));
            r.w[5] = u[0], r.w[6] = u[1], r.w[7] = u[2], r.w[8] = u[3];
        }
    }
    return r;
}

// The lane's local stream: bit 0 = most significant bit of w[0]; local position U (0..31) owns the 16 bits ending at local
// bit (U + 1) * BITS + 32. A state either lies inside one word (one extract), or straddles the boundary between w[i - 1]
// and w[i]: all states that straddle one boundary are cut out of one 32-bit window over it (low half of w[i - 1], high
// half of w[i]): BITS funnel shifts a load step instead of one per state or per pair of states.
template <int BITS>
struct LaneWindows {
    uint32_t b[BITS + 1];  // b[i], i >= 1: the window over the boundary in front of w[i]
};
template <int BITS>
__device__ __forceinline__ LaneWindows<BITS> lane_windows(const LaneWords<BITS>& lw) {
    LaneWindows<BITS> win;
    win.b[0] = 0;
#pragma unroll
    for (int i = 1; i <= BITS; i++) {
        uint32_t r = __builtin_amdgcn_alignbit(lw.w[i - 1], lw.w[i], 16);
        // opaque to the optimizer, which would otherwise fold window and extract into a funnel shift and a mask per state
        asm("" : "+v"(r));
        win.b[i] = r;
    }
    return win;
}

// x = state * MUL1 of local position U.
template <int BITS, int U>
__device__ __forceinline__ uint32_t lane_x(const LaneWords<BITS>& lw, const LaneWindows<BITS>& win) {
    constexpr int end = (U + 1) * BITS + 32, wi = end / 32, r = end % 32;
    uint32_t state;
    if constexpr (r == 0)
        state = lw.w[wi - 1] & 0xffffu;
    else if constexpr (r == 16)
        state = lw.w[wi] >> 16;
    else if constexpr (r > 16)
        state = __builtin_amdgcn_ubfe(lw.w[wi], 32 - r, 16);
    else
        state = __builtin_amdgcn_ubfe(win.b[wi], 16 - r, 16);
    return state * 0x83DCD12Du;
}

// The lane's 32 values as MFMA operands op[h][kh]: rows n = q + 8 h of the tile, k = 8 kh .. 8 kh + 7 in order.
// Local position u = 8 c + i (fragment lane 4q + c, value i) is k = 2c + (i & 1) + 8 ((i >> 1) & 1), n half i >> 2.
template <int BITS>
__device__ __forceinline__ void decode_lane(const LaneWords<BITS>& lw, f16x8 (&op)[2][2]) {
    const LaneWindows<BITS> win = lane_windows<BITS>(lw);
#define FE_PAIR(H, KH, C) mul1_finish2(lane_x<BITS, 8 * (C) + 2 * (KH) + 4 * (H)>(lw, win), lane_x<BITS, 8 * (C) + 2 * (KH) + 4 * (H) + 1>(lw, win))
#define FE_OP(H, KH)                                                                             \
    {                                                                                            \
        u32x4 t = {FE_PAIR(H, KH, 0), FE_PAIR(H, KH, 1), FE_PAIR(H, KH, 2), FE_PAIR(H, KH, 3)};  \
        op[H][KH] = __builtin_bit_cast(f16x8, t);                                                \
    }
    FE_OP(0, 0) FE_OP(0, 1) FE_OP(1, 0) FE_OP(1, 1)
#undef FE_OP
#undef FE_PAIR
}

// Two of the 32 values alone, as packed fp16: values 2 c, 2 c + 1 of decode_lane's op[h][kh]. (Constant arguments.)
template <int BITS>
__device__ __forceinline__ uint32_t decode_lane_pair(const LaneWords<BITS>& lw, const LaneWindows<BITS>& win, int h, int kh, int c) {
    auto x = [&](int u) {  // lane_x of position u
        const int end = (u + 1) * BITS + 32, wi = end / 32, r = end % 32;
        const uint32_t s = r == 0    ? lw.w[wi - 1] & 0xffffu
                           : r == 16 ? lw.w[wi] >> 16
                           : r > 16  ? __builtin_amdgcn_ubfe(lw.w[wi], 32 - r, 16)
                                     : __builtin_amdgcn_ubfe(win.b[wi], 16 - r, 16);
        return s * 0x83DCD12Du;
    };
    const int u = 8 * c + 2 * kh + 4 * h;
    return mul1_finish2(x(u), x(u + 1));
}

// Store 4 consecutive outputs. mode: 0 bf16, 1 f32, 2 bf16 y += v (f32 add, one rounding), 3 f32 y += v.
// (kernels/k-exl3/src/gemv.rs:122-145) old: what stands there, for the adding modes (store4_old), read ahead by the launches that only add sums: behind them
// it is one more trip to memory (decode of 40 rows 112.8 -> 111.5 us; in the GEMV's own finish it gains nothing and costs registers).
__device__ __forceinline__ u32x4 store4_old(const void* y, uint32_t mode, size_t i) {
    u32x4 o = {0, 0, 0, 0};
    if (mode == 3) o = *(const u32x4*)((const float*)y + i);
    if (mode == 2) {
        const u32x2 t = *(const u32x2*)((const uint16_t*)y + i);
        o[0] = t[0], o[1] = t[1];
    }
    return o;
}
__device__ __forceinline__ void store4(void* y, uint32_t mode, size_t i, float (&v)[4], u32x4 old) {
    if (mode & 1) {
        f32x4 o = {v[0], v[1], v[2], v[3]};
        if (mode & 2) o += __builtin_bit_cast(f32x4, old);
        *(f32x4*)((float*)y + i) = o;
    } else {
        if (mode & 2) {
            v[0] += __uint_as_float(old[0] << 16), v[1] += __uint_as_float(old[0] & 0xffff0000u);
            v[2] += __uint_as_float(old[1] << 16), v[3] += __uint_as_float(old[1] & 0xffff0000u);
        }
        u32x2 o = {pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
        *(u32x2*)((uint16_t*)y + i) = o;
    }
}
__device__ __forceinline__ void store4(void* y, uint32_t mode, size_t i, float (&v)[4]) {
    if (mode & 1) {
        float* p = (float*)y + i;
        f32x4 o = {v[0], v[1], v[2], v[3]};
        if (mode & 2) o += *(const f32x4*)p;
        *(f32x4*)p = o;
    } else {
        uint32_t* p = (uint32_t*)((uint16_t*)y + i);
        if (mode & 2) {
            uint32_t a = p[0], b = p[1];
            v[0] += __uint_as_float(a << 16), v[1] += __uint_as_float(a & 0xffff0000u);
            v[2] += __uint_as_float(b << 16), v[3] += __uint_as_float(b & 0xffff0000u);
        }
        u32x2 o = {pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
        *(u32x2*)p = o;
    }
}

// H over the 128 sums of a row (4 a lane of a half wavefront), * svh / sqrt(128), stored. (gemv.rs:172-180) s: the lane's four output scales (fp16).
__device__ __forceinline__ void finish_row(float (&v)[4], uint32_t l32, u32x2 s, void* y, uint32_t mode, size_t at, u32x4 old) {
    fwht128_half_wave(v, l32);
    v[0] = v[0] * FE_HAD_SCALE * f16_bits_to_f32(s[0] & 0xffff);
    v[1] = v[1] * FE_HAD_SCALE * f16_bits_to_f32(s[0] >> 16);
    v[2] = v[2] * FE_HAD_SCALE * f16_bits_to_f32(s[1] & 0xffff);
    v[3] = v[3] * FE_HAD_SCALE * f16_bits_to_f32(s[1] >> 16);
    store4(y, mode, at, v, old);
}
__device__ __forceinline__ void finish_row(float (&v)[4], uint32_t l32, const uint16_t* svh, uint32_t col, void* y,
                                           uint32_t mode, size_t at) {
    finish_row(v, l32, *(const u32x2*)(svh + col), y, mode, at, store4_old(y, mode, at));
}

// The lane's four output scales as finish_row applies them, for callers that finish many rows of the same columns.
__device__ __forceinline__ f32x4 row_scales(const uint16_t* svh, uint32_t col) {
    u32x2 s = *(const u32x2*)(svh + col);
    return (f32x4){f16_bits_to_f32(s[0] & 0xffff), f16_bits_to_f32(s[0] >> 16), f16_bits_to_f32(s[1] & 0xffff),
                   f16_bits_to_f32(s[1] >> 16)};
}
// (Moves that leave no lane out and read no old value: with one, each cost a move of zero in front, five instructions a step instead of three or one.)
// The last word of the lane two before, around the 16 lanes of a DPP row: the word before the lane's run where the two tiles of a k step alternate
// over the lanes.
__device__ __forceinline__ uint32_t lane_prev_word(uint32_t last) { return (uint32_t)__builtin_amdgcn_mov_dpp((int)last, 0x122, 0xf, 0xf, true); }
// The same where lanes 0..7 have the one tile and lanes 8..15 the other: lane i takes lane i - 1 (row_shr:1) or, at q = 0, lane i + 7 (row_ror:9).
__device__ __forceinline__ uint32_t lane_prev_word_halves(uint32_t last) {
    const uint32_t shr = (uint32_t)__builtin_amdgcn_mov_dpp((int)last, 0x111, 0xf, 0xf, true);
    const uint32_t ror = (uint32_t)__builtin_amdgcn_mov_dpp((int)last, 0x129, 0xf, 0xf, true);
    return (threadIdx.x & 7) ? shr : ror;
}
// A lane's accumulators (rows 4 g .. 4 g + 3 of A: columns 2 g, 2 g + 1 of tiles 0 and 1, the tiles alternating) as four neighbouring columns: 16 (g
// & 1) + 4 (g >> 1) .. + 3 of the wavefront's 32 (+ 8 h). Lanes of even g give their tile 1 to the lanes 16 further on for those lanes' tile 0.
__device__ __forceinline__ f32x4 lane_cols(f32x4 a) {
    typedef uint32_t pair_t __attribute__((ext_vector_type(2)));
    const pair_t lo = __builtin_bit_cast(pair_t, __builtin_amdgcn_permlane16_swap(__float_as_uint(a[0]), __float_as_uint(a[1]), false, false));
    const pair_t hi = __builtin_bit_cast(pair_t, __builtin_amdgcn_permlane16_swap(__float_as_uint(a[2]), __float_as_uint(a[3]), false, false));
    return (f32x4){__uint_as_float(lo[0]), __uint_as_float(hi[0]), __uint_as_float(lo[1]), __uint_as_float(hi[1])};
}
