// NVFP4 linear for gfx950: e2m1 codes (element 2i in the low nibble of byte i), one e4m3 scale per 16 elements along
// K, an fp32 scale per output column. Activations are quantized to the same format first (the reference's prompt path
// is W4A4, crates/fe-fp4/src/lib.rs:512-530), then the GEMM runs over the quantized operands.
//
// gfx950's block-scaled MFMA takes e8m0 scales per 32 elements, which cannot express e4m3 per 16. A product
// e2m1 x e4m3 has at most 6 significant bits and lies in [2^-10, 2688], so a small power of two times that value is an
// exact, normal fp16 number: both operands are expanded to fp16 (activations as 2 * code value * block scale, weights
// as 8 * ...) and multiplied on the f16 MFMA with fp32 accumulation, which reproduces the block-scaled dot product up
// to summation order; the factor 16 comes off in the epilogue.
#include <type_traits>

#include "gemm8.h"

// ---- number formats ----------------------------------------------------------------------------------------------------

// Exact e4m3 (fn) -> f32 for non-NaN codes. (crates/fe-fp4/src/format.rs:19-27)
__device__ __forceinline__ float e4m3_to_f32(uint32_t b) {
    uint32_t e = (b >> 3) & 15, mn = b & 7;
    float v = e == 0 ? (float)mn * (1.0f / 512.0f) : __uint_as_float(((e + 120) << 23) | (mn << 20));
    return (b & 0x80) ? -v : v;
}

// a >= 0 -> e4m3 code, round to nearest even, saturating to 448 (0x7e); NaN -> 0x7f.
// (cvt.rn.satfinite.e4m3x2.f32; crates/fe-fp4/src/format.rs:57-63)
__device__ __forceinline__ uint32_t f32_to_e4m3_pos(float a) {
    if (a != a) return 0x7f;
    if (a >= 448.0f) return 0x7e;
    if (a < 0.015625f) return (uint32_t)__builtin_rintf(a * 512.0f);  // subnormals count 2^-9; 8 is the first normal
    uint32_t b = __float_as_uint(a);
    b += 0x7ffffu + ((b >> 20) & 1u);  // nearest even at 3 mantissa bits
    uint32_t c = (((b >> 23) - 120) << 3) | ((b >> 20) & 7u);
    return c > 0x7e ? 0x7e : c;
}

// f32 -> e2m1 code, round to nearest with ties to the even code, saturating to +-6.
// (cvt.rn.satfinite.e2m1x2.f32; crates/fe-fp4/src/format.rs:66-69)
__device__ __forceinline__ uint32_t f32_to_e2m1(float x) {
    float a = __builtin_fabsf(x);
    uint32_t c = (a > 0.25f) + (a >= 0.75f) + (a > 1.25f) + (a >= 1.75f) + (a > 2.5f) + (a >= 3.5f) + (a > 5.0f);
    return c | ((__float_as_uint(x) >> 28) & 8u);
}

// The same conversion for two values at once in hardware: byte `BYTE` of `old` becomes e2m1(a) | e2m1(b) << 4
// (v_cvt_scalef32_pk_fp4_f32 with scale 1). Checked against f32_to_e2m1 on the GPU for every bf16 value, every f32 with
// an exponent of 2^-5 .. 2^4 (all code boundaries and ties), the smallest and the largest magnitudes, infinities, both
// signs: no difference. A NaN is the one input the instruction treats otherwise (largest magnitude, where the
// definition's compare chain and the reference's table search give magnitude 0), so a NaN goes in as a zero of its sign.
__device__ __forceinline__ float e2m1_nan_to_zero(float x) {
    return x == x ? x : __uint_as_float(__float_as_uint(x) & 0x80000000u);
}
template <int BYTE>
__device__ __forceinline__ uint32_t f32x2_to_e2m1_byte(uint32_t old, float a, float b) {
    return __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(old, e2m1_nan_to_zero(a), e2m1_nan_to_zero(b), 1.0f, BYTE);
}

// fp16 of twice the magnitude of the 8 e2m1 magnitudes: 0, 1, 2, 3, 4, 6, 8, 12; every low byte is zero, the high
// bytes are this table.
#define E2M1X2_HI_LO 0x42403c00u  // magnitudes 0..3 -> 0x00, 0x3c, 0x40, 0x42
#define E2M1X2_HI_HI 0x4a484644u  // magnitudes 4..7 -> 0x44, 0x46, 0x48, 0x4a

// 8 codes of one u32 -> 4 packed fp16 pairs (2 * value), elements in order.
__device__ __forceinline__ void e2m1x8_to_f16(uint32_t w, uint32_t (&out)[4]) {
    uint32_t sel_e = w & 0x07070707u;         // even elements (low nibbles) as byte selectors
    uint32_t sel_o = (w >> 4) & 0x07070707u;  // odd elements
    uint32_t hb_e = __builtin_amdgcn_perm(E2M1X2_HI_HI, E2M1X2_HI_LO, sel_e);
    uint32_t hb_o = __builtin_amdgcn_perm(E2M1X2_HI_HI, E2M1X2_HI_LO, sel_o);
    hb_e |= (w << 4) & 0x80808080u;  // sign: bit 3 of the nibble -> bit 7 of the fp16 high byte
    hb_o |= w & 0x80808080u;
    // pair i = (even element i, odd element i): bytes [0, hb_e.i, 0, hb_o.i]; selector 0x0c yields a zero byte
    out[0] = __builtin_amdgcn_perm(hb_o, hb_e, 0x040c000cu);
    out[1] = __builtin_amdgcn_perm(hb_o, hb_e, 0x050c010cu);
    out[2] = __builtin_amdgcn_perm(hb_o, hb_e, 0x060c020cu);
    out[3] = __builtin_amdgcn_perm(hb_o, hb_e, 0x070c030cu);
}

// Positive e4m3 scale -> the same value as packed fp16 (both halves). (b << 7) read as fp16 is value * 2^-8 for
// normal and subnormal codes alike; the multiply by 256 is exact and renormalises.
__device__ __forceinline__ f16x2 e4m3_to_f16x2(uint32_t b) {
    uint32_t h = (b & 0x7f) << 7;
    f16x2 v = __builtin_bit_cast(f16x2, h | (h << 16));
    const f16x2 c = {(_Float16)256.0f, (_Float16)256.0f};
    return v * c;
}

// Weights through the hardware conversion. v_cvt_scalef32_pk_f16_fp4 turns the two e2m1 codes of one byte into fp16 and
// multiplies by a power of two: it takes only the exponent of its f32 scale operand (measured: scale 1.5 gives x1, 448
// gives x256). An e4m3 block scale is 2^(max(e, 1) - 7) * t / 8 with t = m (+ 8 for a normal number), so a weight is
// cvt(code, 2^(max(e, 1) - 7)) * t / 8; code * t has at most 6 significant bits and is exact in fp16. The kernels keep
// the factor 8 (weights as code * 2^E * t, below 23040) and take it off with alpha in the epilogue.
struct Fp4Scale {
    float pow2;  // 2^(max(e, 1) - 7) as f32
    f16x2 t;     // (t, t) as fp16
};
__device__ __forceinline__ Fp4Scale fp4_scale(uint32_t b) {  // b: e4m3 code, sign bit clear
    uint32_t e = b >> 3, e1 = e < 1 ? e : 1;
    Fp4Scale s;
    s.pow2 = __uint_as_float(((e > 1 ? e : 1) + 120) << 23);
    _Float16 t = (_Float16)(uint16_t)((b & 7) | (e1 << 3));
    s.t = (f16x2){t, t};
    return s;
}
// Both forms of all 128 positive e4m3 codes as a 1 KB table in LDS (fp4_scale is about ten vector instructions per 16
// weights; a lookup is two and an LDS read). Filled by the first 128 threads; a barrier must follow before the first lookup.
__device__ __forceinline__ void fp4_scale_lut_fill(u32x2* lut) {
    if (threadIdx.x < 128) {
        Fp4Scale s = fp4_scale(threadIdx.x);
        lut[threadIdx.x] = (u32x2){__float_as_uint(s.pow2), __builtin_bit_cast(uint32_t, s.t)};
    }
}
// at = 8 x the scale's code (the table's byte offset)
__device__ __forceinline__ Fp4Scale fp4_scale_lut(const u32x2* lut, uint32_t at) {
    const u32x2 e = *(const u32x2*)((const char*)lut + at);
    const uint32_t t = e[1];  // (a bit cast straight from the vector's element reads the vector's first bytes)
    Fp4Scale s;
    s.pow2 = __uint_as_float(e[0]), s.t = __builtin_bit_cast(f16x2, t);
    return s;
}
// 8 codes of one u32 -> 8 fp16 (code * 2^E * t), elements in order
__device__ __forceinline__ u32x4 fp4x8_to_f16(uint32_t w, Fp4Scale s) {
    u32x4 o;
    o[0] = __builtin_bit_cast(uint32_t, (f16x2)(__builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, s.pow2, 0) * s.t));
    o[1] = __builtin_bit_cast(uint32_t, (f16x2)(__builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, s.pow2, 1) * s.t));
    o[2] = __builtin_bit_cast(uint32_t, (f16x2)(__builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, s.pow2, 2) * s.t));
    o[3] = __builtin_bit_cast(uint32_t, (f16x2)(__builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, s.pow2, 3) * s.t));
    return o;
}

// ---- activation quantizer ------------------------------------------------------------------------------------------

// Ferrite's tiled scale layout [(rows / 128)][(kb / 8)][128][8] (crates/fe-fp4/src/format.rs:98-111).
__device__ __forceinline__ uint32_t sf_tiled(uint32_t row, uint32_t b, uint32_t kb) {
    return ((row >> 7) * (kb >> 3) + (b >> 3)) * 1024 + (row & 127) * 8 + (b & 7);
}

// A block of 16 bf16 values (r0: 0..7, r1: 8..15): sf = e4m3(amax * (1/6) * g), q = e2m1(x * (g / sf)), and o = 2 * code value * block scale as fp16.
struct Fp4Block {
    u32x2 q;
    uint32_t s8;
    u32x4 o[2];
};
// Without a NaN among the values: their magnitudes as bf16 bits are in order, so the largest is a maximum of 16-bit integers, and the conversions are the
// hardware's; a block with a NaN (a magnitude above infinity's) or an infinity, whose product with the multiplier may be one (g of 0, or so small
// that g / sf is 0), goes through e2m1_nan_to_zero.
__device__ __forceinline__ Fp4Block fp4_quant_block(u32x4 r0, u32x4 r1, float g) {
    typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
    u16x2 top = {0, 0};
#pragma unroll
    for (int j = 0; j < 4; j++) {
        top = __builtin_elementwise_max(top, __builtin_bit_cast(u16x2, r0[j] & 0x7fff7fffu));
        top = __builtin_elementwise_max(top, __builtin_bit_cast(u16x2, r1[j] & 0x7fff7fffu));
    }
    uint32_t amax = top[0] > top[1] ? top[0] : top[1];
    const bool special = amax >= 0x7f80u;
    if (amax > 0x7f80u) {  // the largest of the others
        amax = 0;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const uint32_t w = j < 4 ? r0[j & 3] : r1[j & 3], lo = w & 0x7fffu, hi = (w >> 16) & 0x7fffu;
            if (lo <= 0x7f80u && lo > amax) amax = lo;
            if (hi <= 0x7f80u && hi > amax) amax = hi;
        }
    }
    Fp4Block out;
    out.s8 = f32_to_e4m3_pos(__uint_as_float(amax << 16) * (1.0f / 6.0f) * g);
    float sv = e4m3_to_f32(out.s8);
    float mul = sv > 0.f ? g / sv : 0.f;
    const f16x2 sc = e4m3_to_f16x2(out.s8);
    const bool careful = special || !(mul <= 3.402823466e38f);  // (0 times infinity, on either side)
#pragma unroll
    for (int w = 0; w < 2; w++) {
        float f[8];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const uint32_t v = w ? r1[j] : r0[j];
            f[2 * j] = __uint_as_float(v << 16) * mul, f[2 * j + 1] = __uint_as_float(v & 0xffff0000u) * mul;
        }
        if (careful) {
#pragma unroll
            for (int j = 0; j < 8; j++) f[j] = e2m1_nan_to_zero(f[j]);
        }
        uint32_t q = 0;
        q = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(q, f[0], f[1], 1.0f, 0);
        q = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(q, f[2], f[3], 1.0f, 1);
        q = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(q, f[4], f[5], 1.0f, 2);
        q = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(q, f[6], f[7], 1.0f, 3);
        out.q[w] = q;
        const f16x2 v0 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(q, 2.0f, 0) * sc, v1 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(q, 2.0f, 1) * sc;
        const f16x2 v2 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(q, 2.0f, 2) * sc, v3 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(q, 2.0f, 3) * sc;
        out.o[w] = (u32x4){__builtin_bit_cast(uint32_t, v0), __builtin_bit_cast(uint32_t, v1), __builtin_bit_cast(uint32_t, v2), __builtin_bit_cast(uint32_t, v3)};
    }
    return out;
}
// Block b of row `row` where fe_fp4_quant leaves it.
__device__ __forceinline__ void fp4_store_block(const Fp4Block& v, uint8_t* codes, uint8_t* sf, _Float16* aq, uint32_t row, uint32_t b, uint32_t k) {
    *(u32x2*)(codes + (size_t)row * (k >> 1) + b * 8) = v.q;
    sf[sf_tiled(row, b, k >> 4)] = (uint8_t)v.s8;
    u32x4* ap = (u32x4*)(aq + (size_t)row * k + b * 16);
    ap[0] = v.o[0], ap[1] = v.o[1];
}

// bf16 x[M][ldx] -> codes [M][K/2], e4m3 block scales (tiled layout), and the dequantized operand the GEMM reads:
// aq[M][K] fp16 = 2 * code value * block scale. One thread per 16-element block: grid ceil(M * K / 16 / 256), 256 threads.
// (kernels/k-fp4/src/lib.rs:162-197; CPU form crates/fe-fp4/src/format.rs:72-90)
extern "C" __global__ __launch_bounds__(256) void fe_fp4_quant(uint8_t* codes, uint8_t* sf, _Float16* aq, const uint16_t* x,
                                                               uint32_t m, uint32_t k, uint32_t ldx, float g) {
    uint32_t i = blockIdx.x * 256 + threadIdx.x;
    uint32_t kb = k >> 4;
    if (i >= m * kb) return;
    uint32_t row = i / kb, b = i - row * kb;
    const u32x4* p = (const u32x4*)(x + (size_t)row * ldx + b * 16);
    fp4_store_block(fp4_quant_block(p[0], p[1], g), codes, sf, aq, row, b, k);
}

// ---- GEMM --------------------------------------------------------------------------------------------------------------

// An e4m3 scale (sign bit clear) as packed fp16, both halves, times 2^-8: the code's bits shifted to fp16's place, exact
// for normal and subnormal codes alike. The weight's conversion carries the 2^8.
__device__ __forceinline__ f16x2 fp4_scale_2m8(uint32_t b) { return __builtin_bit_cast(f16x2, b * 0x00800080u); }
// 8 codes of one u32 -> 8 fp16 (code * scale), elements in order: one instruction a weight
__device__ __forceinline__ f16x8 fp4x8_scaled(uint32_t w, f16x2 s) {
    u32x4 o;
    o[0] = __builtin_bit_cast(uint32_t, (f16x2)(__builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 256.0f, 0) * s));
    o[1] = __builtin_bit_cast(uint32_t, (f16x2)(__builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 256.0f, 1) * s));
    o[2] = __builtin_bit_cast(uint32_t, (f16x2)(__builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 256.0f, 2) * s));
    o[3] = __builtin_bit_cast(uint32_t, (f16x2)(__builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 256.0f, 3) * s));
    return __builtin_bit_cast(f16x8, o);
}

// Weight operand of the GEMM: codes and scales of a k tile as they lie in memory, [BN rows][32 bytes of codes] and then [BN
// rows][4 scales] in LDS. Addressed through strides, so both the row-major layout of the format and the k-tile-major layout
// of an uploaded linear ([n / 128][k / 64][128 rows][32 bytes of codes | 4 scales], one contiguous 4.5 KB read per 128 rows
// and k tile) are read by the same kernel. An odd count of 128-row tiles: the last program reads its first tile twice.
template <class T>
struct Fp4Packed {
    static constexpr bool kPerm = true;
    static constexpr int STAGE = T::BN * 36, LOADS = 2;
    u32x4 rw, rs;
    uint32_t wv, sv, w_skt, s_skt;
    struct Raw {
        u32x2 c;
        f16x2 s;
    };
    __device__ __forceinline__ void setup(const uint8_t* w, const uint8_t* sw, uint32_t n, uint32_t k, uint32_t n0, uint32_t w_snt,
                                          uint32_t w_skt_, uint32_t w_sr, uint32_t s_snt, uint32_t s_skt_, uint32_t s_sr) {
        const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nts = n / 128;
        auto at = [&](uint32_t row, uint32_t snt, uint32_t sr) {
            uint32_t nt = (n0 + row) / 128;
            nt = nt < nts ? nt : nts - 1;
            return nt * snt + (row & 127) * sr;
        };
        rw = g8_rsrc(w, n * (k / 2)), rs = g8_rsrc(sw, n * (k / 16));
        wv = at((wave % (T::BN / 32)) * 32 + lane / 2, w_snt, w_sr) + (lane & 1) * 16;
        sv = at((wave % (T::BN / 64)) * 64 + lane, s_snt, s_sr);
        w_skt = w_skt_, s_skt = s_skt_;
    }
    // (fewer pieces than wavefronts: the others move one again)
    __device__ __forceinline__ void issue(uint32_t kt, uint32_t dst, int j, uint32_t wave) const {
        if (j == 0)
            g8_load_lds16(rw, dst + (wave % (T::BN / 32)) * 1024, wv, kt * w_skt);
        else
            g8_load_lds4(rs, dst + T::BN * 32 + (wave % (T::BN / 64)) * 256, sv, kt * s_skt);
    }
    __device__ __forceinline__ Raw read(const unsigned char* st, uint32_t row, uint32_t g) const {
        Raw r;
        r.c = *(const u32x2*)(st + row * 32 + 8 * g);
        r.s = fp4_scale_2m8(__builtin_amdgcn_ubfe(*(const uint32_t*)(st + T::BN * 32 + row * 4), 8 * g, 8));
        return r;
    }
    __device__ __forceinline__ f16x8 expand(const Raw& r, int kk) const { return fp4x8_scaled(kk ? r.c[1] : r.c[0], r.s); }
};

// The fp16 operands of the GEMM are 2 x the quantized activation and the quantized weight; the GEMV's carry 8 x the weight.
#define FP4_GEMM_SCALE 0.5f
#define FP4_OPERAND_SCALE 0.0625f

// One row piece of the output: 4 columns from `col` of row `grow`, bf16((sum) * alpha) (+ res: bf16(bf16(.) + res)).
// (adds, old: whether a residual is added, and its four values)
__device__ __forceinline__ void fp4_store4(uint16_t* c, bool adds, u32x2 old, size_t at, const float (&v)[4], f32x4 al) {
    u32x2 o = {pack_bf16x2(v[0] * al[0], v[1] * al[1]), pack_bf16x2(v[2] * al[2], v[3] * al[3])};
    if (adds) {
#pragma unroll
        for (int e = 0; e < 2; e++)
            o[e] = pack_bf16x2(bf16_bits_to_f32(o[e] & 0xffff) + bf16_bits_to_f32(old[e] & 0xffff),
                               bf16_bits_to_f32(o[e] >> 16) + bf16_bits_to_f32(old[e] >> 16));
    }
    *(u32x2*)(c + at) = o;
}
__device__ __forceinline__ void fp4_store4(uint16_t* c, const uint16_t* res, size_t at, const float (&v)[4], f32x4 al) {
    fp4_store4(c, res != nullptr, res ? *(const u32x2*)(res + at) : (u32x2){0, 0}, at, v, al);
}

// ---- FP8 (e4m3, one scale per tensor) -------------------------------------------------------------------------------------

// The two e4m3 codes of the low (HI = 0) or high half of w as packed fp16, exact (hardware conversion, scale 1).
__device__ __forceinline__ uint32_t e4m3x2_to_f16(uint32_t w, int hi) {
    f16x2 v = hi ? __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w, 1.0f, true) : __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w, 1.0f, false);
    return __builtin_bit_cast(uint32_t, v);
}

// Two f32 -> two e4m3 codes in bytes 0, 1 (HI: 2, 3) of old: round to nearest even, saturating, either sign; NaN -> 0x7f. The hardware
// conversion on clamped values (checked against the definition for every bf16 value). (crates/fe-fp4/src/format.rs:57-63)
template <bool HI>
__device__ __forceinline__ uint32_t f32x2_to_e4m3(uint32_t old, float a, float b) {
    uint32_t q = (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(__builtin_amdgcn_fmed3f(a, -448.f, 448.f), __builtin_amdgcn_fmed3f(b, -448.f, 448.f), (int)old, HI);
    constexpr uint32_t S = HI ? 16 : 0;
    if (a != a) q = (q & ~(0xffu << S)) | (0x7fu << S);
    if (b != b) q = (q & ~(0xff00u << S)) | (0x7f00u << S);
    return q;
}

// bf16 x[M][ldx] -> e4m3 codes [M][K], q = e4m3(x * g). One thread per 16 elements: grid ceil(M * K / 16 / 256), 256 threads. K % 16
// == 0, rows 16-byte aligned. Bound by its 3 bytes an element. (kernels/k-fp4/src/lib.rs:199-214)
extern "C" __global__ __launch_bounds__(256) void fe_fp8_quant(uint8_t* codes, const uint16_t* x, uint32_t m, uint32_t k, uint32_t ldx, float g) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x, k16 = k >> 4;
    if (i >= m * k16) return;
    const uint32_t row = i / k16, c = (i - row * k16) * 16;
    const u32x4* p = (const u32x4*)(x + (size_t)row * ldx + c);
    const u32x4 r[2] = {p[0], p[1]};
    u32x4 q;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const uint32_t lo = r[j >> 1][2 * (j & 1)], hi = r[j >> 1][2 * (j & 1) + 1];
        const uint32_t t = f32x2_to_e4m3<false>(0, __uint_as_float(lo << 16) * g, __uint_as_float(lo & 0xffff0000u) * g);
        q[j] = f32x2_to_e4m3<true>(t, __uint_as_float(hi << 16) * g, __uint_as_float(hi & 0xffff0000u) * g);
    }
    *(u32x4*)(codes + (size_t)row * k + c) = q;
}

// e4m3 codes -> the fp16 operand of the fp16 form of the FP8 GEMM (an e4m3 value is an exact fp16 number). One thread per 8 of
// `count` elements.
extern "C" __global__ __launch_bounds__(256) void fe_fp8_expand(_Float16* aq, const uint8_t* codes, uint32_t count) {
    const uint32_t i = (blockIdx.x * 256 + threadIdx.x) * 8;
    if (i >= count) return;
    const u32x2 q = *(const u32x2*)(codes + i);
    u32x4 o;
#pragma unroll
    for (int j = 0; j < 4; j++) o[j] = e4m3x2_to_f16(q[j >> 1], j & 1);
    *(u32x4*)(aq + i) = o;
}

// Weight operand of the fp16 form of the FP8 GEMM: e4m3 codes, [BN rows][64 bytes] in LDS, expanded with the hardware
// conversion (exact). Addressing as Fp4Packed.
template <class T>
struct Fp8Packed {
    static constexpr bool kPerm = true;
    static constexpr int STAGE = T::BN * 64, LOADS = T::BN / 128;
    u32x4 rw;
    uint32_t wv[LOADS], w_skt;
    struct Raw {
        u32x4 c;
    };
    __device__ __forceinline__ void setup(const uint8_t* w, uint32_t n, uint32_t k, uint32_t n0, uint32_t w_snt, uint32_t w_skt_, uint32_t w_sr) {
        const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nts = n / 128;
        rw = g8_rsrc(w, n * k);
#pragma unroll
        for (int j = 0; j < LOADS; j++) {
            const uint32_t row = (wave + 8 * j) * 16 + lane / 4;
            uint32_t nt = (n0 + row) / 128;
            nt = nt < nts ? nt : nts - 1;
            wv[j] = nt * w_snt + (row & 127) * w_sr + (lane & 3) * 16;
        }
        w_skt = w_skt_;
    }
    __device__ __forceinline__ void issue(uint32_t kt, uint32_t dst, int j, uint32_t wave) const {
        g8_load_lds16(rw, dst + (wave + 8 * j) * 1024, wv[j], kt * w_skt);
    }
    __device__ __forceinline__ Raw read(const unsigned char* st, uint32_t row, uint32_t g) const {
        return Raw{*(const u32x4*)(st + row * 64 + 16 * g)};
    }
    __device__ __forceinline__ f16x8 expand(const Raw& r, int kk) const {
        u32x4 o;
#pragma unroll
        for (int e = 0; e < 4; e++) o[e] = e4m3x2_to_f16(r.c[2 * kk + (e >> 1)], e & 1);
        return __builtin_bit_cast(f16x8, o);
    }
};

// ---- fused gate|up epilogue: SwiGLU and NVFP4 re-quantization ---------------------------------------------------------------

// act = bf16(bf16(silu(g)) * u), g and u the bf16 GEMM outputs (kernels/k-fp4/src/lib.rs:669-673).
__device__ __forceinline__ float swiglu(float g, float u) {
    float s = g * __builtin_amdgcn_rcpf(1.0f + __expf(-g));
    s = bf16_bits_to_f32(f32_to_bf16_bits(s));
    return bf16_bits_to_f32(f32_to_bf16_bits(s * u));
}

template <int CTRL>
__device__ __forceinline__ uint32_t dpp_mov_u32(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, CTRL, 0xf, 0xf, true);
}

// The weight rows of a fused gate|up linear are interleaved in blocks of 8 (gate f..f+7, up f..f+7, ...,
// crates/fe-fp4/src/lib.rs:386-417), so a group of 32 output columns holds 16 features: of the 8 lanes that hold it
// (4 columns each) lanes 0, 1 have gate f0..7, lanes 2, 3 up f0..7, lanes 4, 5 gate f8..15, lanes 6, 7 up f8..15. Takes
// the 4 sums of a lane (v, already times alpha's lane values `al`), forms act = SwiGLU(bf16 gate, bf16 up) on the gate
// lanes, quantizes each 16-feature block to NVFP4 with global scale qg exactly as fe_fp4_quant would quantize the bf16
// act (block scale from the block's amax, codes, tiled scale, fp16 operand), and stores for rows that exist. Every lane
// of the half wavefront must call it. col: the lane's first interleaved column; n: interleaved width (2 * inter).
// (kernels/k-fp4/src/lib.rs:675-745)
__device__ __forceinline__ void swiglu_quant_store(const float (&v)[4], f32x4 al, uint32_t l32, bool live, uint32_t row,
                                                   uint32_t col, uint32_t n, uint8_t* q_codes, uint8_t* q_sf, _Float16* q_aq,
                                                   float qg) {
    const uint32_t j = l32 & 7;
    const bool gate = (j & 2) == 0;
    float act[4], amax = 0.f;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        float y = bf16_bits_to_f32(f32_to_bf16_bits(v[e] * al[e]));
        float u = dpp_mov<DPP_QUAD_XOR2>(y);  // the up value of the same feature, two lanes on
        act[e] = swiglu(y, u);
        if (gate) amax = __builtin_fmaxf(amax, __builtin_fabsf(act[e]));
    }
    amax = __builtin_fmaxf(amax, dpp_mov<DPP_QUAD_XOR1>(amax));
    amax = __builtin_fmaxf(amax, dpp_mov<DPP_QUAD_XOR2>(amax));
    amax = __builtin_fmaxf(amax, dpp_mov<DPP_QUAD_XOR3>(dpp_mov<DPP_HALF_MIRROR>(amax)));  // lane ^ 4
    const uint32_t s8 = f32_to_e4m3_pos(amax * (1.0f / 6.0f) * qg);
    const float sv = e4m3_to_f32(s8);
    const float mul = sv > 0.f ? qg / sv : 0.f;
    uint32_t q = f32x2_to_e2m1_byte<0>(0u, act[0] * mul, act[1] * mul);
    q = f32x2_to_e2m1_byte<1>(q, act[2] * mul, act[3] * mul);
    const uint32_t word = q | (dpp_mov_u32<DPP_QUAD_XOR1>(q) << 16);  // 8 codes: this lane's 4 features and the next lane's
    if (!live || !gate) return;
    const uint32_t inter = n >> 1, kb = inter >> 4, blk = col >> 5;
    const uint32_t feat = blk * 16 + (j >> 2) * 8 + (j & 1) * 4;  // the lane's first feature
    uint32_t t[4];
    e2m1x8_to_f16(q, t);
    const f16x2 sc = e4m3_to_f16x2(s8);
    u32x2 o = {__builtin_bit_cast(uint32_t, (f16x2)(__builtin_bit_cast(f16x2, t[0]) * sc)),
               __builtin_bit_cast(uint32_t, (f16x2)(__builtin_bit_cast(f16x2, t[1]) * sc))};
    *(u32x2*)(q_aq + (size_t)row * inter + feat) = o;
    if ((j & 1) == 0) *(uint32_t*)(q_codes + (size_t)row * (inter >> 1) + (feat >> 1)) = word;
    if (j == 0) q_sf[sf_tiled(row, blk, kb)] = (uint8_t)s8;
}

// The same for a finished tile of the GEMM, without LDS and with every lane at work (through the slab the lanes with up sums computed what they did
// not store): the gate sums of a column tile lie in the wavefront's lower half and the up sums in its upper half, so the two tiles of a 16-feature
// block trade halves, after which lane group fc has gate and up of the block's features 4 fc .. + 3; the block's maximum comes from the lanes 16 and
// 32 away; and two blocks trade rows of 16 lanes, so that a lane stores 8 features of one
// (a tile with one block a wavefront: 4). rows: those that exist from row0 on.
// Bound by its vector instructions, which no matrix instruction hides (a program has its CU alone): about 10 us a program through the slab, half of
// that now. Launch, us: 2048 rows of 34816 x 5120 558 -> 535, 390 rows 144 -> 132; MLP blocks of 2048 / 5 + 390 rows 865 -> 816, 279 -> 269.
template <class T>
__device__ __forceinline__ void fp4_tile_swiglu(f32x4 (&acc)[T::TM][T::TN], const float* alpha, float scale, uint32_t row0, uint32_t rows, uint32_t colb, uint32_t n, uint8_t* q_codes,
                                                uint8_t* q_sf, _Float16* q_aq, float qg) {
    constexpr int TN = T::TN, STEP = TN % 4 == 0 ? 4 : 2;  // column tiles that are stored together
    const uint32_t lane = threadIdx.x & 63, fr = lane & 15, fc = lane >> 4, inter = n >> 1, kb = inter >> 4;
    f32x4 al[TN];
#pragma unroll
    for (int j = 0; j < TN; j++) al[j] = *(const f32x4*)(alpha + colb + 16 * j + 4 * fc) * scale;
    struct Part {
        uint32_t q, s8, o0, o1;  // 4 codes, the block's scale, the 4 values as the GEMM's operand
    };
    auto block = [&](f32x4 a, f32x4 b, f32x4 ala, f32x4 alb) {
        a *= ala, b *= alb;
        uint32_t g[2] = {pack_bf16x2(a[0], a[1]), pack_bf16x2(a[2], a[3])}, u[2] = {pack_bf16x2(b[0], b[1]), pack_bf16x2(b[2], b[3])};
        g8_swap32(g[0], u[0]), g8_swap32(g[1], u[1]);
        float act[4], amax = 0.f;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const uint32_t gw = g[e >> 1], uw = u[e >> 1];
            act[e] = swiglu(__uint_as_float(e & 1 ? gw & 0xffff0000u : gw << 16), __uint_as_float(e & 1 ? uw & 0xffff0000u : uw << 16));
            amax = __builtin_fmaxf(amax, __builtin_fabsf(act[e]));
        }
        uint32_t x = __float_as_uint(amax), y = x;
        g8_swap16(x, y);
        x = y = __float_as_uint(__builtin_fmaxf(__uint_as_float(x), __uint_as_float(y)));
        g8_swap32(x, y);
        amax = __builtin_fmaxf(__uint_as_float(x), __uint_as_float(y));
        Part r;
        r.s8 = f32_to_e4m3_pos(amax * (1.0f / 6.0f) * qg);
        const float sv = e4m3_to_f32(r.s8);
        const float mul = sv > 0.f ? qg / sv : 0.f;
        r.q = f32x2_to_e2m1_byte<0>(0u, act[0] * mul, act[1] * mul);
        r.q = f32x2_to_e2m1_byte<1>(r.q, act[2] * mul, act[3] * mul);
        uint32_t t[4];
        e2m1x8_to_f16(r.q, t);
        const f16x2 sc = e4m3_to_f16x2(r.s8);
        r.o0 = __builtin_bit_cast(uint32_t, (f16x2)(__builtin_bit_cast(f16x2, t[0]) * sc));
        r.o1 = __builtin_bit_cast(uint32_t, (f16x2)(__builtin_bit_cast(f16x2, t[1]) * sc));
        return r;
    };
#pragma unroll
    for (int i = 0; i < T::TM; i++) {
        if (16 * i >= rows) break;
        const uint32_t row = row0 + 16 * i + fr;
#pragma unroll
        for (int j = 0; j < TN; j += STEP) {
            Part x = block(acc[i][j], acc[i][j + 1], al[j], al[j + 1]);
            const uint32_t blk = (colb >> 5) + j / 2;
            if constexpr (STEP == 4) {
                Part y = block(acc[i][j + 2], acc[i][j + 3], al[j + 2], al[j + 3]);
                g8_swap16(x.o0, y.o0), g8_swap16(x.o1, y.o1), g8_swap16(x.q, y.q);
                // lane groups 0, 2 store block blk's features 0..7, 8..15, groups 1, 3 the next block's
                const uint32_t my = blk + (fc & 1), half = fc >> 1;
                if (16 * i + fr < rows) {
                    *(u32x4*)(q_aq + (size_t)row * inter + my * 16 + 8 * half) = (u32x4){x.o0, x.o1, y.o0, y.o1};
                    *(uint32_t*)(q_codes + (size_t)row * (inter >> 1) + my * 8 + 4 * half) = (x.q & 0xffff) | (y.q << 16);
                    if (fc < 2) q_sf[sf_tiled(row, my, kb)] = (uint8_t)(fc ? y.s8 : x.s8);
                }
            } else if (16 * i + fr < rows) {
                *(u32x2*)(q_aq + (size_t)row * inter + blk * 16 + 4 * fc) = (u32x2){x.o0, x.o1};
                *(uint16_t*)(q_codes + (size_t)row * (inter >> 1) + blk * 8 + 2 * fc) = (uint16_t)x.q;
                if (fc == 0) q_sf[sf_tiled(row, blk, kb)] = (uint8_t)x.s8;
            }
        }
    }
}

// ---- GEMM kernels ------------------------------------------------------------------------------------------------------------

// Where the output of a GEMM goes: C (bf16, + residual) or, for a fused gate|up linear, the NVFP4-quantized SwiGLU.
struct FpOut {
    uint16_t* c;
    const uint16_t* res;
    uint32_t ldc;
    uint8_t* q_codes;
    uint8_t* q_sf;
    _Float16* q_aq;
    float qg;
};

// The wavefront's rows of a finished tile, from row0, colb (inside n) on: sums times alpha * scale. (The stream-K forms add a residual through the
// slab: g8_add_bf16's registers, beside what their loop over segments keeps, would cost 30 spilled ones.)
template <class T, bool SWIGLU, bool SK>
__device__ __forceinline__ void fp_tile_store(f32x4 (&acc)[T::TM][T::TN], unsigned char* lds, const FpOut& o, const float* alpha, float scale, uint32_t m, uint32_t n,
                                              uint32_t row0, uint32_t colb) {
    if constexpr (SWIGLU) {
        if (row0 < m) fp4_tile_swiglu<T>(acc, alpha, scale, row0, m - row0, colb, n, o.q_codes, o.q_sf, o.q_aq, o.qg);
        return;
    }
    const uint32_t lane = threadIdx.x & 63, col = colb + 4 * (lane % (4 * T::TN));
    if constexpr (!SK) {
        if (o.res) {
            if (row0 >= m) return;
            f32x4 al[T::TN];
#pragma unroll
            for (int j = 0; j < T::TN; j++) al[j] = *(const f32x4*)(alpha + colb + 16 * j + 4 * (lane >> 4)) * scale;
            const size_t first = (size_t)row0 * o.ldc + colb;
            g8_add_bf16<T>(acc, o.c + first, o.res + first, o.ldc, m - row0, n - colb, [&](f32x4 v, int j) {
                return (u32x2){pack_bf16x2(v[0] * al[j][0], v[1] * al[j][1]), pack_bf16x2(v[2] * al[j][2], v[3] * al[j][3])};
            });
            return;
        }
    }
    const f32x4 al = *(const f32x4*)(alpha + col) * scale;
    auto rows = [&](auto adds_tag) {
        constexpr bool ADDS = decltype(adds_tag)::value;
        g8_epilogue<T>(
            acc, lds, [](auto&, uint32_t) {},
            [&](uint32_t r, uint32_t) {
                if constexpr (ADDS)
                    return row0 + r < m ? *(const u32x2*)(o.res + (size_t)(row0 + r) * o.ldc + col) : (u32x2){0, 0};
                else
                    return G8Nothing{};
            },
            [&](uint32_t r, uint32_t, float (&v)[4], auto old) {
                const uint32_t row = row0 + r;
                if (row >= m) return;
                if constexpr (ADDS)
                    fp4_store4(o.c, true, old, (size_t)row * o.ldc + col, v, al);
                else
                    fp4_store4(o.c, false, (u32x2){0, 0}, (size_t)row * o.ldc + col, v, al);
            });
    };
    if (SK && o.res)
        rows(std::bool_constant<SK>{});
    else
        rows(std::false_type{});
}

// Tiles of 256 x 256, 128 x 256 (S1), 128 x 128 (S2) and 224, 192, 160 x 256 (H7, H6, H5). Packed weights: a wavefront's columns are a quarter of the
// tile's, so that a weight is expanded by two wavefronts only. The GEMM over FP8 codes expands nothing.
typedef G8Tile<2, 4, 8, 4> FpTile;
typedef G8Tile<2, 4, 4, 4> FpTileS1;
typedef G8Tile<2, 4, 4, 2> FpTileS2;
typedef G8Tile<2, 4, 7, 4> FpTileH7;
typedef G8Tile<2, 4, 6, 4> FpTileH6;
typedef G8Tile<2, 4, 5, 4> FpTileH5;
typedef G8Tile<4, 2, 4, 8> Fp8Tile;
typedef G8Tile<4, 2, 2, 8> Fp8TileS1;
typedef G8Tile<4, 2, 2, 4> Fp8TileS2;
// wavefronts a SIMD: two programs of the smallest tile fit a CU; k tiles of A and of packed weights in LDS
template <class T>
struct FpWaves {
    static constexpr int MIN = T::PARTS == 4 ? 4 : 2, NA = T::PARTS == 2 ? 5 : 3, NW = T::PARTS == 2 ? 6 : T::PARTS == 4 ? 4 : 3;
};

// C[M][ldc] = bf16((A_q . W_q^T) * alpha[n]) (+ res: bf16(bf16(.) + res)); A_q = the fp16 operand of the quantizer,
// W_q expanded by the packed operand make_packed(n0) of the tile at column n0; `scale` = 1 / (the factors the two fp16 operands
// carry). Tiles (grouped raster) spread over the grid as sc says (g8_schedule). 512 threads, dynamic LDS as the stages take.
// N % 128 == 0, K % 128 == 0. (kernels/k-fp4/src/lib.rs:285-470)
template <class T, bool SWIGLU, bool SK, class MakePacked>
__device__ __forceinline__ void fp_gemm_body(MakePacked make_packed, const FpOut& out, const _Float16* aq, const float* alpha,
                                             float scale, uint32_t m, uint32_t n, uint32_t k, uint32_t group_m,
                                             const GemmSched& sc) {
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wm = wave / T::WN, wn = wave % T::WN;
    g8_schedule<T, SK>(
        sc, m, n, group_m, k / G8_BK, lds,
        [&](uint32_t m0, uint32_t n0, uint32_t kt0, uint32_t ktn, f32x4(&acc)[T::TM][T::TN]) {
            auto w = make_packed(n0);
            g8_mainloop_packed<T, FpWaves<T>::NA, FpWaves<T>::NW, !SK>(aq, k, m, kt0, ktn, m0, w, lds, acc);
        },
        [&](uint32_t m0, uint32_t n0, f32x4(&acc)[T::TM][T::TN]) {
            const uint32_t row0 = m0 + wm * 16 * T::TM, colb = n0 + wn * 16 * T::TN;
            if (colb >= n) return;
            fp_tile_store<T, SWIGLU, SK>(acc, lds, out, alpha, scale, m, n, row0, colb);
        });
}

// Finishes the tiles that a GEMM kernel cut along K. Grid and threads: g8_reduce_rows.
template <class T, bool SWIGLU>
__device__ __forceinline__ void fp_reduce_body(const FpOut& out, const float* part, const float* alpha, float scale,
                                               uint32_t m, uint32_t n, uint32_t group_m, uint32_t first, uint32_t splits) {
    struct Ahead {
        f32x4 al;
        u32x2 old;
    };
    g8_reduce_rows<T>(
        part, m, n, group_m, first, splits,
        [&](uint32_t row, uint32_t n0, uint32_t l32) {
            const uint32_t col = n0 + 4 * l32;
            Ahead a = {*(const f32x4*)(alpha + col) * scale, {0, 0}};
            if (!SWIGLU && out.res && row < m) a.old = *(const u32x2*)(out.res + (size_t)row * out.ldc + col);
            return a;
        },
        [&](uint32_t row, uint32_t n0, uint32_t l32, float (&v)[4], const Ahead& a) {
            const uint32_t col = n0 + 4 * l32;
            if constexpr (SWIGLU)
                swiglu_quant_store(v, a.al, l32, row < m, row < m ? row : 0, col, n, out.q_codes, out.q_sf, out.q_aq, out.qg);
            else if (row < m)
                fp4_store4(out.c, out.res != nullptr, a.old, (size_t)row * out.ldc + col, v, a.al);
        });
}

// NVFP4: the codes of row r = 128 nt + i, k tile kt are 32 bytes at w + nt * w_snt + kt * w_skt + i * w_sr, its 4 scales
// at sw + nt * s_snt + kt * s_skt + i * s_sr.
// Every GEMM kernel comes in two forms, NAME (one piece a program) and NAME_sk (stream-K), with the same parameters.
#define FP4_GEMM_PARAMS                                                                                                    \
    uint16_t *c, const _Float16 *aq, const uint8_t *w, const uint8_t *sw, const float *alpha, const uint16_t *res, uint32_t m, \
        uint32_t n, uint32_t k, uint32_t ldc, uint32_t group_m, uint32_t w_snt, uint32_t w_skt, uint32_t w_sr, uint32_t s_snt, \
        uint32_t s_skt, uint32_t s_sr, GemmSched sc
template <class T, bool SK>
__device__ __forceinline__ void gemm_nvfp4_kernel(FP4_GEMM_PARAMS) {
    asm volatile("" ::"s"(c), "s"(aq), "s"(w), "s"(sw), "s"(alpha), "s"(res), "s"(m), "s"(n), "s"(k), "s"(ldc), "s"(group_m), "s"(w_snt), "s"(w_skt), "s"(w_sr),
                 "s"(s_snt), "s"(s_skt), "s"(s_sr), GEMM_SCHED_WORDS(sc));
    FpOut out = {c, res, ldc, nullptr, nullptr, nullptr, 0.f};
    fp_gemm_body<T, false, SK>(
        [&](uint32_t n0) {
            Fp4Packed<T> p;
            p.setup(w, sw, n, k, n0, w_snt, w_skt, w_sr, s_snt, s_skt, s_sr);
            return p;
        },
        out, aq, alpha, FP4_GEMM_SCALE, m, n, k, group_m, sc);
}
#define FP4_GEMM_KERNEL(SUFFIX, TILE, SK)                                                                                  \
    extern "C" __global__ __launch_bounds__(512, FpWaves<TILE>::MIN) void fe_gemm_nvfp4##SUFFIX(FP4_GEMM_PARAMS) {         \
        gemm_nvfp4_kernel<TILE, SK>(c, aq, w, sw, alpha, res, m, n, k, ldc, group_m, w_snt, w_skt, w_sr, s_snt, s_skt, s_sr, sc); \
    }
FP4_GEMM_KERNEL(, FpTile, false)
FP4_GEMM_KERNEL(_sk, FpTile, true)
FP4_GEMM_KERNEL(_s1, FpTileS1, false)
FP4_GEMM_KERNEL(_s2, FpTileS2, false)
FP4_GEMM_KERNEL(_h7, FpTileH7, false)
FP4_GEMM_KERNEL(_h6, FpTileH6, false)
FP4_GEMM_KERNEL(_h5, FpTileH5, false)

#define FP_REDUCE_KERNEL(NAME, TILE)                                                                                       \
    extern "C" __global__ __launch_bounds__(512) void NAME(uint16_t* c, const float* part, const float* alpha,             \
                                                           const uint16_t* res, uint32_t m, uint32_t n, uint32_t ldc,      \
                                                           uint32_t group_m, uint32_t first, uint32_t splits, float scale) { \
        FpOut out = {c, res, ldc, nullptr, nullptr, nullptr, 0.f};                                                         \
        fp_reduce_body<TILE, false>(out, part, alpha, scale, m, n, group_m, first, splits);                                \
    }
FP_REDUCE_KERNEL(fe_gemm_nvfp4_reduce, FpTile)
FP_REDUCE_KERNEL(fe_gemm_nvfp4_reduce_s1, FpTileS1)
FP_REDUCE_KERNEL(fe_gemm_nvfp4_reduce_s2, FpTileS2)
FP_REDUCE_KERNEL(fe_gemm_nvfp4_reduce_h7, FpTileH7)
FP_REDUCE_KERNEL(fe_gemm_nvfp4_reduce_h6, FpTileH6)
FP_REDUCE_KERNEL(fe_gemm_nvfp4_reduce_h5, FpTileH5)
FP_REDUCE_KERNEL(fe_gemm_fp8_codes_reduce, Fp8Tile)
FP_REDUCE_KERNEL(fe_gemm_fp8_codes_reduce_s1, Fp8TileS1)
FP_REDUCE_KERNEL(fe_gemm_fp8_codes_reduce_s2, Fp8TileS2)

// Fused MLP front: act = SwiGLU(x . [gate|up]^T), NVFP4-quantized with global scale qg (1 / input_scale of the down
// projection) into q_codes [M][inter/2], q_sf (tiled, kb = inter/16) and the fp16 operand q_aq [M][inter]; w, sw, alpha =
// gate and up interleaved in blocks of 8 rows, N = 2 inter, N % 256 == 0. (kernels/k-fp4/src/lib.rs:747-752)
#define FP4_SWIGLU_PARAMS                                                                                                \
    const _Float16 *aq, const uint8_t *w, const uint8_t *sw, const float *alpha, uint32_t m, uint32_t n, uint32_t k,           \
        uint32_t group_m, uint32_t w_snt, uint32_t w_skt, uint32_t w_sr, uint32_t s_snt, uint32_t s_skt, uint32_t s_sr,        \
        GemmSched sc, uint8_t *q_codes, uint8_t *q_sf, _Float16 *q_aq, float qg
template <class T, bool SK>
__device__ __forceinline__ void gemm_nvfp4_swiglu_kernel(FP4_SWIGLU_PARAMS) {
    asm volatile("" ::"s"(aq), "s"(w), "s"(sw), "s"(alpha), "s"(m), "s"(n), "s"(k), "s"(group_m), "s"(w_snt), "s"(w_skt), "s"(w_sr), "s"(s_snt), "s"(s_skt),
                 "s"(s_sr), GEMM_SCHED_WORDS(sc), "s"(q_codes), "s"(q_sf), "s"(q_aq), "s"(qg));
    FpOut out = {nullptr, nullptr, 0, q_codes, q_sf, q_aq, qg};
    fp_gemm_body<T, true, SK>(
        [&](uint32_t n0) {
            Fp4Packed<T> p;
            p.setup(w, sw, n, k, n0, w_snt, w_skt, w_sr, s_snt, s_skt, s_sr);
            return p;
        },
        out, aq, alpha, FP4_GEMM_SCALE, m, n, k, group_m, sc);
}
#define FP4_SWIGLU_KERNEL(SUFFIX, TILE, SK)                                                                                \
    extern "C" __global__ __launch_bounds__(512, FpWaves<TILE>::MIN) void fe_gemm_nvfp4_swiglu##SUFFIX(FP4_SWIGLU_PARAMS) { \
        gemm_nvfp4_swiglu_kernel<TILE, SK>(aq, w, sw, alpha, m, n, k, group_m, w_snt, w_skt, w_sr, s_snt, s_skt, s_sr, sc, q_codes, \
                                           q_sf, q_aq, qg);                                                                \
    }
FP4_SWIGLU_KERNEL(, FpTile, false)
FP4_SWIGLU_KERNEL(_sk, FpTile, true)
FP4_SWIGLU_KERNEL(_s1, FpTileS1, false)
FP4_SWIGLU_KERNEL(_s2, FpTileS2, false)
FP4_SWIGLU_KERNEL(_h7, FpTileH7, false)
FP4_SWIGLU_KERNEL(_h6, FpTileH6, false)
FP4_SWIGLU_KERNEL(_h5, FpTileH5, false)
#define FP4_SWIGLU_REDUCE_KERNEL(SUFFIX, TILE)                                                                             \
    extern "C" __global__ __launch_bounds__(512) void fe_gemm_nvfp4_swiglu_reduce##SUFFIX(                                 \
        const float* part, const float* alpha, uint32_t m, uint32_t n, uint32_t group_m, uint32_t first, uint32_t splits,  \
        uint8_t* q_codes, uint8_t* q_sf, _Float16* q_aq, float qg) {                                                       \
        FpOut out = {nullptr, nullptr, 0, q_codes, q_sf, q_aq, qg};                                                        \
        fp_reduce_body<TILE, true>(out, part, alpha, FP4_GEMM_SCALE, m, n, group_m, first, splits);                        \
    }
FP4_SWIGLU_REDUCE_KERNEL(, FpTile)
FP4_SWIGLU_REDUCE_KERNEL(_s1, FpTileS1)
FP4_SWIGLU_REDUCE_KERNEL(_s2, FpTileS2)
FP4_SWIGLU_REDUCE_KERNEL(_h7, FpTileH7)
FP4_SWIGLU_REDUCE_KERNEL(_h6, FpTileH6)
FP4_SWIGLU_REDUCE_KERNEL(_h5, FpTileH5)

// FP8: the 64 codes of row r = 128 nt + i, k tile kt are at w + nt * w_snt + kt * w_skt + i * w_sr; both fp16 expansions
// are the values themselves. Finished by fe_gemm_nvfp4_reduce with scale 1. (kernels/k-fp4/src/lib.rs:472-484)
#define FP8_GEMM_PARAMS                                                                                                     \
    uint16_t *c, const _Float16 *aq, const uint8_t *w, const float *alpha, const uint16_t *res, uint32_t m, uint32_t n, uint32_t k, \
        uint32_t ldc, uint32_t group_m, uint32_t w_snt, uint32_t w_skt, uint32_t w_sr, GemmSched sc
template <bool SK>
__device__ __forceinline__ void gemm_fp8_kernel(FP8_GEMM_PARAMS) {
    FpOut out = {c, res, ldc, nullptr, nullptr, nullptr, 0.f};
    fp_gemm_body<FpTile, false, SK>(
        [&](uint32_t n0) {
            Fp8Packed<FpTile> p;
            p.setup(w, n, k, n0, w_snt, w_skt, w_sr);
            return p;
        },
        out, aq, alpha, 1.0f, m, n, k, group_m, sc);
}
extern "C" __global__ __launch_bounds__(512, 2) void fe_gemm_fp8(FP8_GEMM_PARAMS) {
    gemm_fp8_kernel<false>(c, aq, w, alpha, res, m, n, k, ldc, group_m, w_snt, w_skt, w_sr, sc);
}
extern "C" __global__ __launch_bounds__(512, 2) void fe_gemm_fp8_sk(FP8_GEMM_PARAMS) {
    gemm_fp8_kernel<true>(c, aq, w, alpha, res, m, n, k, ldc, group_m, w_snt, w_skt, w_sr, sc);
}

// The same linear on the 8-bit matrix instruction: activations are the quantizer's e4m3 codes [M][K], weights stay codes
// in LDS, a k tile is 128 wide (two of the 64-wide weight tiles of the layout above). Same products (an e4m3 x e4m3
// product is exact in f32) and f32 sums as fe_gemm_fp8, at twice the MFMA rate and half the LDS bytes per flop.
#define FP8C_GEMM_PARAMS                                                                                                   \
    uint16_t *c, const uint8_t *aq, const uint8_t *w, const float *alpha, const uint16_t *res, uint32_t m, uint32_t n, uint32_t k, \
        uint32_t ldc, uint32_t group_m, uint32_t w_snt, uint32_t w_skt, uint32_t w_sr, GemmSched sc
template <class T, bool SK>
__device__ __forceinline__ void gemm_fp8_codes_kernel(FP8C_GEMM_PARAMS) {
    constexpr int NA = T::PARTS == 2 ? 3 : 2;
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
    const uint32_t nts = n / 128, lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wm = wave / T::WN, wn = wave % T::WN;
    FpOut out = {c, res, ldc, nullptr, nullptr, nullptr, 0.f};
    g8_schedule<T, SK>(
        sc, m, n, group_m, k / 128, lds,
        [&](uint32_t m0, uint32_t n0, uint32_t kt0, uint32_t ktn, f32x4(&acc)[T::TM][T::TN]) {
            // a k tile of 128 codes is two of the layout's 64-wide ones: chunks 0..3 of a row from the first, 4..7 from the second
            G8Dense<T> wo;
            wo.rs = g8_rsrc(w, n * k), wo.kstep = 2 * w_skt;
#pragma unroll
            for (int j = 0; j < G8Dense<T>::LOADS; j++) {
                const uint32_t r = 8 * (wave + 8 * j) + (lane >> 3), ch = (lane & 7) ^ (r & 7);
                uint32_t nt = (n0 + r) / 128;
                nt = nt < nts ? nt : nts - 1;  // an odd count of 128-row tiles: the last program reads its first tile twice
                wo.voff[j] = nt * w_snt + (ch >> 2) * w_skt + (r & 127) * w_sr + (ch & 3) * 16;
            }
            g8_mainloop_f8<T, NA, 3, !SK>(aq, k, m, kt0, ktn, m0, wo, lds, acc);
        },
        [&](uint32_t m0, uint32_t n0, f32x4(&acc)[T::TM][T::TN]) {
            const uint32_t row0 = m0 + wm * 16 * T::TM, colb = n0 + wn * 16 * T::TN;
            if (colb >= n) return;
            fp_tile_store<T, false, SK>(acc, lds, out, alpha, 1.0f, m, n, row0, colb);
        });
}
#define FP8C_GEMM_KERNEL(SUFFIX, TILE, SK)                                                                                 \
    extern "C" __global__ __launch_bounds__(512, FpWaves<TILE>::MIN) void fe_gemm_fp8_codes##SUFFIX(FP8C_GEMM_PARAMS) {    \
        gemm_fp8_codes_kernel<TILE, SK>(c, aq, w, alpha, res, m, n, k, ldc, group_m, w_snt, w_skt, w_sr, sc);              \
    }
FP8C_GEMM_KERNEL(, Fp8Tile, false)
FP8C_GEMM_KERNEL(_sk, Fp8Tile, true)
FP8C_GEMM_KERNEL(_s1, Fp8TileS1, false)
FP8C_GEMM_KERNEL(_s2, Fp8TileS2, false)
FP8C_GEMM_KERNEL(_h7, FpTileH7, false)
FP8C_GEMM_KERNEL(_h6, FpTileH6, false)
FP8C_GEMM_KERNEL(_h5, FpTileH5, false)

// ---- FP8 GEMV (few rows): the weights read once, no hand-off -----------------------------------------------------------
//
// c[m][ldc] = bf16((codes . W^T) * alpha[n]) (+ res) for m <= 8 XO rows of e4m3 codes [m][k], weights as in fe_gemm_fp8_codes. grid ceil(N / pc), 256
// threads: a program takes pc <= 8 CO weight rows (gemv_even) over all of K, its four wavefronts a quarter of K's steps of 128 codes each, DEPTH - 1
// steps ahead in LDS stages of their own; a load is 8 rows x 128 bytes, a row's 16-byte chunk c at position c ^ (row & 7). A wavefront adds its
// products in ascending k, the four sums are added in order: a row's bits depend on K and W only. Bound by the weights' way from HBM up to 16 rows,
// by the activations' way from L2 as rows and K grow. It replaces the GEMM, whose tiles of 128 rows are mostly empty and whose pieces of K need a
// reduce launch: kFeGemvFp8 of fe_internal.h has both sides.
template <int XO, int CO>
struct Fp8Gemv {
    static constexpr int L = CO + XO, STAGE = L * 1024;
    static constexpr int FIT = 20 * 1024 / STAGE, DEPTH = FIT < 3 ? 3 : FIT < 8 ? FIT : 8;  // two programs a CU where three steps allow it
    static_assert((DEPTH - 1) * L < 64 && 4 * DEPTH * STAGE <= 160 * 1024, "stages");
};

template <int XO, int CO>
__device__ __forceinline__ void gemv_fp8_body(uint16_t* c, const uint8_t* x, const uint8_t* w, const float* alpha, const uint16_t* res, uint32_t m, uint32_t n, uint32_t k,
                                              uint32_t ldc, uint32_t w_snt, uint32_t w_skt, uint32_t w_sr, uint32_t pc) {
    typedef Fp8Gemv<XO, CO> C;
    constexpr int RG = (XO + 1) / 2, CG = (CO + 1) / 2, AHEAD = C::DEPTH - 1, PITCH = 16 * CG + 4;
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r = lane & 15, g = lane >> 4;
    const uint32_t col0 = blockIdx.x * pc, cols = n - col0 < pc ? n - col0 : pc, nt0 = col0 / 128, span = n / 128 - nt0 < 2 ? n / 128 - nt0 : 2;
    const u32x4 wrs = g8_rsrc(w + (size_t)nt0 * w_snt, span * 128 * k), xrs = g8_rsrc(x, m * k);
    // (columns and rows that do not exist repeat the last one; a step is two of the layout's k tiles: chunks 0..3 of a row from the first, 4..7 from
    // the second)
    const uint32_t lr = lane >> 3, ch = (lane & 7) ^ lr;
    uint32_t vw[CO], vx[XO];
#pragma unroll
    for (int j = 0; j < CO; j++) {
        const uint32_t i = col0 + (8 * j + lr < cols ? 8 * j + lr : cols - 1) - 128 * nt0;
        vw[j] = (i >> 7) * w_snt + (ch >> 2) * w_skt + (i & 127) * w_sr + (ch & 3) * 16;
    }
#pragma unroll
    for (int j = 0; j < XO; j++) vx[j] = (8 * j + lr < m ? 8 * j + lr : m - 1) * k + ch * 16;
    unsigned char* stages = lds + wave * (C::DEPTH * C::STAGE);
    const uint32_t stages0 = g8_lds_addr(stages);
    const uint32_t steps = k / 128, s0 = wave * steps / 4, count = (wave + 1) * steps / 4 - s0;
    auto issue = [&](uint32_t s, uint32_t slot) {
        const uint32_t at = stages0 + slot * C::STAGE;
#pragma unroll
        for (int j = 0; j < CO; j++) g8_load_lds16_nt(wrs, at + j * 1024, vw[j], (s0 + s) * 2 * w_skt);
#pragma unroll
        for (int j = 0; j < XO; j++) g8_load_lds16(xrs, at + (CO + j) * 1024, vx[j], (s0 + s) * 128);
    };
    uint32_t fw[CG][2], fx[RG][2];
    auto frag = [&](uint32_t row, int h) { return row * 128 + (((4 * h + g) ^ (row & 7)) << 4); };
#pragma unroll
    for (int h = 0; h < 2; h++) {
#pragma unroll
        for (int j = 0; j < CG; j++) fw[j][h] = frag(16 * j + r < 8 * CO ? 16 * j + r : 8 * CO - 1, h);
#pragma unroll
        for (int i = 0; i < RG; i++) fx[i][h] = CO * 1024 + frag(16 * i + r < m ? 16 * i + r : m - 1, h);
    }
    f32x4 acc[RG][CG] = {};
    uint32_t slot = 0;
    auto add = [&]() {
        const unsigned char* st = stages + slot * C::STAGE;
        auto read = [&](const uint32_t (&at)[2]) {
            const u32x4 lo = *(const u32x4*)(st + at[0]), hi = *(const u32x4*)(st + at[1]);
            return (g8_i32x8){(int)lo[0], (int)lo[1], (int)lo[2], (int)lo[3], (int)hi[0], (int)hi[1], (int)hi[2], (int)hi[3]};
        };
        g8_i32x8 wv[CG];
#pragma unroll
        for (int j = 0; j < CG; j++) wv[j] = read(fw[j]);
#pragma unroll
        for (int i = 0; i < RG; i++) {
            const g8_i32x8 xv = read(fx[i]);
#pragma unroll
            for (int j = 0; j < CG; j++) acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wv[j], xv, acc[i][j], 0, 0, 0, 0, 0, 0);
        }
        slot = slot + 1 == C::DEPTH ? 0 : slot + 1;
    };
    if (count) {
#pragma unroll
        for (int u = 0; u < AHEAD; u++) issue((uint32_t)u < count ? u : count - 1, u);  // past the end: the last step again, not added
        uint32_t s = 0;
        for (; s + AHEAD < count; s++) {
            g8_loads_wait<(AHEAD - 1) * C::L>();  // (the stage in front of this one has been read, too)
            issue(s + AHEAD, slot ? slot - 1 : AHEAD);
            add();
        }
        auto tail = [&](auto u_tag) {
            constexpr int U = decltype(u_tag)::value;
            if constexpr (U < AHEAD)
                if (s + U < count) {
                    g8_loads_wait<(AHEAD - 1 - U) * C::L>();
                    add();
                }
        };
        tail(std::integral_constant<int, 0>{});
        tail(std::integral_constant<int, 1>{});
        tail(std::integral_constant<int, 2>{});
        tail(std::integral_constant<int, 3>{});
        tail(std::integral_constant<int, 4>{});
        tail(std::integral_constant<int, 5>{});
        tail(std::integral_constant<int, 6>{});
        g8_loads_wait<0>();
    }
    float(*red)[16][PITCH] = (float(*)[16][PITCH])lds;
#pragma unroll
    for (int i = 0; i < RG; i++) {
        __syncthreads();
#pragma unroll
        for (int j = 0; j < CG; j++) *(f32x4*)&red[wave][r][16 * j + 4 * g] = acc[i][j];
        __syncthreads();
        for (uint32_t e = tid; e < 16 * 2 * CO; e += 256) {
            const uint32_t row = e / (2 * CO), j = 4 * (e % (2 * CO));
            if (16 * i + row >= m || j >= cols) continue;
            const f32x4 sum = ((*(const f32x4*)&red[0][row][j] + *(const f32x4*)&red[1][row][j]) + *(const f32x4*)&red[2][row][j]) + *(const f32x4*)&red[3][row][j];
            const float v[4] = {sum[0], sum[1], sum[2], sum[3]};
            fp4_store4(c, res, (size_t)(16 * i + row) * ldc + col0 + j, v, *(const f32x4*)(alpha + col0 + j));
        }
    }
}

#define FP8_GEMV_KERNEL(XO, CO)                                                                                                                              \
    extern "C" __global__ __launch_bounds__(256) void fe_gemv_fp8_r##XO##_c##CO(uint16_t* c, const uint8_t* x, const uint8_t* w, const float* alpha,          \
        const uint16_t* res, uint32_t m, uint32_t n, uint32_t k, uint32_t ldc, uint32_t w_snt, uint32_t w_skt, uint32_t w_sr, uint32_t pc) {                  \
        gemv_fp8_body<XO, CO>(c, x, w, alpha, res, m, n, k, ldc, w_snt, w_skt, w_sr, pc);                                                                         \
    }
#define FP8_GEMV_ROWS(XO) FP8_GEMV_KERNEL(XO, 1) FP8_GEMV_KERNEL(XO, 2) FP8_GEMV_KERNEL(XO, 3) FP8_GEMV_KERNEL(XO, 4) FP8_GEMV_KERNEL(XO, 5)
FP8_GEMV_ROWS(1) FP8_GEMV_ROWS(2) FP8_GEMV_ROWS(4) FP8_GEMV_ROWS(6) FP8_GEMV_ROWS(8)
FP8_GEMV_KERNEL(1, 6) FP8_GEMV_KERNEL(2, 6) FP8_GEMV_KERNEL(4, 6) FP8_GEMV_KERNEL(6, 6)
FP8_GEMV_KERNEL(1, 9) FP8_GEMV_KERNEL(2, 9) FP8_GEMV_KERNEL(4, 9)

// ---- GEMV (1..48 rows) -------------------------------------------------------------------------------------------------

#define FP4_GEMV_RG 8  // 16-row groups of a 128-row weight tile

// One k tile of one 128-row weight tile as a wavefront reads it: lane L = 16 g + r takes, of row 16 rg + r, the 16 codes
// k = 16 g .. 16 g + 15 (8 bytes) and the row's four scale bytes (it uses byte g), and of activation rows r, 16 + r, ...
// (XR groups of 16) the same 16 values. The k index inside an MFMA is only a summation index, so the A operand (weights)
// and the B operand (activations) merely have to agree: MFMA j of a row group multiplies k = 16 g + 8 j .. + 7 of lane
// group g.
template <int XR>
struct Fp4GemvStage {
    u32x2 cw[FP4_GEMV_RG];
    uint32_t sc[FP4_GEMV_RG];
    f16x8 x[XR][2];
};

// c[m][ldc] = bf16((A_q . W_q^T) * alpha[n]) (+ res) for m <= 16 XR rows: the decode-sized form of fe_gemm_nvfp4, bound
// by the read of the weights, which every row count reads once. grid (n / 128) * sk, 256 threads: a program takes one
// 128-row weight tile and one of sk runs of k tiles, its four wavefronts alternate k tiles. Each wavefront expands its
// codes in registers straight into the A operand of v_mfma_f32_16x16x32_f16 (rows = weight rows, columns = activation
// rows; one expansion serves all XR groups of activation rows); the wavefronts' sums meet in LDS. With sk > 1 the
// splits leave f32 partials in z (per weight tile and split, 8 KB per group of 16 activation rows, in the order the
// lanes hold them); the last to arrive (counters[tile]) adds them in split order, finishes the tile and re-arms the
// counter, so the result does not depend on timing. A row's sums do not depend on XR. Weight
// addressing as in fe_gemm_nvfp4.
// NT: non-temporal loads of the weights. Not of rows as they lie in a checkpoint (_v): a wavefront's piece of such a row is a quarter of its cache
// line, which the next wavefronts then read again from memory: 34816 x 5120 at 32 rows 131 us with, 102 without; 17408 x 5120 51 -> 39. (Weight
// tiles: 41.6 with, 42.2 without.) SWIGLU: a fused gate|up linear, whose finished tile goes through LDS to swiglu_quant_store (out), a row a half
// wavefront. 34816 x 5120 at 17 / 32 / 48 rows 37 / 42 / 51 us against 63 in the GEMM (swiglu_takes_gemv of fe_fp4.cpp).
template <int XR, bool NT, bool SWIGLU>
__device__ __forceinline__ void gemv_nvfp4_body(const FpOut out, const _Float16* aq, const uint8_t* w, const uint8_t* sw,
                                                const float* alpha, float* z, uint32_t* counters,
                                                uint32_t m, uint32_t n, uint32_t k, uint32_t sk,
                                                uint32_t w_snt, uint32_t w_skt, uint32_t w_sr, uint32_t s_snt,
                                                uint32_t s_skt, uint32_t s_sr) {
    __shared__ f32x4 red[4][FP4_GEMV_RG][64];
    __shared__ uint32_t last_flag;
    __shared__ u32x2 scale_lut[128];  // the loop is bound by vector instruction issue and the LDS pipe is idle in it
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r = lane & 15, g = lane >> 4;
    fp4_scale_lut_fill(scale_lut);
    const uint32_t scale_rot = (8 * g + 29) & 31;  // rotating right by this leaves the lane's scale byte times 8 in bits 3..10
    const uint32_t nts = n / 128, nt = blockIdx.x % nts, split = blockIdx.x / nts;
    const uint32_t ktiles = k / 64, kt_begin = split * ktiles / sk, kt_end = (split + 1) * ktiles / sk;
    const uint8_t* wp = w + (size_t)nt * w_snt + (size_t)r * w_sr + 8 * g;
    const uint8_t* sp = sw + (size_t)nt * s_snt + (size_t)r * s_sr;
    const _Float16* xp[XR];
#pragma unroll
    for (int xr = 0; xr < XR; xr++) xp[xr] = aq + (size_t)(16 * xr + r < m ? 16 * xr + r : m - 1) * k + 16 * g;

    auto load = [&](Fp4GemvStage<XR>& st, uint32_t kt) {
        const uint8_t* wk = wp + (size_t)kt * w_skt;
        const uint8_t* sk_ = sp + (size_t)kt * s_skt;
#pragma unroll
        for (int rg = 0; rg < FP4_GEMV_RG; rg++) {
            const u32x2* cw = (const u32x2*)(wk + (size_t)(16 * rg) * w_sr);
            const uint32_t* sc = (const uint32_t*)(sk_ + (size_t)(16 * rg) * s_sr);
            st.cw[rg] = NT ? __builtin_nontemporal_load(cw) : *cw;
            st.sc[rg] = NT ? __builtin_nontemporal_load(sc) : *sc;
        }
#pragma unroll
        for (int xr = 0; xr < XR; xr++) {
            st.x[xr][0] = *(const f16x8*)(xp[xr] + kt * 64);
            st.x[xr][1] = *(const f16x8*)(xp[xr] + kt * 64 + 8);
        }
    };
    f32x4 acc[XR][FP4_GEMV_RG];
#pragma unroll
    for (int xr = 0; xr < XR; xr++)
#pragma unroll
        for (int rg = 0; rg < FP4_GEMV_RG; rg++) acc[xr][rg] = (f32x4){0.f, 0.f, 0.f, 0.f};
    auto compute = [&](const Fp4GemvStage<XR>& st) {
#pragma unroll
        for (int rg = 0; rg < FP4_GEMV_RG; rg++) {
            const uint32_t at = __builtin_amdgcn_alignbit(st.sc[rg], st.sc[rg], scale_rot) & 0x3f8;
            const Fp4Scale s = fp4_scale_lut(scale_lut, at);
#pragma unroll
            for (int j = 0; j < 2; j++) {
                u32x4 a = fp4x8_to_f16(st.cw[rg][j], s);
#pragma unroll
                for (int xr = 0; xr < XR; xr++)
                    acc[xr][rg] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), st.x[xr][j], acc[xr][rg], 0, 0, 0);
            }
        }
    };
    // NS k tiles in flight per wavefront (a ring of stages indexed by constants; three, four and six were measured and
    // are no faster). Loads past the end of the run are skipped (a wavefront-uniform branch).
    constexpr int NS = 2;
    Fp4GemvStage<XR> st[NS];
    uint32_t kt = kt_begin + wave;
#pragma unroll
    for (int i = 0; i < NS; i++)
        if (kt + 4 * i < kt_end) load(st[i], kt + 4 * i);
    __syncthreads();  // scale_lut
    // (the scheduling barriers keep each refill where it is written: the compiler otherwise sinks the loads to just
    // before their use, a whole stage later)
    for (; kt < kt_end; kt += 4 * NS) {
#pragma unroll
        for (int i = 0; i < NS; i++) {
            if (kt + 4 * i < kt_end) compute(st[i]);
            __builtin_amdgcn_sched_barrier(0);
            if (kt + 4 * (i + NS) < kt_end) load(st[i], kt + 4 * (i + NS));
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    // The four wavefronts' sums meet in LDS, one group of activation rows at a time; wavefront v finishes weight row
    // groups 2 v and 2 v + 1. Lane (r, g) then holds, for weight row group rg, output row 16 xr + r, columns
    // n0 + 16 rg + 4 g .. + 3.
    const uint32_t col = nt * 128 + 32 * wave + 4 * g;  // + 16 h
    f32x4 sum[XR][2];
#pragma unroll
    for (int xr = 0; xr < XR; xr++) {
        if (xr) __syncthreads();
#pragma unroll
        for (int rg = 0; rg < FP4_GEMV_RG; rg++) red[wave][rg][lane] = acc[xr][rg];
        __syncthreads();
#pragma unroll
        for (int h = 0; h < 2; h++) {
            sum[xr][h] = red[0][2 * wave + h][lane];
#pragma unroll
            for (int v = 1; v < 4; v++) sum[xr][h] += red[v][2 * wave + h][lane];
        }
    }
    auto finish = [&](uint32_t row, const f32x4 (&v)[2]) {
        if (row >= m) return;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            uint32_t cc = col + 16 * h;
            float o[4] = {v[h][0], v[h][1], v[h][2], v[h][3]};
            fp4_store4(out.c, out.res, (size_t)row * out.ldc + cc, o, *(const f32x4*)(alpha + cc) * FP4_OPERAND_SCALE);
        }
    };
    constexpr uint32_t PITCH = 132;
    float* tile = (float*)red;  // SWIGLU: [16 XR][PITCH] of the finished tile
    static_assert(sizeof(red) >= 16 * XR * PITCH * 4, "tile");
    auto finish_tile = [&](const f32x4 (&v)[XR][2]) {
#pragma unroll
        for (int xr = 0; xr < XR; xr++)
#pragma unroll
            for (int h = 0; h < 2; h++) *(f32x4*)(tile + (16 * xr + r) * PITCH + 32 * wave + 16 * h + 4 * g) = v[xr][h];
        __syncthreads();
        const uint32_t l32 = tid & 31, at = nt * 128 + 4 * l32;
        const f32x4 al = *(const f32x4*)(alpha + at) * FP4_OPERAND_SCALE;
        for (uint32_t row = tid >> 5; row < 16 * XR; row += 8) {
            const f32x4 p = *(const f32x4*)(tile + row * PITCH + 4 * l32);
            const float o[4] = {p[0], p[1], p[2], p[3]};
            swiglu_quant_store(o, al, l32, row < m, row < m ? row : 0, at, n, out.q_codes, out.q_sf, out.q_aq, out.qg);
        }
    };
    if (sk == 1) {
        if constexpr (SWIGLU) {
            __syncthreads();  // (the last group's sums have been read)
            finish_tile(sum);
        } else {
#pragma unroll
            for (int xr = 0; xr < XR; xr++) finish(16 * xr + r, sum[xr]);
        }
        return;
    }
    // Partials cross to another program, possibly on another XCD with its own L2: agent-scope accesses, ordered by the
    // barriers around the arrival counter. A program's partial lies in z as its lanes hold it (a wavefront's store is 1 KB
    // in one piece), and the finisher's lanes hold the same elements: zp(split, xr, h) is this lane's f32x4.
    auto zp = [&](uint32_t sp, int xr, int h) {
        return z + ((((size_t)nt * sk + sp) * XR + xr) * 8 + 2 * wave + h) * 256 + 4 * lane;
    };
#pragma unroll
    for (int xr = 0; xr < XR; xr++) {
        if (16 * xr + r < m) {
#pragma unroll
            for (int h = 0; h < 2; h++) store_agent_f32x4(zp(split, xr, h), sum[xr][h]);
        }
    }
    agent_stores_wait();  // this lane's stores are acknowledged at agent scope
    __syncthreads();
    if (tid == 0) {
        uint32_t old = __hip_atomic_fetch_add(&counters[nt], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        last_flag = (old == sk - 1);
    }
    __syncthreads();
    if (!last_flag) return;
    if (tid == 0) __hip_atomic_store(&counters[nt], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    // the loads of up to 8 splits are in flight together (an agent-scope load takes a trip to memory); sums in split order
    const __amdgpu_buffer_rsrc_t zrs = __builtin_amdgcn_make_buffer_rsrc((void*)z, 0, nts * sk * XR * 8192u, 0x00020000);
#pragma unroll
    for (int xr = 0; xr < XR; xr++) {
        const uint32_t row = 16 * xr + r;
        if (row >= m) {
            if constexpr (SWIGLU) sum[xr][0] = sum[xr][1] = f32x4{};
            continue;
        }
        f32x4 tot[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
        for (uint32_t s0 = 0; s0 < sk; s0 += 8) {
            f32x4 t[16];
#pragma unroll
            for (int b = 0; b < 8; b++) {
                if (s0 + b < sk) {
#pragma unroll
                    for (int h = 0; h < 2; h++)
                        t[2 * b + h] = load_agent_f32x4(zrs, (uint32_t)((const char*)zp(s0 + b, xr, h) - (const char*)z), 0);
                } else {
                    t[2 * b] = t[2 * b + 1] = (f32x4){0.f, 0.f, 0.f, 0.f};
                }
            }
            agent_loads_wait(t);
#pragma unroll
            for (int b = 0; b < 8; b++)
                if (s0 + b < sk) {
#pragma unroll
                    for (int h = 0; h < 2; h++) tot[h] += t[2 * b + h];
                }
        }
        if constexpr (SWIGLU)
            sum[xr][0] = tot[0], sum[xr][1] = tot[1];
        else
            finish(row, tot);
    }
    if constexpr (SWIGLU) finish_tile(sum);  // (two barriers since red was read)
}

#define FP4_GEMV_KERNEL(XR, SUFFIX, NT)                                                                                \
    extern "C" __global__ __launch_bounds__(256, 2) void fe_gemv_nvfp4_x##XR##SUFFIX(                                  \
        uint16_t* c, const _Float16* aq, const uint8_t* w, const uint8_t* sw, const float* alpha, const uint16_t* res, \
        float* z, uint32_t* counters, uint32_t m, uint32_t n, uint32_t k, uint32_t ldc, uint32_t sk, uint32_t w_snt,   \
        uint32_t w_skt, uint32_t w_sr, uint32_t s_snt, uint32_t s_skt, uint32_t s_sr) {                                \
        gemv_nvfp4_body<XR, NT, false>(FpOut{c, res, ldc, nullptr, nullptr, nullptr, 0.f}, aq, w, sw, alpha, z, counters, m, n, k, sk, \
                                       w_snt, w_skt, w_sr, s_snt, s_skt, s_sr);                                        \
    }                                                                                                                  \
    extern "C" __global__ __launch_bounds__(256, 2) void fe_gemv_nvfp4_swiglu_x##XR##SUFFIX(                           \
        const _Float16* aq, const uint8_t* w, const uint8_t* sw, const float* alpha, float* z, uint32_t* counters,     \
        uint32_t m, uint32_t n, uint32_t k, uint32_t sk, uint32_t w_snt, uint32_t w_skt, uint32_t w_sr, uint32_t s_snt, \
        uint32_t s_skt, uint32_t s_sr, uint8_t* q_codes, uint8_t* q_sf, _Float16* q_aq, float qg) {                    \
        gemv_nvfp4_body<XR, NT, true>(FpOut{nullptr, nullptr, 0, q_codes, q_sf, q_aq, qg}, aq, w, sw, alpha, z, counters, m, n, k, sk, \
                                      w_snt, w_skt, w_sr, s_snt, s_skt, s_sr);                                         \
    }
FP4_GEMV_KERNEL(1, , true) FP4_GEMV_KERNEL(1, _v, false)
FP4_GEMV_KERNEL(2, , true) FP4_GEMV_KERNEL(2, _v, false)
FP4_GEMV_KERNEL(3, , true) FP4_GEMV_KERNEL(3, _v, false)  // (four groups of rows would not fit the registers of two programs a CU)

// ---- GEMV over programs of 8 CO columns (1..16 rows): no hand-off, every operand straight into LDS ---------------------------------
//
// y[r][n] for r < m <= 2 XP. grid ceil(N / 8 CO), 64 WV threads: a program takes 8 CO weight rows over all of K, its wavefronts (four or eight:
// wide_form of fe_fp4.cpp) a quarter or an eighth of K's steps of 256 each (four k tiles). Sums of quarters are added in order; where wide_form sums
// eighths (EIGHTHS: all forms of such a linear alike), two of them make a quarter. A row's bits depend on W's shape and values and, by wide_form's
// line, on the device's count of CUs only. K % 256 == 0. Lane L = 16 g + r multiplies, for 16 weight rows, row r's k tile 4 s + g (64 codes, four
// block scales) with the activations of the same k; the order of k inside a step does not matter. Stages belong to one wavefront (no barrier in the
// loop). Codes: 8 weight rows a load, [4 k tiles][8 rows][32 bytes]; lanes of odd g read the second half of a row's k tile first, so that 16 lanes
// that read together cover the 64 banks. Scales: 16 rows a load, [4 k tiles][16 rows][4]. Activations: 2 rows a load, 512 bytes each, chunk c at
// position c ^ (row & 15) in its half.
//
// Bound by the codes' way from HBM and the start of a launch at one row, by the activations' way from L2 from 8 rows on. It replaces programs of 16
// weight rows with the activations staged whole (one and two rows: too many programs, each waiting for its own staging) and, up to 16 rows, weight
// tiles cut along K (whose partial sums meet through memory; 17 rows and more still run there). us with the quantizer's launch, before -> now: 5120 x
// 34816 at 1 / 4 / 8 / 16 rows 25.6 -> 22.1, 32.2 -> 22.1, 32.4 -> 25.7, 34.4 -> 28.8; 17408 x 5120 19.0 -> 14.3, 17.8 -> 14.9, 18.0 -> 18.4, 19.3 ->
// 20.7; 5120 x 5120 9.6 -> 9.0, 10.3 -> 9.0, 12.2 -> 9.1, 12.5 -> 10.1 (four wavefronts). Eight wavefronts against four: wide_form. Deeper stages in
// place of more wavefronts lose: 5120 x 17408 at 1 row 17.3 -> 18.8 with eight steps in flight for three.
//
// Q: the program quantizes the activations itself, in front of its first step. aq is then bf16 rows [m][ldx]: a wavefront moves its quarter of K into LDS as
// it is, in front of the first weights, makes fe_fp4_quant's values of it in their places (a block of 16 a lane) while the weights are on their way, and every
// step reads them there; program 0 leaves codes, scales and operand in memory as that kernel does. The same bits, and a launch less: for few values
// (fp4_quants_itself of fe_fp4.cpp), since every program quantizes all of them.
struct Fp4QuantTo {
    uint8_t *codes, *sf;
    _Float16* aq;
    uint32_t ldx;
    float g;
};
template <int XP, int CO, bool Q, int WV>
struct Fp4Wide {
    static constexpr int CG = (CO + 1) / 2, XL = Q ? 0 : XP, L = CO + CG + XL;
    static constexpr int SC_AT = CO * 1024, X_AT = SC_AT + CG * 256, STAGE = X_AT + XL * 1024;
    static constexpr int FIT = (Q ? 60 : 80) * 1024 / (WV * STAGE), DEPTH = FIT < 2 ? 2 : FIT < 6 ? FIT : 6;  // two programs a CU where two steps allow it
    static constexpr int RED = WV * 16 * (16 * CG + 4) * 4, LDS = WV * DEPTH * STAGE > RED ? WV * DEPTH * STAGE : RED;
    static_assert(DEPTH >= 2 && (DEPTH - 1) * L < (Q ? 48 : 64) && LDS <= 160 * 1024, "stages");
};

template <int XP, int CO, bool Q, int WV, bool EIGHTHS>
__device__ __forceinline__ void gemv_nvfp4_wide_body(uint16_t* c, const _Float16* aq, const uint8_t* w, const uint8_t* sw,
                                                     const float* alpha, const uint16_t* res, uint32_t m, uint32_t n, uint32_t k,
                                                     uint32_t ldc, uint32_t w_snt, uint32_t w_skt, uint32_t w_sr, uint32_t s_snt,
                                                     uint32_t s_skt, uint32_t s_sr, const Fp4QuantTo qt) {
    typedef Fp4Wide<XP, CO, Q, WV> C;
    constexpr int CG = C::CG, AHEAD = C::DEPTH - 1, PITCH = 16 * CG + 4;
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r = lane & 15, g = lane >> 4;
    const uint32_t col0 = blockIdx.x * 8 * CO, nt0 = col0 / 128, nts = n / 128, span = nts - nt0 < 2 ? nts - nt0 : 2;
    const u32x4 wrs = g8_rsrc(w + (size_t)nt0 * w_snt, span * 128 * (k / 2)), srs = g8_rsrc(sw + (size_t)nt0 * s_snt, span * 128 * (k / 16));
    const u32x4 xrs = g8_rsrc(aq, Q ? ((m - 1) * qt.ldx + k) * 2 : m * k * 2);
    // weight row `row` of the program (past n: the last one again, not stored), byte offset from weight tile nt0
    auto at = [&](uint32_t row, uint32_t snt, uint32_t sr) {
        const uint32_t i = (col0 + row < n ? col0 + row : n - 1) - 128 * nt0;
        return (i >> 7) * snt + (i & 127) * sr;
    };
    uint32_t vw[CO], vs[CG], vx[C::XL + 1];
#pragma unroll
    for (int j = 0; j < CO; j++) vw[j] = at(8 * j + ((lane >> 1) & 7), w_snt, w_sr) + g * w_skt + (lane & 1) * 16;
#pragma unroll
    for (int j = 0; j < CG; j++) vs[j] = at(16 * j + r, s_snt, s_sr) + g * s_skt;
#pragma unroll
    for (int j = 0; j < C::XL; j++) {
        const uint32_t row = 2 * j + (lane >> 5), chunk = (lane & 16) | ((lane ^ row) & 15);
        vx[j] = (row < m ? row : m - 1) * k * 2 + chunk * 16;
    }
    unsigned char* stages = lds + wave * (C::DEPTH * C::STAGE);
    const uint32_t stages0 = g8_lds_addr(stages);
    // EIGHTHS with four wavefronts: two eighths each, steps up to mid and from mid on, summed apart
    constexpr bool TWO = EIGHTHS && WV == 4;
    const uint32_t steps = k / 256, s0 = wave * steps / WV, count = (wave + 1) * steps / WV - s0, mid = TWO ? (2 * wave + 1) * steps / 8 - s0 : 0;
    auto issue = [&](uint32_t s, uint32_t slot) {
        const uint32_t to = stages0 + slot * C::STAGE;
#pragma unroll
        for (int j = 0; j < CO; j++) g8_load_lds16_nt(wrs, to + j * 1024, vw[j], (s0 + s) * 4 * w_skt);
#pragma unroll
        for (int j = 0; j < CG; j++) g8_load_lds4(srs, to + C::SC_AT + j * 256, vs[j], (s0 + s) * 4 * s_skt);
#pragma unroll
        for (int j = 0; j < C::XL; j++) g8_load_lds16(xrs, to + C::X_AT + j * 1024, vx[j], (s0 + s) * 512);
    };
    const uint32_t odd = g & 1, xr = r < m ? r : m - 1;
    // Q: the wavefront's activations, [its steps][m rows][512 bytes] (a whole number of loads), chunks placed as in a stage
    unsigned char* xq = lds + WV * C::DEPTH * C::STAGE + wave * (((steps + WV - 1) / WV * m + 1) / 2 * 1024);
    // half h of the lane's row and k tile; the 16-byte chunk of 8 activations that goes with code 32 (h ^ odd) + 8 e on
    uint32_t fw[CG], fx[8];
#pragma unroll
    for (int j = 0; j < CG; j++) {
        const uint32_t row = 16 * j + r < 8 * CO ? 16 * j + r : 8 * CO - 1;
        fw[j] = (row >> 3) * 1024 + g * 256 + (row & 7) * 32;
    }
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const uint32_t chunk = 8 * g + 4 * (h ^ odd) + e;
            fx[4 * h + e] = (Q ? 0 : C::X_AT) + xr * 512 + (((chunk & 16) | ((chunk ^ xr) & 15)) << 4);
        }
    f32x4 acc[CG] = {}, low[CG] = {};
    auto half = [&]() {
#pragma unroll
        for (int j = 0; j < CG; j++) low[j] = acc[j], acc[j] = f32x4{};
    };
    uint32_t slot = 0;
    auto add = [&](uint32_t s) {
        const unsigned char *st = stages + slot * C::STAGE, *xst = Q ? xq + s * (m * 512) : st;
        uint32_t sc[CG];
#pragma unroll
        for (int j = 0; j < CG; j++) {
            const uint32_t b = *(const uint32_t*)(st + C::SC_AT + j * 256 + lane * 4);
            sc[j] = __builtin_amdgcn_alignbit(b, b, 16 * odd);
        }
#pragma unroll
        for (int h = 0; h < 2; h++) {
            f16x8 x[4];
#pragma unroll
            for (int e = 0; e < 4; e++) x[e] = *(const f16x8*)(xst + fx[4 * h + e]);
#pragma unroll
            for (int j = 0; j < CG; j++) {
                const u32x4 codes = *(const u32x4*)(st + fw[j] + 16 * (h ^ odd));
#pragma unroll
                for (int e = 0; e < 4; e++)
                    acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                        fp4x8_scaled(codes[e], fp4_scale_2m8(__builtin_amdgcn_ubfe(sc[j], 16 * h + 8 * (e >> 1), 8))), x[e], acc[j], 0, 0, 0);
            }
        }
        slot = slot + 1 == C::DEPTH ? 0 : slot + 1;
    };
    if (count) {
        if constexpr (Q) {
            const uint32_t xq0 = g8_lds_addr(xq), units = count * m;  // a unit: 256 values of a row, half a load
            for (uint32_t u0 = 0; u0 < units; u0 += 2) {
                const uint32_t u = u0 + (lane >> 5) < units ? u0 + (lane >> 5) : u0, s = u / m, row = u - s * m;
                g8_load_lds16(xrs, xq0 + u0 * 512, (row * qt.ldx + (s0 + s) * 256) * 2 + ((lane & 16) | ((lane ^ row) & 15)) * 16, 0);
            }
        }
#pragma unroll
        for (int u = 0; u < AHEAD; u++) issue((uint32_t)u < count ? u : count - 1, u);  // past the end: the last step again, not added
        if constexpr (Q) {
            g8_loads_wait<AHEAD * C::L>();
            for (uint32_t i = lane; i < count * m * 16; i += 64) {
                const uint32_t u = i >> 4, b = i & 15, s = u / m, row = u - s * m, c = 2 * b;
                u32x4 *p0 = (u32x4*)(xq + u * 512 + (((c & 16) | ((c ^ row) & 15)) << 4)), *p1 = (u32x4*)(xq + u * 512 + ((((c + 1) & 16) | (((c + 1) ^ row) & 15)) << 4));
                const Fp4Block v = fp4_quant_block(*p0, *p1, qt.g);
                *p0 = v.o[0], *p1 = v.o[1];
                if (blockIdx.x == 0) fp4_store_block(v, qt.codes, qt.sf, qt.aq, row, (s0 + s) * 16 + b, k);
            }
            asm volatile("" ::: "memory");
        }
        uint32_t s = 0;
        if constexpr (TWO && AHEAD == 1) {  // (with the sums taken apart inside one loop they would move between register files every step)
            for (; s < mid; s++) {
                g8_loads_wait<0>();
                issue(s + 1, slot ? 0 : 1);  // (mid < count)
                add(s);
            }
            half();
        }
        for (; s + AHEAD < count; s++) {
            if (TWO && AHEAD > 1 && s == mid) half();
            g8_loads_wait<(AHEAD - 1) * C::L>();  // (the stage in front of this one has been read, too)
            issue(s + AHEAD, slot ? slot - 1 : AHEAD);
            add(s);
        }
        auto tail = [&](auto u_tag) {
            constexpr int U = decltype(u_tag)::value;
            if constexpr (U < AHEAD)
                if (s + U < count) {
                    if (TWO && AHEAD > 1 && s + U == mid) half();
                    g8_loads_wait<(AHEAD - 1 - U) * C::L>();
                    add(s + U);
                }
        };
        tail(std::integral_constant<int, 0>{});
        tail(std::integral_constant<int, 1>{});
        tail(std::integral_constant<int, 2>{});
        tail(std::integral_constant<int, 3>{});
        tail(std::integral_constant<int, 4>{});
        g8_loads_wait<0>();
    }
    float(*red)[16][PITCH] = (float(*)[16][PITCH])lds;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < CG; j++) *(f32x4*)&red[wave][r][16 * j + 4 * g] = TWO ? low[j] + acc[j] : acc[j];
    __syncthreads();
    for (uint32_t i = tid; i < m * 2 * CO; i += 64 * WV) {
        const uint32_t row = i / (2 * CO), j = 4 * (i % (2 * CO)), col = col0 + j;
        if (col >= n) continue;
        auto quarter = [&](int p) { return WV == 8 ? *(const f32x4*)&red[2 * p][row][j] + *(const f32x4*)&red[2 * p + 1][row][j] : *(const f32x4*)&red[p][row][j]; };
        const f32x4 sum = ((quarter(0) + quarter(1)) + quarter(2)) + quarter(3);
        const float v[4] = {sum[0], sum[1], sum[2], sum[3]};
        fp4_store4(c, res, (size_t)row * ldc + col, v, *(const f32x4*)(alpha + col) * FP4_GEMM_SCALE);
    }
}

#define FP4_WIDE_KERNEL(XP, CO, SUFFIX, WV, EIGHTHS)                                                                      \
    extern "C" __global__ __launch_bounds__(64 * WV) void fe_gemv_nvfp4_r##XP##_c##CO##SUFFIX(                            \
        uint16_t* c, const _Float16* aq, const uint8_t* w, const uint8_t* sw, const float* alpha, const uint16_t* res,   \
        uint32_t m, uint32_t n, uint32_t k, uint32_t ldc, uint32_t w_snt, uint32_t w_skt, uint32_t w_sr, uint32_t s_snt, \
        uint32_t s_skt, uint32_t s_sr) {                                                                                  \
        gemv_nvfp4_wide_body<XP, CO, false, WV, EIGHTHS>(c, aq, w, sw, alpha, res, m, n, k, ldc, w_snt, w_skt, w_sr, s_snt, s_skt, s_sr, Fp4QuantTo{}); \
    }
#define FP4_WIDE_QUANT_KERNEL(XP, CO, SUFFIX, WV, EIGHTHS)                                                                \
    extern "C" __global__ __launch_bounds__(64 * WV) void fe_gemv_nvfp4_q##XP##_c##CO##SUFFIX(                            \
        uint16_t* c, const _Float16* x, const uint8_t* w, const uint8_t* sw, const float* alpha, const uint16_t* res,    \
        uint32_t m, uint32_t n, uint32_t k, uint32_t ldc, uint32_t w_snt, uint32_t w_skt, uint32_t w_sr, uint32_t s_snt, \
        uint32_t s_skt, uint32_t s_sr, Fp4QuantTo qt) {                                                                   \
        gemv_nvfp4_wide_body<XP, CO, true, WV, EIGHTHS>(c, x, w, sw, alpha, res, m, n, k, ldc, w_snt, w_skt, w_sr, s_snt, s_skt, s_sr, qt); \
    }
// "": quarters of K. "_e": eighths, by eight wavefronts where two stages of eight fit the LDS, else by four.
#define FP4_WIDE_FIVE(KERNEL, XP, SUFFIX, WV, EIGHTHS) \
    KERNEL(XP, 2, SUFFIX, WV, EIGHTHS) KERNEL(XP, 3, SUFFIX, WV, EIGHTHS) KERNEL(XP, 4, SUFFIX, WV, EIGHTHS) KERNEL(XP, 5, SUFFIX, WV, EIGHTHS) KERNEL(XP, 6, SUFFIX, WV, EIGHTHS)
#define FP4_WIDE_SIX(KERNEL, XP, SUFFIX, WV, EIGHTHS) KERNEL(XP, 1, SUFFIX, WV, EIGHTHS) FP4_WIDE_FIVE(KERNEL, XP, SUFFIX, WV, EIGHTHS)
FP4_WIDE_SIX(FP4_WIDE_KERNEL, 1, , 4, false) FP4_WIDE_KERNEL(1, 9, , 4, false)
FP4_WIDE_SIX(FP4_WIDE_KERNEL, 2, , 4, false) FP4_WIDE_KERNEL(2, 9, , 4, false)
FP4_WIDE_SIX(FP4_WIDE_KERNEL, 4, , 4, false) FP4_WIDE_KERNEL(4, 9, , 4, false)
FP4_WIDE_SIX(FP4_WIDE_KERNEL, 8, , 4, false) FP4_WIDE_KERNEL(8, 9, , 4, false)
FP4_WIDE_SIX(FP4_WIDE_QUANT_KERNEL, 1, , 4, false)
FP4_WIDE_SIX(FP4_WIDE_QUANT_KERNEL, 2, , 4, false)
FP4_WIDE_SIX(FP4_WIDE_QUANT_KERNEL, 4, , 4, false)
FP4_WIDE_SIX(FP4_WIDE_KERNEL, 1, _e, 8, true)
FP4_WIDE_SIX(FP4_WIDE_KERNEL, 2, _e, 8, true)
FP4_WIDE_KERNEL(4, 1, _e, 8, true) FP4_WIDE_KERNEL(4, 2, _e, 8, true) FP4_WIDE_KERNEL(4, 3, _e, 8, true) FP4_WIDE_KERNEL(4, 4, _e, 8, true)
FP4_WIDE_KERNEL(4, 5, _e, 4, true) FP4_WIDE_KERNEL(4, 6, _e, 4, true)
FP4_WIDE_SIX(FP4_WIDE_KERNEL, 8, _e, 4, true)
FP4_WIDE_FIVE(FP4_WIDE_QUANT_KERNEL, 1, _e, 8, true)
FP4_WIDE_FIVE(FP4_WIDE_QUANT_KERNEL, 2, _e, 8, true)
FP4_WIDE_FIVE(FP4_WIDE_QUANT_KERNEL, 4, _e, 8, true)

// ---- matrix-unit peak probe ---------------------------------------------------------------------------------------------
//
// Every wavefront issues iters x 16 independent matrix instructions (the GEMM core's 4 x 4 accumulator pieces, 256
// accumulator registers) on operands that stay in registers: no memory traffic, no LDS (kernels/k-fp4/src/lib.rs:866-916,
// fe_fp4_peak). KIND 0: v_mfma_f32_32x32x16_f16, 1: v_mfma_f32_32x32x16_bf16, 2: v_mfma_f32_32x32x64_f8f6f4 on e4m3
// codes (the unscaled form). seed == 0: every operand element is 0.5 or 1 (few bits toggle from one instruction to the
// next, the reference's kind of pattern); otherwise signs and mantissas are random bits of the seed (an even seed:
// only the top five mantissa bits of the 16-bit kinds), magnitudes in [0.5, 2), as the operands of a GEMM on real data toggle: the clock the board
// holds under its power limit depends on it. One float a lane is written so that nothing is dead code. Flops of a launch: wavefronts x iters x 16 x 2
// x 32 x 32 x
// (16 or 64).
template <int KIND>
__device__ __forceinline__ void mfma_peak_body(float* out, uint32_t iters, uint32_t seed) {
    const uint32_t lane = threadIdx.x & 63;
    f32x16 acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 4; j++)
#pragma unroll
            for (int e = 0; e < 16; e++) acc[i][j][e] = 0.f;
    uint32_t rs = seed * 0x9e3779b9u + (blockIdx.x * 256 + threadIdx.x) * 0x85ebca6bu;
    auto rnd = [&]() {
        rs ^= rs << 13, rs ^= rs >> 17, rs ^= rs << 5;
        return seed ? rs : 0u;
    };
    // 16-bit pairs: sign and mantissa from the random word, exponent of 0.5 or 1; e4m3 quadruples likewise
    // (an even seed keeps only the top five mantissa bits of the 16-bit kinds: the six significant bits of an NVFP4 operand)
    const uint32_t keep16 = seed & 1 ? (KIND == 1 ? 0x80ff80ffu : 0x87ff87ffu) : (KIND == 1 ? 0x80fc80fcu : 0x87e087e0u);
    const uint32_t base16 = KIND == 1 ? 0x3f003f00u : 0x38003800u;
    auto h = [&](uint32_t flip) { return ((rnd() & keep16) | base16) ^ flip; };
    auto c = [&](uint32_t flip) { return (int)(((rnd() & 0x8f8f8f8fu) | 0x30303030u) ^ flip); };
    u32x4 a16[4], b16[4];
    g8_i32x8 a8[4], b8[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        a16[i] = (u32x4){h(0), h((lane & 1) << 15), h(0), h((uint32_t)i << 31)};
        b16[i] = (u32x4){h((lane & 2) << 14), h(0), h((uint32_t)i << 15), h(0)};
        a8[i] = (g8_i32x8){c(0), c((lane & 1) << 7), c((uint32_t)i << 31), c(0), c(0), c(0), c(0), c(0)};
        b8[i] = (g8_i32x8){c(0), c((lane & 2) << 6), c(0), c(0), c(0), c((uint32_t)i << 15), c(0), c(0)};
    }
    for (uint32_t it = 0; it < iters; it++) {
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                if constexpr (KIND == 0)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a16[i]), __builtin_bit_cast(f16x8, b16[j]),
                                                                      acc[i][j], 0, 0, 0);
                else if constexpr (KIND == 1)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a16[i]), __builtin_bit_cast(bf16x8, b16[j]),
                                                                       acc[i][j], 0, 0, 0);
                else
                    acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a8[i], b8[j], acc[i][j], 0, 0, 0, 0, 0, 0);
            }
    }
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 4; j++)
#pragma unroll
            for (int e = 0; e < 16; e++) sum += acc[i][j][e];
    out[blockIdx.x * blockDim.x + threadIdx.x] = sum;
}
extern "C" __global__ __launch_bounds__(256, 1) void fe_mfma_peak_f16(float* out, uint32_t iters, uint32_t seed) {
    mfma_peak_body<0>(out, iters, seed);
}
extern "C" __global__ __launch_bounds__(256, 1) void fe_mfma_peak_bf16(float* out, uint32_t iters, uint32_t seed) {
    mfma_peak_body<1>(out, iters, seed);
}
extern "C" __global__ __launch_bounds__(256, 1) void fe_mfma_peak_f8(float* out, uint32_t iters, uint32_t seed) {
    mfma_peak_body<2>(out, iters, seed);
}
