// EXL3 (trellis-coded, Hadamard-rotated) linear for gfx950: input rotation, the decode GEMV for 1..64 rows,
// whole-tensor reconstruct, and probes. (The prefill GEMMs are in k_exl3_gemm.hip, the decode in exl3_trellis.h.)
#include <type_traits>

#include "exl3_trellis.h"
#include "gemm8.h"

// ---- whole-tensor reconstruct (bits at run time: load-time code) ---------------------------------------------------

// 16-bit state of position p of a tile: two words and a funnel shift (kernels/k-exl3/src/recon.rs:12-22).
__device__ __forceinline__ uint32_t tile_state_rt(const uint32_t* tile, uint32_t bits, uint32_t p) {
    uint32_t words = 8 * bits;
    uint32_t b1 = (p + 1) * bits + 256 * bits;
    uint32_t b0 = b1 - 16;
    uint32_t i0 = b0 / 32, i1 = (b1 - 1) / 32;
    uint32_t s = (i1 + 1) * 32 - b1;
    uint32_t a = tile[i0 % words], b = tile[i1 % words];
    return (uint32_t)((((uint64_t)a << 32) | b) >> s) & 0xffff;
}

// W_hat (rotated basis) of columns nt0 * 16 .. + ns: grid (ns / 128, k / 16), 256 threads; half-wavefront w of the
// block decodes tile (blockIdx.y, nt0 + 8 blockIdx.x + w), lane f of it the 8 values of fragment lane f.
// OUT_F32 = 0: fp16 bits [k][ns]; 1: f32 [k][ns]. (kernels/k-exl3/src/recon.rs:24-51, 131-157)
template <int OUT_F32>
__device__ __forceinline__ void recon_hat_body(void* out, const uint32_t* trellis, uint32_t n_tiles, uint32_t nt0,
                                               uint32_t ns, uint32_t bits) {
    uint32_t hw = threadIdx.x / 32, f = threadIdx.x % 32;
    uint32_t kt = blockIdx.y, ntl = blockIdx.x * 8 + hw;
    const uint32_t* tile = trellis + (size_t)(kt * n_tiles + nt0 + ntl) * 8 * bits;
#pragma unroll
    for (uint32_t j = 0; j < 8; j += 2) {
        uint32_t h = decode2_mul1(tile_state_rt(tile, bits, f * 8 + j), tile_state_rt(tile, bits, f * 8 + j + 1));
#pragma unroll
        for (uint32_t e = 0; e < 2; e++) {
            uint32_t jj = j + e, v = e ? (h >> 16) : (h & 0xffff);
            uint32_t row = 2 * (f & 3) + (jj & 1) + 8 * ((jj >> 1) & 1);
            uint32_t col = (f >> 2) + 8 * (jj >> 2);
            size_t at = (size_t)(kt * 16 + row) * ns + ntl * 16 + col;
            if (OUT_F32)
                ((float*)out)[at] = f16_bits_to_f32(v);
            else
                ((uint16_t*)out)[at] = (uint16_t)v;
        }
    }
}

extern "C" __global__ __launch_bounds__(256) void exl3_recon_hat_f16(uint16_t* out, const uint32_t* trellis,
                                                                     uint32_t n_tiles, uint32_t nt0, uint32_t ns,
                                                                     uint32_t bits) {
    recon_hat_body<0>(out, trellis, n_tiles, nt0, ns, bits);
}

extern "C" __global__ __launch_bounds__(256) void exl3_recon_hat_f32(float* out, const uint32_t* trellis,
                                                                     uint32_t n_tiles, uint32_t nt0, uint32_t ns,
                                                                     uint32_t bits) {
    recon_hat_body<1>(out, trellis, n_tiles, nt0, ns, bits);
}

// In place: H over each row's 128-column blocks, * svh[n0 + col] / sqrt(128). grid (ns / 256, k), 64 threads: each
// half of the wavefront owns one 128-column block (ns / 128 odd: the last block's upper half idles).
// (kernels/k-exl3/src/recon.rs:54-64)
extern "C" __global__ __launch_bounds__(64) void exl3_had_rows(float* buf, uint32_t ns, const uint16_t* svh, uint32_t n0) {
    uint32_t lane = threadIdx.x, l32 = lane & 31;
    uint32_t c = (blockIdx.x * 2 + (lane >> 5)) * 128 + 4 * l32;
    bool live = c < ns;
    float* p = buf + (size_t)blockIdx.y * ns + (live ? c : 0);
    float v[4] = {p[0], p[1], p[2], p[3]};
    fwht128_half_wave(v, l32);
    if (live) {
#pragma unroll
        for (int q = 0; q < 4; q++) p[q] = v[q] * FE_HAD_SCALE * f16_bits_to_f32(svh[n0 + c + q]);
    }
}

// H over k (128-row blocks) * suh / sqrt(128) -> bf16, [k][n] (nk = 0, ld = n) or [n][k] (nk = 1, ld = k).
// grid (ns / 32, k / 128), 128 threads, a 128 x 32 f32 tile in LDS. (kernels/k-exl3/src/recon.rs:66-128)
extern "C" __global__ __launch_bounds__(128) void exl3_had_cols_bf16(const float* buf, uint16_t* out, uint32_t ns,
                                                                      const uint16_t* suh, uint32_t n0, uint32_t ld,
                                                                      uint32_t nk) {
    constexpr uint32_t PITCH = 33;
    __shared__ float sm[128 * PITCH];
    uint32_t hw = threadIdx.x / 32, l32 = threadIdx.x % 32;
    uint32_t r0 = blockIdx.y * 128, c0 = blockIdx.x * 32;
    for (uint32_t i = 0; i < 32; i++) {
        uint32_t r = hw * 32 + i;
        sm[r * PITCH + l32] = buf[(size_t)(r0 + r) * ns + c0 + l32];
    }
    __syncthreads();
    for (uint32_t cc = 0; cc < 8; cc++) {
        uint32_t c = hw * 8 + cc;
        float v[4];
#pragma unroll
        for (uint32_t q = 0; q < 4; q++) v[q] = sm[(4 * l32 + q) * PITCH + c];
        fwht128_half_wave(v, l32);
#pragma unroll
        for (uint32_t q = 0; q < 4; q++) {
            uint32_t r = 4 * l32 + q;
            sm[r * PITCH + c] = v[q] * FE_HAD_SCALE * f16_bits_to_f32(suh[r0 + r]);
        }
    }
    __syncthreads();
    if (nk) {
        for (uint32_t cc = 0; cc < 8; cc++) {
            uint32_t c = hw * 8 + cc;
            float v[4];
#pragma unroll
            for (uint32_t q = 0; q < 4; q++) v[q] = sm[(4 * l32 + q) * PITCH + c];
            uint32_t* p = (uint32_t*)(out + (size_t)(n0 + c0 + c) * ld + r0 + 4 * l32);
            p[0] = pack_bf16x2(v[0], v[1]);
            p[1] = pack_bf16x2(v[2], v[3]);
        }
    } else {
        for (uint32_t i = 0; i < 32; i++) {
            uint32_t r = hw * 32 + i;
            out[(size_t)(r0 + r) * ld + n0 + c0 + l32] = (uint16_t)f32_to_bf16_bits(sm[r * PITCH + l32]);
        }
    }
}

// ---- input rotation ------------------------------------------------------------------------------------------------

// One 128-element block of a row: fp16(H(x * suh) / sqrt(128)), 4 elements a lane of a half wavefront. The input is
// bf16 (mode 0) or f32 (mode 1) rows, or (mode 2) SwiGLU of two bf16 arrays, x = gate and x2 = up, taken on the way in:
// bf16(bf16(silu(gate)) * up), the bits fe_silu_mul would have left in memory. `xat` indexes the input (row * ld + c),
// `c` is the block's channel of this lane. Split in two so that a caller can issue the loads early; all 32 lanes of the
// half wavefront take part in rot_finish.
struct RotSrc {
    const void *x, *x2;
    uint32_t mode, ld;  // ld: elements between input rows
};
struct RotRaw {
    f32x4 xf;
    u32x2 xb, ub, s;
};
__device__ __forceinline__ RotRaw rot_load(const RotSrc& src, const uint16_t* suh, size_t xat, uint32_t c) {
    RotRaw r;
    if (src.mode == 1) {
        r.xf = *(const f32x4*)((const float*)src.x + xat);
    } else {
        r.xb = *(const u32x2*)((const uint16_t*)src.x + xat);
        if (src.mode == 2) r.ub = *(const u32x2*)((const uint16_t*)src.x2 + xat);
    }
    r.s = *(const u32x2*)(suh + c);
    return r;
}
// The same for mode 2 when gate and up were written by other programs of this launch, possibly on another XCD: the
// loads are agent-scope buffer loads (gs, us: resources over the two arrays), which miss this XCD's L2.
__device__ __forceinline__ RotRaw rot_load_agent(__amdgpu_buffer_rsrc_t gs, __amdgpu_buffer_rsrc_t us, const uint16_t* suh,
                                                 uint32_t xat, uint32_t c) {
    RotRaw r;
    r.xb = __builtin_amdgcn_raw_buffer_load_b64(gs, 2 * xat, 0, 16);
    r.ub = __builtin_amdgcn_raw_buffer_load_b64(us, 2 * xat, 0, 16);
    r.s = *(const u32x2*)(suh + c);
    return r;
}
__device__ __forceinline__ u32x2 rot_finish(const RotRaw& r, uint32_t mode, uint32_t l32) {
    float v[4];
    if (mode == 1) {
        v[0] = r.xf[0], v[1] = r.xf[1], v[2] = r.xf[2], v[3] = r.xf[3];
    } else {
        u32x2 xb = r.xb;
        if (mode == 2) xb = (u32x2){silu_mul_bf16x2(r.xb[0], r.ub[0]), silu_mul_bf16x2(r.xb[1], r.ub[1])};
        v[0] = __uint_as_float(xb[0] << 16), v[1] = __uint_as_float(xb[0] & 0xffff0000u);
        v[2] = __uint_as_float(xb[1] << 16), v[3] = __uint_as_float(xb[1] & 0xffff0000u);
    }
    v[0] *= f16_bits_to_f32(r.s[0] & 0xffff), v[1] *= f16_bits_to_f32(r.s[0] >> 16);
    v[2] *= f16_bits_to_f32(r.s[1] & 0xffff), v[3] *= f16_bits_to_f32(r.s[1] >> 16);
    fwht128_half_wave(v, l32);
    return (u32x2){pack_f16x2(v[0] * FE_HAD_SCALE, v[1] * FE_HAD_SCALE), pack_f16x2(v[2] * FE_HAD_SCALE, v[3] * FE_HAD_SCALE)};
}

// xh[row][k] = fp16(H(x * suh) / sqrt(128)). grid (ceil(k / 512), rows), 128 threads: each half wavefront one
// 128-element block, 4 elements a lane. (kernels/k-exl3/src/gemv.rs:147-170)
__device__ __forceinline__ void rot_in_body(const RotSrc& src, const uint16_t* suh, uint16_t* xh, uint32_t k) {
    uint32_t l32 = threadIdx.x & 31;
    uint32_t blk = blockIdx.x * 4 + threadIdx.x / 32;
    bool live = blk * 128 < k;
    uint32_t c = (live ? blk : 0) * 128 + 4 * l32;
    u32x2 o = rot_finish(rot_load(src, suh, (size_t)blockIdx.y * src.ld + c, c), src.mode, l32);
    if (live) *(u32x2*)(xh + (size_t)blockIdx.y * k + c) = o;
}
extern "C" __global__ __launch_bounds__(128) void exl3_rot_in(const void* x, uint32_t x_mode, const uint16_t* suh,
                                                               uint16_t* xh, uint32_t k, const void* x2, uint32_t ldx) {
    rot_in_body(RotSrc{x, x2, x_mode, ldx}, suh, xh, k);
}

#define FE_EXL3_GROUP_MAX 4  // linears of one launch

// The same input rotated for several linears (each by its own suh into its own xh): grid (ceil(k / 512), rows, members).
struct RotGroup {
    const uint16_t* suh[FE_EXL3_GROUP_MAX];
    uint16_t* xh[FE_EXL3_GROUP_MAX];
};
extern "C" __global__ __launch_bounds__(128) void exl3_rot_in_group(RotGroup g, const void* x, uint32_t x_mode, uint32_t k) {
    rot_in_body(RotSrc{x, nullptr, x_mode, k}, g.suh[blockIdx.z], g.xh[blockIdx.z], k);
}

#ifndef FE_STAGE_NB1
#define FE_STAGE_NB1 4
#endif
#define GEMV_RED_PITCH 132  // floats a row of the 128-column partial sums (16-byte aligned, banks spread)

// ---- decode GEMV, balanced over the CUs (1..16 rows) ------------------------------------------------------------------
//
// Work unit = one 128-channel block of K of one 128-column block of N (two load steps); units are ordered column block
// by column block and the member's `programs` programs each take one contiguous run of them, base + 1 units for the first
// rem programs and base for the rest, whatever the shape: with a multiple of the CU count of programs, which the CUs take
// round by round, the CUs' shares differ by at most one unit. (Spreading the longer runs evenly over the program numbers
// is worse: their period can divide the CU count, and then a CU gets only long runs or only short ones.) A run may start and end inside a column
// block, so a block's sum is assembled from segments: each program leaves the partial sums of its segment of block nb in z[program + nb] and bumps
// the block's arrival counter; the program that arrives last adds the segments, those of programs 2 j and 2 j + 1 to each other first and the pairs
// in program order
// (so that gemv_wide_body can run a pair as one workgroup; the order does not depend on who is last: deterministic), applies the output rotation and
// re-arms the counter. The partition depends on (k, n, programs) only, never on the row count: row r of a batch has the bits of the single-row call.
// Inside a program: 4 wavefronts owning 2 of the block's 8 tiles each, the rotated inputs of the run staged in LDS (rotated here when src.x is set),
// four load steps in flight per lane. Several linears of one input share a launch: each member's programs are exactly those of its own launch (same
// runs, same sums, same bits). (kernels/k-exl3/src/gemv.rs:412-587 is the reference's split-K form.)
struct GemvMember {
    const uint32_t* trellis;
    const uint16_t *svh, *suh;
    uint16_t* xh;        // rotated inputs [m][k]: read, or (rotating here) left there by the programs of column block 0
    void* y;
    float* z;            // segment partial sums [programs + n / 128][m][128]
    uint32_t* counters;  // arrivals per column block, zero at rest
    uint32_t n, programs, stride_k, stride_nb;
    uint32_t base, rem;            // units / programs, units % programs, units = (n / 128) * (k / 128)
    uint32_t inv_base, inv_base1;  // floor((2^32 - 1) / base), floor((2^32 - 1) / (base + 1))
};
struct GemvJob {
    uint32_t count, first[FE_EXL3_GROUP_MAX + 1];  // member i owns workgroups first[i] .. first[i + 1] - 1 of the grid
    GemvMember m[FE_EXL3_GROUP_MAX];
};

// A launch's arguments lie in memory that no cache of the XCD holds when the launch begins, so the first scalar load of each of their lines is a trip to
// memory, and left to itself the compiler loads an argument where it is first used: seven such waits, one behind the other, in front of a program's
// first weights. As inputs of one empty statement (which needs them in registers) every scalar and a word of every line of the members are asked for at
// once, and then the program's member whole, out of the cache that now holds it. 0.4 us a launch (nothing in launches of few arguments, the
// rotations): a decode layer of the 5120 / 17408 model at 1 row 69.7 -> 68.5 us, of 7 rows at 5 bits 97.0 -> 94.4, of 40 rows 113.1 -> 109.2; 1024 /
// 2816 at 1 row (three launches) 27.9 -> 26.7.
#define GEMV_JOB_LINES(job)                                                                                                              \
    "s"((job).count), "s"((job).first[1]), "s"((job).first[2]), "s"((job).first[3]), "s"((job).first[4]), "s"((job).m[0].n), "s"((job).m[1].n), \
        "s"((job).m[2].trellis), "s"((job).m[2].n), "s"((job).m[3].n)
// the member that workgroup wg belongs to, and that member's first workgroup
__device__ __forceinline__ uint32_t gemv_member_of(const GemvJob& job, uint32_t wg, uint32_t& first) {
    uint32_t i = 0;
    first = 0;
#pragma unroll
    for (uint32_t j = 1; j < FE_EXL3_GROUP_MAX; j++)
        if (j < job.count && wg >= job.first[j]) i = j, first = job.first[j];
    return i;
}
__device__ __forceinline__ void gemv_member_now(const GemvMember& mb) {
    asm volatile("" ::"s"(mb.trellis), "s"(mb.svh), "s"(mb.suh), "s"(mb.xh), "s"(mb.y), "s"(mb.z), "s"(mb.counters), "s"(mb.n), "s"(mb.programs),
                 "s"(mb.stride_k), "s"(mb.stride_nb), "s"(mb.base), "s"(mb.rem), "s"(mb.inv_base), "s"(mb.inv_base1));
}

// x / d for x < 2^31 with inv = floor((2^32 - 1) / d): a multiply-high and one correction (uniform operands: scalar code).
__device__ __forceinline__ uint32_t udiv_inv(uint32_t x, uint32_t d, uint32_t inv) {
    uint32_t q = __umulhi(x, inv);
    return q + ((q + 1) * d <= x ? 1u : 0u);
}

// The ring of load steps turned left by `phase` slots (phase < DEPTH), so that the oldest step in flight sits in slot 0
// again: one pass of moves whatever the phase.
template <int BITS, int DEPTH>
__device__ __forceinline__ void ring_turn(LaneWords<BITS> (&ring)[DEPTH], uint32_t phase) {
    static_assert(DEPTH == 4, "the turns below are written out for four slots");
    if (phase == 1) {
        LaneWords<BITS> t = ring[0];
        ring[0] = ring[1], ring[1] = ring[2], ring[2] = ring[3], ring[3] = t;
    } else if (phase == 2) {
        LaneWords<BITS> t0 = ring[0], t1 = ring[1];
        ring[0] = ring[2], ring[1] = ring[3], ring[2] = t0, ring[3] = t1;
    } else if (phase == 3) {
        LaneWords<BITS> t = ring[3];
        ring[3] = ring[2], ring[2] = ring[1], ring[1] = ring[0], ring[0] = t;
    }
}

// A lane's words of one load step through a buffer resource over the whole trellis: the lane's byte offsets (run, word
// before the run) are loop constants in vector registers and the step's position is a scalar offset, so walking the run
// costs no vector instructions; reads past the end of the trellis return zero instead of faulting. Streaming (nt) loads.
template <int BITS>
__device__ __forceinline__ LaneWords<BITS> load_lane_words_buf(__amdgpu_buffer_rsrc_t rs, uint32_t run_b, uint32_t prev_b,
                                                               uint32_t soff) {
    constexpr int NT = 2;
    LaneWords<BITS> r;
    (void)prev_b;
    r.w[0] = 0;  // the word before the run comes from the neighbouring lane when the step is decoded (lane_prev_word)
    if constexpr (BITS == 1) {
        r.w[1] = __builtin_amdgcn_raw_buffer_load_b32(rs, run_b, soff, NT);
    } else if constexpr (BITS == 2) {
        u32x2 t = __builtin_amdgcn_raw_buffer_load_b64(rs, run_b, soff, NT);
        r.w[1] = t[0], r.w[2] = t[1];
    } else if constexpr (BITS == 3) {
        u32x3 t = __builtin_amdgcn_raw_buffer_load_b96(rs, run_b, soff, NT);
        r.w[1] = t[0], r.w[2] = t[1], r.w[3] = t[2];
    } else {
        u32x4 t = __builtin_amdgcn_raw_buffer_load_b128(rs, run_b, soff, NT);
        r.w[1] = t[0], r.w[2] = t[1], r.w[3] = t[2], r.w[4] = t[3];
        if constexpr (BITS == 5) {
            r.w[5] = __builtin_amdgcn_raw_buffer_load_b32(rs, run_b + 16, soff, NT);
        } else if constexpr (BITS == 6) {
            u32x2 u = __builtin_amdgcn_raw_buffer_load_b64(rs, run_b + 16, soff, NT);
            r.w[5] = u[0], r.w[6] = u[1];
        } else if constexpr (BITS == 7) {
            u32x3 u = __builtin_amdgcn_raw_buffer_load_b96(rs, run_b + 16, soff, NT);
            r.w[5] = u[0], r.w[6] = u[1], r.w[7] = u[2];
        } else if constexpr (BITS == 8) {
            u32x4 u = __builtin_amdgcn_raw_buffer_load_b128(rs, run_b + 16, soff, NT);
            r.w[5] = u[0], r.w[6] = u[1], r.w[7] = u[2], r.w[8] = u[3];
        }
    }
    return r;
}


// Timeline of the decode GEMV (a build with -DFE_GEMV_STAMPS, never the shipped one): wavefront w of workgroup g leaves
// the 100 MHz wall clock at up to twelve points of its life at stamps[(4 g + w) * 12 + slot], u64, where stamps lies
// 128 KB into the rotated-input area of the launch's first member (single-row launches on a workspace of 64 rows).
#ifdef FE_GEMV_STAMPS
#define FE_STAMP(slot)                                                                                  \
    do {                                                                                                \
        if (stamp_at && (threadIdx.x & 63) == 0) stamp_at[slot] = __builtin_amdgcn_s_memrealtime();     \
    } while (0)
#else
#define FE_STAMP(slot) \
    do {               \
    } while (0)
#endif

// The decode MLP in one launch (exl3_mlp_b*): the front stage's programs (gate and up, CHAIN = 1) write their outputs
// through to memory and publish every finished column block; the programs of the down stage (CHAIN = 2), which follow
// them in the grid, request their first weights, wait for the blocks their channels need and rotate SwiGLU(gate, up)
// straight from the front stage's outputs. Workgroups are dispatched in grid order, so a waiting program only ever waits
// for programs that are already resident or done; the wait is bounded all the same (spin_limit polls, then the error
// word is set and the program goes on with what it finds, so every launch ends). state: [0] sequence number of the
// last completed launch, [1] error word, [2] finished column blocks of the down stage,
// [(1 + i * nbf + b) * FE_CHAIN_STRIDE] the ready word of front member i's block b = the sequence number of the launch
// that finished it. The down stage's last finisher advances [0]; nothing is cleared between launches, so a captured
// launch replays. Polls are trips to memory: with the ready words packed into a few cache lines the watchers crowd
// one memory channel and slow the front stage's own hand-offs down (56.5 us for the 27B-shaped MLP at 4 bits against
// 46.5 us with a word per 256 bytes and 50.9 us for the two launches), and polling more often than every half
// microsecond costs more than it finds out.
#ifndef FE_CHAIN_STRIDE
#define FE_CHAIN_STRIDE 64  // u32 words from one ready word to the next
#endif
#ifndef FE_CHAIN_SLEEP
#define FE_CHAIN_SLEEP 16  // s_sleep units (64 cycles each) between two polls of a waiting program
#endif
struct ChainCtx {
    uint32_t* state;
    uint32_t* ready;  // front stage: this member's ready words; down stage: those of front members 0 (gate) and 1 (up)
    uint32_t nbf;     // column blocks of a front member = 128-channel blocks of the down stage's input
    uint32_t nb_down, spin_limit;
};
__device__ __forceinline__ uint32_t load_agent_u32(const uint32_t* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// FENCED: the hand-off written with the memory model's own means (plain stores, a release fence at agent scope, the
// arrival, an acquire fence, plain loads) instead of write-through stores and loads that pass the L2: the slow form
// (the release writes the whole L2 back), kept as a cross-check of the fast one (option "handoff_fenced").
template <int BITS, int CHAIN = 0, bool FENCED = false>
__device__ __forceinline__ void gemvb_body(const GemvMember mb, uint32_t p0, uint32_t np, uint32_t k, uint32_t m, uint32_t y_mode,
                                           uint32_t chunk, uint32_t inv_spb, const RotSrc src, uint16_t* stamp_base,
                                           const ChainCtx ch = ChainCtx{}) {
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    __shared__ uint32_t last_flag;
    uint32_t chain_target = 0;  // this launch's sequence number
    if constexpr (CHAIN != 0) chain_target = load_agent_u32(ch.state) + 1;
#ifdef FE_GEMV_STAMPS
    unsigned long long* stamp_at =
        stamp_base && m == 1 ? (unsigned long long*)(stamp_base + 65536) + (size_t)(blockIdx.x * 4 + (threadIdx.x >> 6)) * 12 : nullptr;
    FE_STAMP(0);
#else
    (void)stamp_base;
#endif
    constexpr uint32_t tw = 8 * BITS;
    constexpr bool PAIRS = CHAIN == 1;  // (in the grouped launches: 0.2 us slower for one linear, 0.2 us faster for gate and up)
    constexpr int DEPTH = 4;  // load steps in flight per lane (5 and 6 measured 2..5 % slower, 8 10 %: 22.9 against 20.7 us)
    constexpr int GROUP = 8;  // steps of straight-line code per loop iteration (a multiple of DEPTH)
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint32_t r = lane & 15, g = lane >> 4, q = r >> 1, tau = r & 1;
    const uint32_t n = mb.n, spb = k / 64, upb = spb / 2;  // load steps, units a column block
    const uint32_t base = mb.base, rem = mb.rem;
    // This workgroup runs the programs p0 .. p0 + np - 1 of the partition one after the other. Their runs are contiguous, so
    // to the loads and the staging they are one run; where one program's run ends its sums are flushed as that program's
    // (its own slot in z, its own arrival), exactly as if it had been launched on its own: the same sums in the same
    // order, without a second start-up.
    auto run_start = [&](uint32_t q) { return q * base + (q < rem ? q : rem); };
    const uint32_t u0 = run_start(p0);
    const uint32_t S = 2 * (run_start(p0 + np) - u0);  // load steps of this workgroup's run
    if (S == 0) return;
    uint32_t pl = p0, lend = 2 * (run_start(p0 + 1) - u0);  // the program at work and the load step at which its run ends
    uint32_t nb = udiv_inv(2 * u0, spb, inv_spb), st = 2 * u0 - nb * spb;  // where the run stands: column block, load step
    const uint32_t nb_run0 = nb, st_run0 = st;

    float* red = (float*)lds;                                        // [m][GEMV_RED_PITCH] sums of a finished segment
    unsigned char* xs = (unsigned char*)(red + m * GEMV_RED_PITCH);  // [m][xpitch] rotated inputs of a chunk of the run
    const uint32_t xpitch = chunk * 128 + 16;

    const uint32_t lane_word = g * mb.stride_k + (2 * wave + tau) * tw;
    const uint32_t run_b = 4 * (lane_word + q * BITS), prev_b = 4 * (lane_word + (q * BITS + tw - 1) % tw);
    const uint32_t step_bytes = 16 * mb.stride_k;                     // 4 k steps
    const uint32_t wrap_bytes = 4 * mb.stride_nb - spb * step_bytes;  // from the end of a column block to the next (mod 2^32)
    const __amdgpu_buffer_rsrc_t trs =
        __builtin_amdgcn_make_buffer_rsrc((void*)mb.trellis, 0, (k / 16) * (n / 16) * tw * 4, 0x00020000);
    uint32_t snext = nb * mb.stride_nb * 4 + st * step_bytes;  // byte offset of the next load step to request

    const uint32_t xrow = (r < m ? r : m - 1) * xpitch + g * 32;
    f32x4 acc[2];
    acc[0] = acc[1] = (f32x4){0.f, 0.f, 0.f, 0.f};

    const uint32_t hw = tid >> 5, l32 = tid & 31;
    // Rotating here: (row, 128-channel block) pairs of a chunk go to the half wavefronts: half wavefront hw takes blocks hw,
    // hw + 8, ... of every row. The first pair's loads go out ahead of the trellis loads (loads return in order), so
    // that the rotation runs while the first trellis words are still on their way.
    // (CHAIN: always, and up to 8 rows only, mlp_chain_fits. Code for what never comes is not free: with it the kernel is 47 KB, which with the 23 KB
    // of the GEMV is more than the 64 KB of instructions that two CUs cache, and a layer's launches displace each other's: 5120 / 17408 at 4 bits, 1
    // row, two layers 134.6 -> 133.5 us, 1024 / 2816 26.11 -> 25.84.)
    const bool rotating = CHAIN != 0 || src.x != nullptr;
    struct RotAt {
        size_t at, xat;
        uint32_t c, off;
        bool keep;
    };
    auto rot_at = [&](uint32_t c0, uint32_t row, uint32_t b) {
        RotAt a;
        uint32_t gst = st_run0 + c0 + 2 * b, blk = 0;  // load step counted from the start of the run's first column block
        if (gst >= spb) gst -= spb, blk = 1;
        if (gst >= spb) blk += gst / spb, gst %= spb;
        a.c = gst * 64 + 4 * l32;
        a.at = (size_t)row * k + a.c;
        a.xat = (size_t)row * src.ld + a.c;
        a.off = row * xpitch + b * 256 + 8 * l32;
        a.keep = nb_run0 + blk == 0;  // column block 0 sees every channel: its programs leave xh behind
        return a;
    };
    RotRaw rot_raw = {};
    // (resources over gate and up for the down stage's agent-scope loads; unused otherwise)
    const __amdgpu_buffer_rsrc_t chain_gs = __builtin_amdgcn_make_buffer_rsrc((void*)src.x, 0, m * src.ld * 2, 0x00020000);
    const __amdgpu_buffer_rsrc_t chain_us = __builtin_amdgcn_make_buffer_rsrc((void*)src.x2, 0, m * src.ld * 2, 0x00020000);
    auto load_pair = [&](const RotAt& a) {
        if constexpr (CHAIN == 2)
            return rot_load_agent(chain_gs, chain_us, mb.suh, (uint32_t)a.xat, a.c);
        else
            return rot_load(src, mb.suh, a.xat, a.c);
    };
    const uint32_t rot_mode = CHAIN == 2 ? 2u : src.mode;
    if (rotating && CHAIN != 2) {
        const uint32_t nblk = (S < chunk ? S : chunk) / 2;
        if (hw < nblk) {
            RotAt a = rot_at(0, 0, hw);
            rot_raw = load_pair(a);
        }
    }
    // the output scales of this lane's four columns of the block the run stands in (for the program that finishes it)
    u32x2 sv = *(const u32x2*)(mb.svh + nb * 128 + 4 * l32);

    // refill cursor: the next load step to request
    uint32_t rj = 0, rst = st;
    auto issue = [&](LaneWords<BITS>& slot) {
        slot = load_lane_words_buf<BITS>(trs, run_b, prev_b, snext);
        if (rj + 1 < S) {  // past the end of the run the last step is requested again (and never used)
            rj++;
            snext += step_bytes;
            if (++rst == spb) rst = 0, snext += wrap_bytes;
        }
    };
    LaneWords<BITS> ring[DEPTH];  // indexed by constants only, so it stays in registers
#pragma unroll
    for (int j = 0; j < DEPTH; j++) issue(ring[j]);
    FE_STAMP(1);
    if constexpr (CHAIN == 2) {
        // Unit j of the run reads channels block (st_run0 / 2 + j) % upb of the input: lanes 0..31 of the workgroup's first
        // wavefront watch gate's ready words of the run's units, lanes 32..63 up's (the host keeps a run within 32 units);
        // the other wavefronts wait at the barrier, which costs no issue slots. A poll is a trip to memory; between polls
        // the wavefront sleeps, so that the watchers do not crowd the memory channel that holds the words.
        uint32_t chain_spins = 0;
        if (wave == 0) {
            const uint32_t units = S / 2, j = lane & 31;
            uint32_t kb = st_run0 / 2 + j;
            kb -= kb >= upb ? upb : 0;
            kb = kb >= upb ? kb % upb : kb;
            const uint32_t* rw = ch.ready + ((lane >> 5) * ch.nbf + kb) * FE_CHAIN_STRIDE;
            bool pending = true;
            for (uint32_t spins = 0; spins < ch.spin_limit; spins++, chain_spins++) {
                const uint32_t v = j < units ? load_agent_u32(rw) : chain_target;
                pending = __builtin_amdgcn_ballot_w64(v != chain_target) != 0;
                if (!pending) break;
                __builtin_amdgcn_s_sleep(FE_CHAIN_SLEEP);
            }
            if (pending && lane == 0) __hip_atomic_fetch_or(ch.state + 1, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        __syncthreads();
        FE_STAMP(9);
#ifdef FE_GEMV_STAMPS
        if (stamp_at && lane == 0) stamp_at[10] = chain_spins;
#endif
    }

    auto one = [&](LaneWords<BITS>& slot, uint32_t t) {  // t: load step within the staged chunk
        f16x8 op[2][2];
        // the inputs are asked for in front of the decode: behind it their way out of LDS holds the products up (with the word before a lane's run in one
        // instruction instead of five: a layer of 5120 / 17408 at 1 row 68.4 -> 67.5 us, 1024 / 2816 26.7 -> 26.3)
        const unsigned char* xp = xs + xrow + t * 128;
        const f16x8 x0 = *(const f16x8*)xp, x1 = *(const f16x8*)(xp + 16);
        slot.w[0] = lane_prev_word(slot.w[BITS]);
        decode_lane<BITS>(slot, op);
        issue(slot);
        // keep the refill where it is issued: left alone, the scheduler sinks the loads to the end of the group, right in
        // front of the wait for them
        __builtin_amdgcn_sched_barrier(0);
        acc[0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(op[0][0], x0, acc[0], 0, 0, 0);
        acc[1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(op[1][0], x0, acc[1], 0, 0, 0);
        acc[0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(op[0][1], x1, acc[0], 0, 0, 0);
        acc[1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(op[1][1], x1, acc[1], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
    };

    // H over the 128 sums of a row (4 a lane of a half wavefront), * svh / sqrt(128) with the prefetched scales, stored.
    auto finish = [&](float (&v)[4], uint32_t col0, uint32_t row) {
        fwht128_half_wave(v, l32);
        v[0] = v[0] * FE_HAD_SCALE * f16_bits_to_f32(sv[0] & 0xffff);
        v[1] = v[1] * FE_HAD_SCALE * f16_bits_to_f32(sv[0] >> 16);
        v[2] = v[2] * FE_HAD_SCALE * f16_bits_to_f32(sv[1] & 0xffff);
        v[3] = v[3] * FE_HAD_SCALE * f16_bits_to_f32(sv[1] >> 16);
        if constexpr (CHAIN == 1)  // bf16, written through: the down stage's programs read it in this launch
            store_agent_u32x2((uint16_t*)mb.y + (size_t)row * n + col0 + 4 * l32,
                              (u32x2){pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])});
        else
            store4(mb.y, y_mode, (size_t)row * n + col0 + 4 * l32, v);
    };
    // A column block is finished (all of the workgroup's threads come here). Front stage: once every lane's stores are
    // acknowledged, its ready word takes this launch's number. Down stage: the block is counted, and the last one
    // completes the launch.
    auto block_done = [&](uint32_t fnb) {
        if constexpr (CHAIN == 1) {
            agent_stores_wait();
            __syncthreads();
            if (tid == 0) __hip_atomic_store(ch.ready + fnb * FE_CHAIN_STRIDE, chain_target, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#ifdef FE_GEMV_STAMPS
            if (tid == 0 && stamp_at)
                ((unsigned long long*)(stamp_base + 65536))[16384 * 12 + (ch.ready - (ch.state + FE_CHAIN_STRIDE)) / FE_CHAIN_STRIDE + fnb] = __builtin_amdgcn_s_memrealtime();
#endif
        } else if constexpr (CHAIN == 2) {
            if (tid == 0) {
                const uint32_t old = __hip_atomic_fetch_add(ch.state + 2, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (old + 1 == ch.nb_down) {
                    __hip_atomic_store(ch.state + 2, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    __hip_atomic_store(ch.state, chain_target, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
            }
        }
        (void)fnb;
    };

    // The segment of column block fnb that ends here: its sums meet in LDS, and then either are the block's sums (the
    // block lies in this run alone) or go to z for the program that arrives last at the block.
    // PAIRS: where the workgroup also runs the other program of a pair in the same block, the first one's sums wait in LDS and leave
    // with the second's as one segment, which saves a hand-off in the middle of the run (the MLP of 5120 x 17408 in one launch, 1 / 4 rows, us: 3 bits
    // 45.0 / 51.8 -> 44.1 / 51.1, 4 bits 46.5 / 53.4 -> 45.8 / 52.6).
    uint32_t pending = 0;
    auto flush = [&](uint32_t fnb, uint32_t p, bool keep) {
        __syncthreads();  // the previous segment's readers are done with `red`
        // a lane's four sums of either half: columns 16 (g & 1) + 4 (g >> 1) + 8 h .. + 3 of the wavefront's 32
        acc[0] = lane_cols(acc[0]), acc[1] = lane_cols(acc[1]);
        float* rp = red + 32 * wave + 16 * (g & 1) + 4 * (g >> 1);
        if (r < m) {  // accumulator column = input row
            f32x4 *r0 = (f32x4*)(rp + r * GEMV_RED_PITCH), *r1 = (f32x4*)(rp + r * GEMV_RED_PITCH + 8);
            if (PAIRS && pending) acc[0] = *r0 + acc[0], acc[1] = *r1 + acc[1];
            *r0 = acc[0], *r1 = acc[1];
        }
        acc[0] = acc[1] = (f32x4){0.f, 0.f, 0.f, 0.f};
        if (PAIRS && keep) {
            pending = 1;
            return;
        }
        const uint32_t two = PAIRS ? pending : 0;  // the segment is that of programs p - 1 and p
        pending = 0;
        __syncthreads();
        FE_STAMP(4);
        const uint32_t col0 = fnb * 128;
        // programs of the block's first and last unit
        const uint32_t cut = rem * (base + 1), ua = fnb * upb, ub = ua + upb - 1;
        const uint32_t first_prog = ua < cut ? udiv_inv(ua, base + 1, mb.inv_base1) : rem + udiv_inv(ua - cut, base, mb.inv_base);
        const uint32_t last_prog = ub < cut ? udiv_inv(ub, base + 1, mb.inv_base1) : rem + udiv_inv(ub - cut, base, mb.inv_base);
        if (first_prog + two == last_prog) {
            for (uint32_t row = hw; row < m; row += 8) {
                f32x4 t = *(const f32x4*)(red + row * GEMV_RED_PITCH + 4 * l32);
                float v[4] = {t[0], t[1], t[2], t[3]};
                finish(v, col0, row);
            }
            block_done(fnb);
            return;
        }
        // Hand-off of the segment's sums to another program, possibly on another XCD with its own L2:
        //  1. every lane stores its piece with agent-scope (write-through) stores and waits until they are acknowledged;
        //  2. the workgroup barrier orders all lanes' acknowledged stores before lane 0's arrival at the counter
        //     (an agent-scope atomic, performed at the shared level);
        //  3. the program whose arrival completes the count reads the segments with agent-scope loads (past its own L2)
        //     after the barrier that publishes last_flag.
        // Every byte that crosses is written through and read through, so no cache write-back or invalidate is needed.
        float* zseg = mb.z + (size_t)(p - two + fnb) * m * 128;
        if constexpr (FENCED) {
            for (uint32_t row = hw; row < m; row += 8)
                *(f32x4*)(zseg + row * 128 + 4 * l32) = *(const f32x4*)(red + row * GEMV_RED_PITCH + 4 * l32);
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
        } else {
            for (uint32_t row = hw; row < m; row += 8)
                store_agent_f32x4(zseg + row * 128 + 4 * l32, *(const f32x4*)(red + row * GEMV_RED_PITCH + 4 * l32));
            if (PAIRS && two)
                for (uint32_t row = hw; row < m; row += 8) store_agent_f32x4(zseg + (m + row) * 128 + 4 * l32, (f32x4){0.f, 0.f, 0.f, 0.f});
            agent_stores_wait();
        }
        FE_STAMP(5);
        __syncthreads();
        if (tid == 0) {
            uint32_t old = __hip_atomic_fetch_add(&mb.counters[fnb], 1u + two, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            last_flag = (old + two == last_prog - first_prog);
        }
        __syncthreads();
        FE_STAMP(6);
        if (last_flag) {
            if constexpr (FENCED) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
            // A half wavefront finishes rows hw, hw + 8, ...: RB of them at a time with SB segments each, 8 or 12 agent-scope
            // loads in flight (each takes a trip to memory: the trips overlap); every row's segments are added pair by pair, in
            // program order (as many in flight as the registers hold without costing the kernel a resident wavefront). Up to 8 rows
            // every half wavefront has at most one row and takes all of the batch from it. An odd first program is the second of its
            // pair: slot 0 is then where its partner, which has no part in this block, would leave its sums, and counts as zero. (What lies
            // past the last segment reads zero, so the sums need no conditions: 5120 x 5120 at 1 / 4 rows 10.9 / 12.7 -> 10.7 / 12.3 us.)
            const uint32_t odd = first_prog & 1, slots = last_prog - first_prog + 1 + odd;
            const __amdgpu_buffer_rsrc_t zrs = __builtin_amdgcn_make_buffer_rsrc(
                (void*)(mb.z + (size_t)(first_prog - odd + fnb) * m * 128), 0, slots * m * 512, 0x00020000);
            auto rows_of = [&](auto rb_tag) {
                constexpr int RB = decltype(rb_tag)::value, SB = (BITS <= 4 ? 12 : 8) / RB;
                for (uint32_t row0 = hw; row0 < m; row0 += 8 * RB) {
                    float v[RB][4];
#pragma unroll
                    for (int j = 0; j < RB; j++) v[j][0] = v[j][1] = v[j][2] = v[j][3] = 0.f;
                    for (uint32_t sp0 = 0; sp0 < slots; sp0 += SB) {
                        f32x4 t[RB * SB];
#pragma unroll
                        for (int j = 0; j < RB; j++) {
                            const uint32_t row = row0 + 8 * j < m ? row0 + 8 * j : row0;
#pragma unroll
                            for (int b = 0; b < SB; b++)  // (past the last segment: out of the buffer's range, reads zero)
                                t[j * SB + b] = FENCED ? __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                                             zrs, row * 512 + 16 * l32, (sp0 + b) * m * 512, 0))
                                                       : load_agent_f32x4(zrs, row * 512 + 16 * l32, (sp0 + b) * m * 512);
                            if (odd > sp0) t[j * SB] = (f32x4){0.f, 0.f, 0.f, 0.f};
                        }
#pragma unroll
                        for (int j = 0; j < RB; j++)
#pragma unroll
                            for (int b = 0; b < SB; b += 2)
#pragma unroll
                                for (int e = 0; e < 4; e++) v[j][e] += t[j * SB + b][e] + t[j * SB + b + 1][e];
                    }
#pragma unroll
                    for (int j = 0; j < RB; j++) {
                        const uint32_t row = row0 + 8 * j;
                        if (row < m) finish(v[j], col0, row);
                    }
                }
            };
            if (CHAIN != 0 || m <= 8)
                rows_of(std::integral_constant<int, 1>{});
            else
                rows_of(std::integral_constant<int, 2>{});
            if (tid == 0) __hip_atomic_store(&mb.counters[fnb], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            block_done(fnb);
            FE_STAMP(7);
        }
    };

    for (uint32_t c0 = 0; c0 < S; c0 += chunk) {
        const uint32_t cs = S - c0 < chunk ? S - c0 : chunk;
        if (c0) __syncthreads();  // the previous chunk's readers are done with xs
        if (rotating) {
            const uint32_t nblk = cs / 2;
            uint32_t row = 0, b = hw;
            RotAt a = {};
            const bool any = b < nblk;
            if (any) {
                a = rot_at(c0, row, b);
                if (c0 || CHAIN == 2) rot_raw = load_pair(a);
            }
            while (any && row < m) {
                u32x2 o = rot_finish(rot_raw, rot_mode, l32);
                *(u32x2*)(xs + a.off) = o;
                if (a.keep && mb.xh) *(u32x2*)(mb.xh + a.at) = o;
                b += 8;
                if (b >= nblk) b = hw, row++;
                if (row < m) {
                    a = rot_at(c0, row, b);
                    rot_raw = load_pair(a);
                }
            }
        } else {  // rotated inputs of the chunk's load steps -> xs [row][cs * 64 fp16], NB 16-byte pieces in flight a thread
            constexpr int NB = FE_STAGE_NB1;
            const uint32_t chunks16 = cs * 8, total = m * chunks16, inv16 = 0xffffffffu / chunks16;
            for (uint32_t i0 = tid; i0 < total; i0 += 256 * NB) {
                u32x4 v[NB];
                uint32_t off[NB];
#pragma unroll
                for (int j = 0; j < NB; j++) {
                    const uint32_t i = i0 + 256 * j < total ? i0 + 256 * j : i0;  // past the end: a piece again, not stored
                    const uint32_t row = udiv_inv(i, chunks16, inv16), c = i - row * chunks16;
                    uint32_t gst = st_run0 + c0 + (c >> 3);
                    if (gst >= spb) gst -= spb;
                    if (gst >= spb) gst %= spb;
                    v[j] = *(const u32x4*)(mb.xh + (size_t)row * k + gst * 64 + (c & 7) * 8);
                    off[j] = row * xpitch + c * 16;
                }
#pragma unroll
                for (int j = 0; j < NB; j++)
                    if (i0 + 256 * j < total) *(u32x4*)(xs + off[j]) = v[j];
            }
        }
        __syncthreads();
        FE_STAMP(2);
        // the chunk's load steps, segment by segment (a segment ends with its column block, with the chunk ...
        uint32_t i = 0;
        while (i < cs) {
            uint32_t seg = cs - i < spb - st ? cs - i : spb - st;
            seg = seg < lend - (c0 + i) ? seg : lend - (c0 + i);  // ... or with the program's run
            // Whole groups of GROUP steps run as straight-line code: no branches inside, and the refill of a ring slot is
            // unconditional, so each load lands straight in the slot its words were just decoded from and only that
            // slot's next use waits for it. The wait at the top of a group has to cover every load in flight (the
            // compiler cannot count across the back edge).
            const uint32_t full = seg / GROUP * GROUP;
            for (uint32_t s0 = 0; s0 < full; s0 += GROUP) {
#pragma unroll
                for (int j = 0; j < GROUP; j++) one(ring[j % DEPTH], i + s0 + j);
            }
            for (uint32_t s0 = full; s0 < seg; s0 += DEPTH) {  // the remainder, slot by slot
#pragma unroll
                for (int j = 0; j < DEPTH; j++)
                    if (s0 + j < seg) one(ring[j], i + s0 + j);
            }
            ring_turn<BITS, DEPTH>(ring, seg % DEPTH);
            FE_STAMP(3);
            i += seg, st += seg;
            const bool block_end = st == spb, run_end = c0 + i == lend;
            if (block_end || run_end) {
                flush(nb, pl, PAIRS && !block_end && !(pl & 1) && pl + 1 < p0 + np);
                if (block_end) {
                    nb++, st = 0;
                    if (c0 + i < S) sv = *(const u32x2*)(mb.svh + nb * 128 + 4 * l32);  // the next block's output scales
                }
                if (run_end) pl++, lend = 2 * (run_start(pl + 1) - u0);
            }
        }
    }
    FE_STAMP(8);
}

// (second launch bound: wavefronts per SIMD the registers must allow: four programs a CU)
#define GEMVB_KERNEL(NAME, BITS, FENCED)                                                                          \
    extern "C" __global__ __launch_bounds__(256, 4) void NAME(                                                        \
        GemvJob job, const void* x, const void* x2, uint32_t x_mode, uint32_t ldx, uint32_t k, uint32_t m,             \
        uint32_t y_mode, uint32_t chunk, uint32_t inv_spb, uint32_t fuse) {                                            \
        asm volatile("" ::GEMV_JOB_LINES(job), "s"(x), "s"(x2), "s"(x_mode), "s"(ldx), "s"(k), "s"(m), "s"(y_mode), "s"(chunk), "s"(inv_spb), "s"(fuse)); \
        uint32_t first;                                                                                               \
        const GemvMember mb = job.m[gemv_member_of(job, blockIdx.x, first)];                                          \
        gemv_member_now(mb);                                                                                          \
        const uint32_t p0 = (blockIdx.x - first) * fuse;                                                              \
        const uint32_t left = mb.programs - p0;                                                                       \
        gemvb_body<BITS, 0, FENCED>(mb, p0, left < fuse ? left : fuse, k, m, y_mode, chunk, inv_spb,                  \
                                    RotSrc{x, x2, x_mode, ldx}, job.m[0].xh);                                         \
    }
#define GEMVB_FAMILY(BITS) GEMVB_KERNEL(exl3_gemvb_b##BITS##_r1, BITS, false) GEMVB_KERNEL(exl3_gemvb_b##BITS##_r1_fenced, BITS, true)

// The decode MLP in one launch, 1..16 rows: grid = the front stage's workgroups (gate and up, alternating when their
// counts are equal, so that block b of both is finished at about the same time), then the down stage's. Down workgroup
// w runs program perm[w] (the host's table: the programs sorted by the last channel block their run reads, so that they
// come in the order in which the front stage finishes their inputs; null: program w).
struct MlpChain {
    GemvJob front;
    GemvMember down;
    uint32_t* state;
    const uint32_t* perm;
    uint32_t front_wgs, interleave;
    uint32_t k1, chunk1, inv_spb1, fuse1;
    uint32_t k2, chunk2, inv_spb2, fuse2;
    uint32_t spin_limit, pad;
};
#define MLP_KERNEL(BITS)                                                                                              \
    extern "C" __global__ __launch_bounds__(256, 4) void exl3_mlp_b##BITS(MlpChain c, const void* x, uint32_t x_mode,  \
                                                                          uint32_t ldx, uint32_t m, uint32_t y_mode) { \
        asm volatile("" ::"s"(c.front.count), "s"(c.front.first[1]), "s"(c.front.m[0].n), "s"(c.front.m[1].trellis), "s"(c.front.m[1].n),        \
                     "s"(c.front.m[1].inv_base1), "s"(c.down.trellis), "s"(c.down.n), "s"(c.state), "s"(c.perm), "s"(c.front_wgs), "s"(c.interleave), \
                     "s"(c.k1), "s"(c.chunk1), "s"(c.inv_spb1), "s"(c.fuse1), "s"(c.k2), "s"(c.chunk2), "s"(c.inv_spb2), "s"(c.fuse2),   \
                     "s"(c.spin_limit), "s"(x), "s"(x_mode), "s"(ldx), "s"(m), "s"(y_mode));                                          \
        const uint32_t w = blockIdx.x, nbf = c.front.m[0].n / 128, nbd = c.down.n / 128;                              \
        if (w < c.front_wgs) {                                                                                        \
            const uint32_t i = c.interleave ? w & 1 : c.front.count > 1 && w >= c.front.first[1];                     \
            const uint32_t lw = c.interleave ? w >> 1 : i ? w - c.front.first[1] : w;                                 \
            const GemvMember mb = c.front.m[i];                                                                       \
            gemv_member_now(mb);                                                                                      \
            const uint32_t p0 = lw * c.fuse1, left = mb.programs - p0;                                                \
            gemvb_body<BITS, 1>(mb, p0, left < c.fuse1 ? left : c.fuse1, c.k1, m, 0, c.chunk1, c.inv_spb1,            \
                                   RotSrc{x, nullptr, x_mode, ldx}, c.front.m[0].xh,                                  \
                                   ChainCtx{c.state, c.state + (1 + i * nbf) * FE_CHAIN_STRIDE, nbf, nbd, c.spin_limit}); \
        } else {                                                                                                      \
            uint32_t lw = w - c.front_wgs;                                                                            \
            if (c.perm) lw = c.perm[lw];                                                                              \
            const GemvMember mb = c.down;                                                                             \
            gemv_member_now(mb);                                                                                      \
            const uint32_t p0 = lw * c.fuse2, left = mb.programs - p0;                                                \
            gemvb_body<BITS, 2>(mb, p0, left < c.fuse2 ? left : c.fuse2, c.k2, m, y_mode, c.chunk2, c.inv_spb2,       \
                                   RotSrc{c.front.m[0].y, c.front.m[1].y, 2, c.front.m[0].n}, c.front.m[0].xh,        \
                                   ChainCtx{c.state, c.state + FE_CHAIN_STRIDE, nbf, nbd, c.spin_limit});             \
        }                                                                                                             \
    }
MLP_KERNEL(2)
MLP_KERNEL(3)
MLP_KERNEL(4)
MLP_KERNEL(5)
MLP_KERNEL(6)
MLP_KERNEL(8)
GEMVB_FAMILY(2)
GEMVB_FAMILY(3)
GEMVB_FAMILY(4)
GEMVB_FAMILY(5)
GEMVB_FAMILY(6)
GEMVB_FAMILY(8)

// ---- the same GEMV for more rows ------------------------------------------------------------------------------------------
//
// 17..64 rows, and gate and up of an MLP block from 9 rows on. The programs, their runs, the order of every sum and so the bits are gemvb_body's. With PER 2 a
// workgroup runs the programs 2 j and 2 j + 1 as one: where the first's run ends inside a column block its sums step aside, and are
// added to the second's before they leave as one segment, as the finisher of gemvb_body adds them. What differs is how a program
// gets its operands and hands its sums over: both grow with the rows while the decode does not. The rotated inputs and the trellis words of a
// load step go straight from memory into LDS, DEPTH - 1 steps ahead. Every segment's sums go to z as the accumulators hold them, whole
// wavefronts at a time, and a launch behind this one (exl3_gemvw_finish*) adds and finishes them with all CUs, unless the host has the programs finish
// the column blocks that lie in one run (wide_end). (In gemvb_body's hand-off the
// program that arrives last at a block reads its segments alone, 12 loads in flight: at 40 rows and 4 bits 10.4 of 22.2 us for q + k + v of the
// 5120 / 17408 layer, 8.0 of 17.6 for o, 7.6 of 42.8 for gate and up, 14.2 of 34.9 for down; now 13.7 + 4.6, 11.3 + 4.7, 36.4 + 6.1, 21.8 + 5, and the launch
// behind gate and up leaves down's rotated input as well, which took a launch of 5 us.) A layer at 17 / 40 / 64 rows 107 / 138 / 173 -> 99 / 116 /
// 140 us. Written through
// (a plain store leaves the launch's end to write 14 MB back: 1 to 2 us more). Registers stay under 128, so that four programs share a
// CU. Bound by the decode and each program's start and end: at 40 rows and 4 bits gate and up issue vector instructions for 20 us, 70 % of the time
// between the first wavefront and the last, in a launch of 37 (matrix pipe busy in 23 %, LDS bank conflicts 12 % of the cycles). Decoding the next
// step between the products of this one was measured and changes nothing.
template <int BITS, int RG>
struct GemvWide {
    static constexpr int X_STAGE = RG * 2048, W_STAGE = 1024 * BITS;
    static constexpr int DEPTH = 4 * (X_STAGE + W_STAGE) <= 40 * 1024 ? 4 : 3;  // (so that four programs fit a CU, up to 5 bits)
    static constexpr int W_AT = DEPTH * X_STAGE;
    static constexpr int LX = (2 * RG + 3) / 4, LW = (BITS + 3) / 4;  // loads a wavefront issues a step: 1 KB pieces, some twice
    static_assert(16 * RG * GEMV_RED_PITCH * 4 <= DEPTH * (X_STAGE + W_STAGE), "a finished block's sums take the stages' place");
};
// ENDS: a column block that lies in one run is finished here, from LDS: its sums would travel to memory and back for nothing. (Kernels of their own: beside
// the code for it the loop takes 1 % longer, decode of 40 rows.)
template <int BITS, int RG, int PER, bool ENDS>
__device__ __forceinline__ void gemv_wide_body(const GemvMember mb, uint32_t p, uint32_t k, uint32_t m, uint32_t y_mode) {
    typedef GemvWide<BITS, RG> C;
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t r = lane & 15, g = lane >> 4;
    const uint32_t n = mb.n, upb = k / 128, base = mb.base, rem = mb.rem;
    const u32x4 xrs = g8_rsrc(mb.xh, m * k * 2), wrs = g8_rsrc(mb.trellis, (k / 16) * (n / 16) * 32 * BITS);
    const uint32_t step_bytes = 16 * mb.stride_k, lds0 = g8_lds_addr(lds);
    uint32_t vx[C::LX], vw[C::LW];
#pragma unroll
    for (int j = 0; j < C::LX; j++) {  // piece: 8 rows x 64 channels; 16-byte chunk c of a row at position c ^ (row & 7)
        const uint32_t row = (wave + 4 * j) % (2 * RG) * 8 + (lane >> 3);
        vx[j] = ((row < m ? row : m - 1) * k + ((lane & 7) ^ (row & 7)) * 8) * 2;
    }
#pragma unroll
    for (int j = 0; j < C::LW; j++) {  // [4 k steps][8 tiles][8 BITS words]
        const uint32_t at = (wave + 4 * j) % BITS * 1024 + lane * 16;
        vw[j] = 4 * (at / (256 * BITS) * mb.stride_k) + at % (256 * BITS);
    }
    const unsigned char* xp = lds + r * 128;
    const uint32_t xo0 = ((2 * g) ^ (r & 7)) << 4, xo1 = ((2 * g + 1) ^ (r & 7)) << 4;
    const unsigned char* wp = lds + C::W_AT + (g * 8 + 2 * wave + (r >> 3)) * (32 * BITS) + (r & 7) * (4 * BITS);

    f32x4 acc[RG][2];
    // Rows 16 rg .. of the accumulators lie in z one after the other: of each half h, wavefront and g 4 columns of the rows that exist.
    auto zoff = [&](int rg, int h) {
        const uint32_t mr = m - 16 * rg < 16 ? m - 16 * rg : 16;
        return (uint32_t)(16 * rg) * 512 + ((h * 16 + wave * 4 + g) * mr + r) * 16;
    };
    auto run_start = [&](uint32_t q) { return q * base + (q < rem ? q : rem); };
    uint32_t u = run_start(PER * p);
    const uint32_t uend = run_start(PER * p + PER < mb.programs ? PER * p + PER : mb.programs), mid = run_start(PER * p + 1);
    while (u < uend) {
        // A step's offsets and stages are running scalars: the quotient comes from the vector unit, and left there it takes the loads' offsets, a
        // 32-bit multiply among them, and the stages along, 133..139 vector instructions a step where the decode takes 119; 123 so. A layer of 5120 /
        // 17408 again and again, 17 / 32 / 40 / 64 rows at 3 bits 88.6 / 92.9 / 101.5 / 118.3 -> 83.7 / 87.9 / 99.2 / 116.5 us, at 4 bits 87.2 / 91.4
        // / 101.6 / 120.9 -> 84.8 / 88.7 / 99.8 / 117.4, 9 rows 86.6 -> 84.2; three layers in turn, whose weights no cache holds: 94.8 / 98.0 / 106.6
        // / 125.6 -> 90.1 / 93.4 / 104.2 / 124.0, 94.8 / 98.6 / 108.0 / 130.0 -> 93.4 / 96.0 / 106.3 / 125.4, 88.2 -> 86.8.
        const uint32_t nb = __builtin_amdgcn_readfirstlane(u / upb), in = u - nb * upb, units = uend - u < upb - in ? uend - u : upb - in, steps = 2 * units;
        const uint32_t aside = mid > u && mid < u + units ? 2 * (mid - u) : steps;  // the step at which the second program's run starts
        u += units;
        uint32_t w_at = nb * mb.stride_nb * 4 + 2 * in * step_bytes, x_at = 2 * in * 128, left = steps;  // the next step to ask for
        auto issue = [&](uint32_t x_to, uint32_t w_to) {
#pragma unroll
            for (int j = 0; j < C::LX; j++) g8_load_lds16(xrs, x_to + (wave + 4 * j) % (2 * RG) * 1024, vx[j], x_at);
#pragma unroll
            for (int j = 0; j < C::LW; j++) g8_load_lds16(wrs, w_to + (wave + 4 * j) % BITS * 1024, vw[j], w_at);
            const bool more = --left != 0;  // past the end: the last step again, never used
            x_at += more ? 128 : 0, w_at += more ? step_bytes : 0, left += more ? 0 : 1;
        };
#pragma unroll
        for (int s = 0; s < C::DEPTH - 1; s++) issue(lds0 + s * C::X_STAGE, lds0 + C::W_AT + s * C::W_STAGE);
#pragma unroll
        for (int rg = 0; rg < RG; rg++) acc[rg][0] = acc[rg][1] = (f32x4){0.f, 0.f, 0.f, 0.f};
        uint32_t slot = 0, to = C::DEPTH - 1;  // the stage of this step, the one that is free
        auto step = [&]() {
            g8_loads_wait<(C::DEPTH - 2) * (C::LX + C::LW)>();
            g8_barrier();
            issue(lds0 + to * C::X_STAGE, lds0 + C::W_AT + to * C::W_STAGE);
            LaneWords<BITS> lw;
            const uint32_t* words = (const uint32_t*)(wp + slot * C::W_STAGE);
            if constexpr (BITS % 4 == 0) {
#pragma unroll
                for (int i = 0; i < BITS; i += 4) {
                    const u32x4 t = *(const u32x4*)(words + i);
                    lw.w[i + 1] = t[0], lw.w[i + 2] = t[1], lw.w[i + 3] = t[2], lw.w[i + 4] = t[3];
                }
            } else {
#pragma unroll
                for (int i = 0; i < BITS; i++) lw.w[i + 1] = words[i];
            }
            lw.w[0] = lane_prev_word_halves(lw.w[BITS]);
            f16x8 op[2][2];
            decode_lane<BITS>(lw, op);
            const unsigned char* xs = xp + slot * C::X_STAGE;
#pragma unroll
            for (int rg = 0; rg < RG; rg++) {
                const f16x8 b0 = *(const f16x8*)(xs + rg * 2048 + xo0), b1 = *(const f16x8*)(xs + rg * 2048 + xo1);
                acc[rg][0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(op[0][0], b0, acc[rg][0], 0, 0, 0);
                acc[rg][1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(op[1][0], b0, acc[rg][1], 0, 0, 0);
                acc[rg][0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(op[0][1], b1, acc[rg][0], 0, 0, 0);
                acc[rg][1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(op[1][1], b1, acc[rg][1], 0, 0, 0);
            }
            to = slot, slot = slot + 1 == C::DEPTH ? 0 : slot + 1;
        };
        if constexpr (PER == 1) {
            for (uint32_t s = 0; s < steps; s++) step();
        } else {
            f32x4 hold[RG][2] = {};
            uint32_t s = 0, stop = aside;
            for (;;) {
                do step();
                while (++s < stop);
                if (s == steps) break;
#pragma unroll
                for (int rg = 0; rg < RG; rg++) {
                    hold[rg][0] = acc[rg][0], hold[rg][1] = acc[rg][1];
                    acc[rg][0] = acc[rg][1] = (f32x4){0.f, 0.f, 0.f, 0.f};
                }
                stop = steps;
            }
            if (aside != steps) {
#pragma unroll
                for (int rg = 0; rg < RG; rg++) acc[rg][0] = hold[rg][0] + acc[rg][0], acc[rg][1] = hold[rg][1] + acc[rg][1];
            }
        }
        if (ENDS && units == upb) {
            g8_loads_wait<0>();  // (the repeated last steps' too)
            g8_barrier();        // the stages are free for the sums, rows of GEMV_RED_PITCH
            float* red = (float*)lds + 32 * wave + 16 * (g >> 1) + 4 * (g & 1);
#pragma unroll
            for (int rg = 0; rg < RG; rg++)
#pragma unroll
                for (int h = 0; h < 2; h++) *(f32x4*)(red + (16 * rg + r) * GEMV_RED_PITCH + 8 * h) = acc[rg][h];
            __syncthreads();
            const uint32_t l32 = tid & 31, col = nb * 128 + 4 * l32;
            for (uint32_t row = tid >> 5; row < m; row += 8) {
                const f32x4 t = *(const f32x4*)((const float*)lds + row * GEMV_RED_PITCH + 4 * l32);
                float v[4] = {t[0], t[1], t[2], t[3]};
                finish_row(v, l32, mb.svh, col, mb.y, y_mode, (size_t)row * n + col);
            }
            __syncthreads();
            continue;
        }
        unsigned char* zseg = (unsigned char*)(mb.z + (size_t)(p + nb) * m * 128);
#pragma unroll
        for (int rg = 0; rg < RG; rg++) asm volatile("" : "+v"(acc[rg][0]), "+v"(acc[rg][1]));
        asm volatile("s_nop 15\n\ts_nop 3");  // the last product's wait states, which the compiler does not know of in front of stores in inline assembly
#pragma unroll
        for (int rg = 0; rg < RG; rg++)
            if (16 * rg + r < m) {
                store_agent_f32x4((float*)(zseg + zoff(rg, 0)), acc[rg][0]);
                store_agent_f32x4((float*)(zseg + zoff(rg, 1)), acc[rg][1]);
            }
        g8_loads_wait<2 * RG>();  // the repeated last steps (the stores, 2 RG of every wavefront, may be in flight)
        g8_barrier();             // the stages are free
    }
}
// The workgroups whose runs have part in a column block: first .. last (PER programs each).
struct WideSpan {
    uint32_t first, last, odd;  // odd: PER 1, the first one is the second of its pair of programs
};
template <int PER>
__device__ __forceinline__ WideSpan wide_span(const GemvMember& mb, uint32_t nb, uint32_t upb) {
    const uint32_t base = mb.base, rem = mb.rem, cut = rem * (base + 1), ua = nb * upb, ub = ua + upb - 1;
    const uint32_t first = ua < cut ? udiv_inv(ua, base + 1, mb.inv_base1) : rem + udiv_inv(ua - cut, base, mb.inv_base);
    const uint32_t last = ub < cut ? udiv_inv(ub, base + 1, mb.inv_base1) : rem + udiv_inv(ub - cut, base, mb.inv_base);
    if constexpr (PER == 2) return {first >> 1, last >> 1, 0};
    return {first, last, first & 1};
}
// The sums of row `row`, column block nb: what gemv_wide_body's programs left of them, added in gemvb_body's order (programs 2 j and 2 j + 1 to
// each other, the pairs in order; PER 2: a segment is a pair's). A lane of the half wavefront gets columns 4 l32 .. + 3.
template <int PER>
__device__ __forceinline__ f32x4 wide_row_sums(const GemvMember& mb, uint32_t nb, const WideSpan& sp, uint32_t m, uint32_t row, uint32_t l32) {
    const uint32_t odd = sp.odd, slots = sp.last - sp.first + 1 + odd;
    const __amdgpu_buffer_rsrc_t zrs =
        __builtin_amdgcn_make_buffer_rsrc((void*)(mb.z + (size_t)(sp.first - odd + nb) * m * 128), 0, slots * m * 512, 0x00020000);
    // (zoff of gemv_wide_body: column 32 wave + 16 (g >> 1) + 8 h + 4 (g & 1))
    const uint32_t rg = row / 16, r = row % 16, mr = m - 16 * rg < 16 ? m - 16 * rg : 16, c = l32 & 7;
    const uint32_t piece = ((c >> 1) & 1) * 16 + (l32 >> 3) * 4 + 2 * (c >> 2) + (c & 1), at = 16 * rg * 512 + (piece * mr + r) * 16;
    constexpr uint32_t SB = 4;  // segments in flight a lane (8: 0.4 us slower, 18: 2 us at gate and up; a whole wave of rows hides the trips)
    f32x4 sum = {0.f, 0.f, 0.f, 0.f};
    for (uint32_t s0 = 0; s0 < slots; s0 += SB) {
        f32x4 t[SB];
#pragma unroll
        for (uint32_t b = 0; b < SB; b++)  // (past the last segment: out of range by the vector offset, reads zero)
            t[b] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(zrs, at + (s0 + b) * m * 512, 0, 0));
        if (PER == 1 && odd > s0) t[0] = (f32x4){0.f, 0.f, 0.f, 0.f};  // where the first segment's partner, which has no part in the block, would leave its sums
#pragma unroll
        for (uint32_t b = 0; b < SB; b += 2) {
            if constexpr (PER == 2)
                sum = sum + t[b] + t[b + 1];
            else
                sum += t[b] + t[b + 1];
        }
    }
    return sum;
}
// Finishes the outputs of a launch of gemv_wide_body: grid (column blocks of all members, ceil(m / 8)), 256 threads, a half wavefront a
// row. Bound by its one read of the segments, which other XCDs have just written (14 MB for down of 40 rows: 5 us). y_mode + WIDE_WHOLE: blocks
// that lie in one run are finished already.
#define WIDE_WHOLE 4u
template <int PER>
__device__ __forceinline__ void wide_finish_body(const GemvJob& job, uint32_t k, uint32_t m, uint32_t y_mode) {
    asm volatile("" ::GEMV_JOB_LINES(job), "s"(k), "s"(m), "s"(y_mode));
    const uint32_t l32 = threadIdx.x & 31, row = blockIdx.y * 8 + (threadIdx.x >> 5);
    uint32_t i = 0, nb = blockIdx.x, before = 0;
#pragma unroll
    for (uint32_t j = 1; j < FE_EXL3_GROUP_MAX; j++) {
        before += job.m[j - 1].n / 128;
        if (j < job.count && blockIdx.x >= before) i = j, nb = blockIdx.x - before;
    }
    const GemvMember mb = job.m[i];
    gemv_member_now(mb);
    const WideSpan sp = wide_span<PER>(mb, nb, k / 128);
    if (row >= m || ((y_mode & WIDE_WHOLE) && sp.first == sp.last)) return;
    const uint32_t col = nb * 128 + 4 * l32;
    const size_t at = (size_t)row * mb.n + col;
    const u32x2 sv = *(const u32x2*)(mb.svh + col);  // (these two on their way beside the segments)
    const u32x4 old = store4_old(mb.y, y_mode & 3, at);
    const f32x4 s = wide_row_sums<PER>(mb, nb, sp, m, row, l32);
    float v[4] = {s[0], s[1], s[2], s[3]};
    finish_row(v, l32, sv, mb.y, y_mode & 3, at, old);
}
// The same for gate and up in front of down: both outputs (bf16), and down's rotated input of SwiGLU(gate, up), a 128-channel block of which
// is a column block of the two. grid (column blocks of one of them, ceil(m / 8)).
template <int PER>
__device__ __forceinline__ void wide_finish_mlp_body(const GemvJob& job, uint32_t k, uint32_t m, const uint16_t* suh, uint16_t* xh) {
    const uint32_t l32 = threadIdx.x & 31, row = blockIdx.y * 8 + (threadIdx.x >> 5), nb = blockIdx.x, c = nb * 128 + 4 * l32, n = job.m[0].n;
    gemv_member_now(job.m[0]);
    if (row >= m) return;
    gemv_member_now(job.m[1]);
    RotRaw raw = {};
    raw.s = *(const u32x2*)(suh + c);
    const u32x2 svs[2] = {*(const u32x2*)(job.m[0].svh + c), *(const u32x2*)(job.m[1].svh + c)};  // (on their way beside the segments)
    u32x2 y[2];
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const f32x4 s = wide_row_sums<PER>(job.m[i], nb, wide_span<PER>(job.m[i], nb, k / 128), m, row, l32);
        float v[4] = {s[0], s[1], s[2], s[3]};
        fwht128_half_wave(v, l32);
        const u32x2 sv = svs[i];
        v[0] = v[0] * FE_HAD_SCALE * f16_bits_to_f32(sv[0] & 0xffff);  // finish_row's products
        v[1] = v[1] * FE_HAD_SCALE * f16_bits_to_f32(sv[0] >> 16);
        v[2] = v[2] * FE_HAD_SCALE * f16_bits_to_f32(sv[1] & 0xffff);
        v[3] = v[3] * FE_HAD_SCALE * f16_bits_to_f32(sv[1] >> 16);
        y[i] = (u32x2){pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
        *(u32x2*)((uint16_t*)job.m[i].y + (size_t)row * n + c) = y[i];
    }
    raw.xb = y[0], raw.ub = y[1];
    *(u32x2*)(xh + (size_t)row * n + c) = rot_finish(raw, 2, l32);
}
#define WIDE_FINISH_KERNELS(SUFFIX, PER)                                                                                         \
    extern "C" __global__ __launch_bounds__(256) void exl3_gemvw_finish##SUFFIX(GemvJob job, uint32_t k, uint32_t m, uint32_t y_mode) { \
        wide_finish_body<PER>(job, k, m, y_mode);                                                                                \
    }                                                                                                                            \
    extern "C" __global__ __launch_bounds__(256) void exl3_gemvw_finish_mlp##SUFFIX(GemvJob job, uint32_t k, uint32_t m,          \
                                                                                     const uint16_t* suh, uint16_t* xh) {         \
        wide_finish_mlp_body<PER>(job, k, m, suh, xh);                                                                           \
    }
WIDE_FINISH_KERNELS(, 1)
WIDE_FINISH_KERNELS(_pairs, 2)
#define GEMV_WIDE_KERNEL(NAME, BITS, RG, PER, ENDS)                                                                   \
    extern "C" __global__ __launch_bounds__(256, 4) void NAME(GemvJob job, uint32_t k, uint32_t m, uint32_t y_mode) { \
        asm volatile("" ::GEMV_JOB_LINES(job), "s"(k), "s"(m), "s"(y_mode));                                          \
        uint32_t first;                                                                                               \
        const GemvMember mb = job.m[gemv_member_of(job, blockIdx.x, first)];                                          \
        gemv_member_now(mb);                                                                                          \
        gemv_wide_body<BITS, RG, PER, ENDS>(mb, blockIdx.x - first, k, m, y_mode);                                    \
    }
#define GEMV_WIDE_ROWS(BITS, RG)                                    \
    GEMV_WIDE_KERNEL(exl3_gemvw_b##BITS##_r##RG, BITS, RG, 1, false)        \
    GEMV_WIDE_KERNEL(exl3_gemvw_b##BITS##_r##RG##_ends, BITS, RG, 1, true) \
    GEMV_WIDE_KERNEL(exl3_gemvw_b##BITS##_r##RG##_pairs, BITS, RG, 2, false) \
    GEMV_WIDE_KERNEL(exl3_gemvw_b##BITS##_r##RG##_pairs_ends, BITS, RG, 2, true)
#define GEMV_WIDE_FAMILY(BITS) GEMV_WIDE_ROWS(BITS, 1) GEMV_WIDE_ROWS(BITS, 2) GEMV_WIDE_ROWS(BITS, 3) GEMV_WIDE_ROWS(BITS, 4)
GEMV_WIDE_FAMILY(2)
GEMV_WIDE_FAMILY(3)
GEMV_WIDE_FAMILY(4)
GEMV_WIDE_FAMILY(5)
GEMV_WIDE_FAMILY(6)
GEMV_WIDE_FAMILY(8)

// ---- probes ----------------------------------------------------------------------------------------------------------

// Streaming read of `bytes` (a multiple of 16 * 256 * gridDim.x * unroll) with 16-byte loads; each thread xors what it
// read into one word of out so the loads stay. (kernels/k-exl3/src/probe.rs:7-36)
extern "C" __global__ __launch_bounds__(256) void exl3_probe_v4(const u32x4* in, uint32_t* out, uint64_t vec_count) {
    uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x, stride = (uint64_t)gridDim.x * 256;
    u32x4 a = {0, 0, 0, 0};
    for (; i + 3 * stride < vec_count; i += 4 * stride) {
        u32x4 v0 = __builtin_nontemporal_load(in + i), v1 = __builtin_nontemporal_load(in + i + stride);
        u32x4 v2 = __builtin_nontemporal_load(in + i + 2 * stride), v3 = __builtin_nontemporal_load(in + i + 3 * stride);
        a ^= v0 ^ v1 ^ v2 ^ v3;
    }
    for (; i < vec_count; i += stride) a ^= __builtin_nontemporal_load(in + i);
    uint32_t x = a[0] ^ a[1] ^ a[2] ^ a[3];
    if (x == 0x9e3779b9u) out[0] = x;  // practically never: keeps the loads alive without a store stream
}

// Decode-only probe: every lane decodes `iters` load steps of synthetic words and feeds them to the matrix instruction as
// the GEMV does (no memory traffic, no LDS): the ALU ceiling of the trellis decode in weights per second at the GEMV's
// occupancy (launch 4 programs a CU). The words change from step to step by additions that do not depend on the results,
// as words from memory would not. out receives a checksum.
template <int BITS>
__device__ __forceinline__ void probe_decode_body(uint32_t* out, uint32_t iters, uint32_t seed) {
    LaneWords<BITS> lw;
#pragma unroll
    for (int i = 0; i <= BITS; i++) lw.w[i] = (seed + i) * 0x9e3779b9u * (threadIdx.x + 1 + blockIdx.x * 256);
    f32x4 acc0 = {0.f, 0.f, 0.f, 0.f}, acc1 = {0.f, 0.f, 0.f, 0.f};
    const f16x8 xb = {1, 1, 1, 1, 1, 1, 1, 1};
    for (uint32_t it = 0; it < iters; it++) {
        f16x8 op[2][2];
        decode_lane<BITS>(lw, op);
        acc0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(op[0][0], xb, acc0, 0, 0, 0);
        acc1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(op[1][0], xb, acc1, 0, 0, 0);
        acc0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(op[0][1], xb, acc0, 0, 0, 0);
        acc1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(op[1][1], xb, acc1, 0, 0, 0);
#pragma unroll
        for (int i = 0; i <= BITS; i++) lw.w[i] += 0x9e3779b9u + i;
    }
    const float sum = acc0[0] + acc0[1] + acc0[2] + acc0[3] + acc1[0] + acc1[1] + acc1[2] + acc1[3];
    out[blockIdx.x * blockDim.x + threadIdx.x] = __float_as_uint(sum);
}
extern "C" __global__ __launch_bounds__(256, 4) void exl3_probe_decode_b3(uint32_t* out, uint32_t iters, uint32_t seed) {
    probe_decode_body<3>(out, iters, seed);
}
extern "C" __global__ __launch_bounds__(256, 4) void exl3_probe_decode_b4(uint32_t* out, uint32_t iters, uint32_t seed) {
    probe_decode_body<4>(out, iters, seed);
}
extern "C" __global__ __launch_bounds__(256, 4) void exl3_probe_decode_b5(uint32_t* out, uint32_t iters, uint32_t seed) {
    probe_decode_body<5>(out, iters, seed);
}

// Instruction throughput probes: 8 independent chains of `iters` dependent instructions a lane, no memory traffic
// (kernels/k-exl3/src/probe.rs:38-67 measures its decode's instructions the same way). The instructions are the ones the
// trellis decode is made of, plus an add and an and as the plain 32-bit yardsticks; the issue rate of an instruction is
// lanes x 8 x iters over the launch time. 128 of them between two branches, as in the decode's straight code: with 8 the
// branches took a tenth of the time (four wavefronts a SIMD: 4.75 cycles an instruction instead of 4.25).
#define OP_PROBE(NAME, ASM)                                                                                            \
    extern "C" __global__ __launch_bounds__(256) void exl3_probe_op_##NAME(uint32_t* out, uint32_t iters, uint32_t seed) { \
        uint32_t x[8];                                                                                                 \
        _Pragma("unroll") for (int j = 0; j < 8; j++) x[j] = (seed + j) ^ (threadIdx.x * 0x9e3779b9u);                 \
        const uint32_t c = 0x83DCD12Du;                                                                                \
        uint32_t i = 0;                                                                                                \
        for (; iters - i >= 16; i += 16) {                                                                             \
            _Pragma("unroll") for (int j = 0; j < 128; j++) asm volatile(ASM : "+v"(x[j % 8]) : "v"(c));               \
        }                                                                                                              \
        for (; i < iters; i++) {                                                                                       \
            _Pragma("unroll") for (int j = 0; j < 8; j++) asm volatile(ASM : "+v"(x[j]) : "v"(c));                     \
        }                                                                                                              \
        const uint32_t r = x[0] ^ x[1] ^ x[2] ^ x[3] ^ x[4] ^ x[5] ^ x[6] ^ x[7];                                      \
        if (r == 0x12345678u) *out = r;                                                                                \
    }
OP_PROBE(add, "v_add_u32 %0, %0, %1")
OP_PROBE(and, "v_and_b32 %0, %0, %1")
OP_PROBE(mul_lo, "v_mul_lo_u32 %0, %0, %1")
OP_PROBE(mad_u24, "v_mad_u32_u24 %0, %0, %1, %1")
OP_PROBE(bfe, "v_bfe_u32 %0, %0, 5, 16")
OP_PROBE(alignbit, "v_alignbit_b32 %0, %0, %1, 16")
OP_PROBE(perm, "v_perm_b32 %0, %0, %1, %1")
OP_PROBE(sad_u8, "v_sad_u8 %0, %0, 0, %1")
OP_PROBE(sad_hi_u8, "v_sad_hi_u8 %0, %0, 0, %1")
OP_PROBE(pk_fma_f16, "v_pk_fma_f16 %0, %0, %1, %1")
OP_PROBE(fma_f32, "v_fma_f32 %0, %0, %1, %1")
OP_PROBE(dpp_mov, "v_mov_b32_dpp %0, %0 row_shr:1 row_mask:0xf bank_mask:0xf")
