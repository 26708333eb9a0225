// Matrix-core GEMM core for prompt-sized products of 16-bit operands, C[m, n] = sum_k A[m, k] * B[n, k], both K-contiguous, f32
// accumulation.  Shared by the bf16 linears (linear_generic.hip) and the integer form of the I-quant linears (split_gemm.hip).
//
// A workgroup owns a tile of C, a wave a part of it in 32 x 32 accumulators of v_mfma_f32_32x32x16 (TgShape).  What bounds such a kernel on gfx950 is everything beside the matrix cores, so:
//   * both operand tiles (64 deep) go from global memory straight into LDS (global_load_lds, 16 bytes per lane: no registers, no
//     vector-ALU work).  A staged row is 128 bytes, unpadded; the 16-byte chunk c of row r sits at position c ^ (r & 7), so the eight
//     rows that a group of eight lanes reads lie in eight different bank groups;
//   * the requests are issued by an instruction the compiler does not track (tg_request_1k), because behind one that it does it
//     makes every LDS read wait for all requests under way, the other stage's included.  The waits are written out instead;
//   * a request occupies the address path of the compute unit for 16 clocks and a wave that issues several in a row stands still while the
//     path is busy, its products included.  In shapes of three or more stages tg_product therefore spreads the requests of the stage STAGES - 1 ahead between
//     the products of the stage in use, and reads a stage's first fragments under the last products of the one before it.  (Two stages: two workgroups a
//     compute unit, of which one multiplies while the other issues.)  Against all requests at the
//     head of a stage, bf16, rows x columns x depth: 128 x 128 tiles 1500 x 2048 x 6144 51 -> 43 us (727 -> 889 TFLOP/s), 256 x 128 tiles 2048 x 24576 x
//     4096 404 -> 369 us (1116 TFLOP/s; products alone, no memory: 1550 on random numbers, where the clock falls to 1.6 GHz);
//   * tiles are numbered row-fastest and dealt to the eight XCDs in contiguous runs (workgroup i runs on XCD i % 8), so the rows of a
//     column block are multiplied out of one XCD's L2.
#pragma once
#include <type_traits>
#include "vmx_kernels.h"

typedef float tg_f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 tg_f16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t tg_u32x4 __attribute__((ext_vector_type(4)));   // a native vector: HIP's uint4 in arrays ends in scratch or in 4-byte LDS reads

constexpr int TG_BK = 64;

// bf16 -> fp16, saturating at the largest finite half (a bf16 value inside fp16's normal range converts exactly; smaller ones
// lose bits that are below 2^-24 in absolute terms)
__device__ __forceinline__ uint16_t bf16_value_to_f16(uint16_t v) {
    return __builtin_bit_cast(uint16_t, (_Float16)fminf(fmaxf(vmx_bf16_to_f32(v), -65504.0f), 65504.0f));
}

template <bool F16>
__device__ __forceinline__ tg_f32x16 tg_mfma(tg_u32x4 a, tg_u32x4 b, tg_f32x16 c) {
    if constexpr (F16)
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(tg_f16x8, a), __builtin_bit_cast(tg_f16x8, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(vmx_bf16x8, a), __builtin_bit_cast(vmx_bf16x8, b), c, 0, 0, 0);
}

// Tile of workgroup `id` in a grid of tg_grid(tiles) workgroups, or -1.
__device__ __forceinline__ int tg_tile(int id, int tiles) {
    const int run = (tiles + 7) >> 3, t = (id & 7) * run + (id >> 3);
    return t < tiles ? t : -1;
}
inline unsigned tg_grid(int tiles) { return (unsigned)((tiles + 7) / 8 * 8); }

// Row of element r (0 .. 15) of a 32 x 32 accumulator in lane `lane` (its column is lane & 31).
__device__ __forceinline__ int tg_acc_row(int lane, int r) { return 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3); }

// LDS byte address of a __shared__ array (taken once: the cast of a pointer computed from it costs a null check each time)
__device__ __forceinline__ uint32_t tg_lds_at(const void *array) { return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) char *)array; }
// 16 bytes of LDS at a byte address
__device__ __forceinline__ tg_u32x4 tg_lds_read(uint32_t at) { return *(const __attribute__((address_space(3))) tg_u32x4 *)(uintptr_t)at; }

// 64 lanes x 16 bytes from base + off (per lane) to the 1 KiB of LDS from byte `at` on (wave-uniform), in flight until vmcnt says otherwise.
__device__ __forceinline__ void tg_request_1k(uint32_t at, const char *base, uint32_t off) {
    at = __builtin_amdgcn_readfirstlane(at);
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(at), "v"(off), "s"(base) : "m0", "memory");
}

// Shape of a workgroup: WM x WN waves, each MI x NJ accumulators; STAGES tiles of both operands in LDS.  A32: the rows of A are f32, staged as they
// are (256 bytes a row: the chunk c of row r at c ^ 2 (r & 7)) and rounded to bf16 as fragments.
template <int WM_, int WN_, int MI_, int NJ_, int STAGES_, bool A32_ = false>
struct TgShape {
    static constexpr int WM = WM_, WN = WN_, MI = MI_, NJ = NJ_, STAGES = STAGES_;
    static constexpr bool A32 = A32_;
    static constexpr int BM = WM * MI * 32, BN = WN * NJ * 32, WAVES = WM * WN, THREADS = 64 * WAVES;
    static constexpr int AR = A32 ? 2 * BM : BM;                                  // 128-byte pieces of A a stage
    static constexpr int AQ = AR / (8 * WAVES), BQ = BN / (8 * WAVES);            // requests of eight pieces a wave makes per operand and stage
    static constexpr int STAGE = (AR + BN) * TG_BK, LDS = STAGES * STAGE * 2;     // 16-bit elements, bytes
    static constexpr int PER_UNIT = 160 * 1024 / LDS, PER_SIMD = PER_UNIT * WAVES > 4 ? PER_UNIT * WAVES / 4 : 1;   // workgroups a compute unit, waves a SIMD
    static_assert(BM % (8 * WAVES) == 0 && BN % (8 * WAVES) == 0 && STAGES >= 2, "whole requests per wave");
};

// Row of a tile that the lane fetches for request q of its wave (Q requests a wave), and the byte its chunk starts at in that row.
template <int Q>
__device__ __forceinline__ int tg_src_row(int wave, int lane, int q) { return (wave * Q + q) * 8 + (lane >> 3); }
__device__ __forceinline__ uint32_t tg_src_byte(int lane) { return (uint32_t)(((lane & 7) ^ (lane >> 3)) << 4); }
// ... and of an f32 operand (four rows a request)
template <int Q>
__device__ __forceinline__ int tg_src_row32(int wave, int lane, int q) { return (wave * Q + q) * 4 + (lane >> 4); }
__device__ __forceinline__ uint32_t tg_src_byte32(int lane, int row) { return (uint32_t)(((lane & 15) ^ (2 * (row & 7))) << 4); }

// What the two products below share: where a lane's fragments lie, the requests of one 64 deep step, the products of one stage.
template <bool F16, class S>
struct TgCore {
    const char *A, *B;                       // uniform; the lane's chunks at a_src / b_src bytes from them (tg_src_row, tg_src_byte)
    const uint32_t (&a_src)[S::AQ];
    const uint32_t (&b_src)[S::BQ];
    uint32_t lds;                            // byte address of the stages (tg_lds_at)
    int wave, lane;

    // request q (of AQ + BQ) of this wave for step t
    __device__ __forceinline__ void request_one(int t, int stage, int q) const {
        const uint32_t to = lds + stage * (S::STAGE * 2);
        if (q < S::AQ) tg_request_1k(to + (wave * S::AQ + q) * (8 * TG_BK * 2), A + (int64_t)t * ((S::A32 ? 4 : 2) * TG_BK), a_src[q < S::AQ ? q : 0]);
        else tg_request_1k(to + (S::AR + (wave * S::BQ + q - S::AQ) * 8) * (TG_BK * 2), B + (int64_t)t * (2 * TG_BK), b_src[q < S::AQ ? 0 : q - S::AQ]);
    }
    __device__ __forceinline__ void request(int t, int stage) const {
#pragma unroll
        for (int q = 0; q < S::AQ + S::BQ; q++) request_one(t, stage, q);
    }
    // the wave's fragments of the 16 deep step s of a stage.  Chunk c lies at c ^ (row & 7), so step s is step 0 with 32 s flipped in.
    __device__ __forceinline__ void read(int stage, int s, tg_u32x4 (&af)[S::MI], tg_u32x4 (&bf)[S::NJ]) const {
        const int fr = lane & 31, first = (((lane >> 5) ^ (fr & 7)) << 4);
        const uint32_t from = lds + stage * (S::STAGE * 2);
        const uint32_t arow = from + ((wave / S::WN) * (S::MI * 32) + fr) * (TG_BK * 2) + first;
        const uint32_t brow = from + (S::AR + (wave % S::WN) * (S::NJ * 32) + fr) * (TG_BK * 2) + first;
        if constexpr (S::A32) {   // chunks 4 s + 2 (lane / 32) and the one behind it
            const uint32_t at = from + ((wave / S::WN) * (S::MI * 32) + fr) * (TG_BK * 4) + (((lane >> 5) ^ (fr & 7)) << 5);
#pragma unroll
            for (int i = 0; i < S::MI; i++) {
                const uint32_t chunk = (at ^ (64 * s)) + i * (32 * TG_BK * 4);
                const tg_u32x4 lo = tg_lds_read(chunk), hi = tg_lds_read(chunk + 16);
                const float f[8] = {__uint_as_float(lo[0]), __uint_as_float(lo[1]), __uint_as_float(lo[2]), __uint_as_float(lo[3]),
                                    __uint_as_float(hi[0]), __uint_as_float(hi[1]), __uint_as_float(hi[2]), __uint_as_float(hi[3])};
                af[i] = __builtin_bit_cast(tg_u32x4, vmx_pack16x8<false>(f));
            }
        } else {
#pragma unroll
            for (int i = 0; i < S::MI; i++) af[i] = tg_lds_read((arow ^ (32 * s)) + i * (32 * TG_BK * 2));
        }
#pragma unroll
        for (int j = 0; j < S::NJ; j++) bf[j] = tg_lds_read((brow ^ (32 * s)) + j * (32 * TG_BK * 2));
    }
    // acc += the 64 deep products of a stage; FRESH: acc = them
    template <bool FRESH = false>
    __device__ __forceinline__ void multiply(int stage, tg_f32x16 (&acc)[S::MI][S::NJ]) const {
        tg_u32x4 af[2][S::MI], bf[2][S::NJ];   // fragments of the 16 deep step in use and of the next one
        read(stage, 0, af[0], bf[0]);
#pragma unroll
        for (int s = 0; s < TG_BK / 16; s++) {
            if (s + 1 < TG_BK / 16) read(stage, s + 1, af[(s + 1) & 1], bf[(s + 1) & 1]);
#pragma unroll
            for (int i = 0; i < S::MI; i++)
#pragma unroll
                for (int j = 0; j < S::NJ; j++) acc[i][j] = tg_mfma<F16>(af[s & 1][i], bf[s & 1][j], FRESH && s == 0 ? tg_f32x16{} : acc[i][j]);
            __builtin_amdgcn_sched_barrier(0);   // the reads stay ahead of the products they run under
        }
    }
    // all but N of this wave's requests have landed, and everybody's of that step; nobody reads the step before it any more
    template <int N>
    __device__ __forceinline__ void arrive() const {
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" : : "n"(N) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    }
};

// acc += sum over k in [0, K), K a positive multiple of 64.
template <bool F16, class S>
__device__ __forceinline__ void tg_product(const TgCore<F16, S> &core, int K, tg_f32x16 (&acc)[S::MI][S::NJ]) {
    if constexpr (S::STAGES == 2) {   // a whole stage's requests at its head; the other workgroup of the compute unit multiplies meanwhile
        const int steps = K / TG_BK;
        core.request(0, 0);
        for (int t = 0; t < steps; t++) {
            core.template arrive<0>();
            if (t + 1 < steps) core.request(t + 1, (t + 1) & 1);
            core.multiply(t & 1, acc);
        }
        return;
    }
    constexpr int AHEAD = S::STAGES - 1, R = S::AQ + S::BQ, SUB = TG_BK / 16, P = S::MI * S::NJ;
    const int steps = K / TG_BK;
    tg_u32x4 af[2][S::MI], bf[2][S::NJ];   // fragments of the 16 deep step in use and of the next one
    // the products of stage `cur` (its first fragments are in af[0], bf[0]); REQUEST: with the requests of step t + AHEAD between them, which go to
    // the stage that was read before this one; MORE: the next stage's first fragments are read
    auto stage = [&](auto request, auto more, int t, int cur) {
        constexpr bool REQUEST = decltype(request)::value, MORE = decltype(more)::value;
        const int next = cur == AHEAD ? 0 : cur + 1, free = cur == 0 ? AHEAD : cur - 1;
#pragma unroll
        for (int s = 0; s < SUB; s++) {
            if (s + 1 < SUB) {
                core.read(cur, s + 1, af[(s + 1) & 1], bf[(s + 1) & 1]);
            } else if (MORE) {
                core.template arrive<REQUEST ? R * (AHEAD - 1) : 0>();
                core.read(next, 0, af[0], bf[0]);
            }
#pragma unroll
            for (int i = 0; i < S::MI; i++)
#pragma unroll
                for (int j = 0; j < S::NJ; j++) {
                    acc[i][j] = tg_mfma<F16>(af[s & 1][i], bf[s & 1][j], acc[i][j]);
                    // behind product n of the first SUB - 1 sub-steps: requests up to R (n + 1) / all of those products
                    const int n = s * P + i * S::NJ + j;
                    if (REQUEST && s + 1 < SUB) {
#pragma unroll
                        for (int q = 0; q < R; q++)
                            if (q >= (n * R + (SUB - 1) * P - 1) / ((SUB - 1) * P) && q < ((n + 1) * R + (SUB - 1) * P - 1) / ((SUB - 1) * P)) {
                                __builtin_amdgcn_sched_barrier(0);
                                core.request_one(t + AHEAD, free, q);
                            }
                    }
                }
            __builtin_amdgcn_sched_barrier(0);   // the reads stay ahead of the products they run under
        }
    };
    const std::true_type yes;
    const std::false_type no;
#pragma unroll
    for (int t = 0; t < AHEAD; t++)
        if (t < steps) core.request(t, t);
    if (steps >= AHEAD) core.template arrive<R * (AHEAD - 1)>();
    else core.template arrive<0>();
    core.read(0, 0, af[0], bf[0]);
    int cur = 0, t = 0;
    for (; t + AHEAD < steps; t++) {
        stage(yes, yes, t, cur);
        cur = cur == AHEAD ? 0 : cur + 1;
    }
    for (; t + 1 < steps; t++) {
        stage(no, yes, t, cur);
        cur = cur == AHEAD ? 0 : cur + 1;
    }
    stage(no, no, t, cur);
}

// acc[m][n] += sum over groups of 256 k of scale(group, n) * (sum over the group's k), groups of them; two stages.
// load(g, d): the lane's NJ scales of group g.
template <bool F16, class S, class Load>
__device__ __forceinline__ void tg_product_scaled(const TgCore<F16, S> &core, int groups, tg_f32x16 (&acc)[S::MI][S::NJ], Load &&load) {
    static_assert(S::STAGES == 2, "the scales of a group are requested between two waits for everything");
    const int steps = groups * 4;
    if (steps > 0) core.request(0, 0);
    for (int g = 0; g < groups; g++) {
        tg_f32x16 part[S::MI][S::NJ];
        float d[S::NJ];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            core.template arrive<0>();
            if (u == 0) load(g, d);
            if (u == 1) {   // a use right behind that wait: the compiler's own wait for the scales falls here, where it costs nothing
#pragma unroll
                for (int j = 0; j < S::NJ; j++) asm volatile("" : "+v"(d[j]));
            }
            if (4 * g + u + 1 < steps) core.request(4 * g + u + 1, (u + 1) & 1);
            if (u == 0) core.template multiply<true>(0, part);
            else core.multiply(u & 1, part);
        }
#pragma unroll
        for (int i = 0; i < S::MI; i++)
#pragma unroll
            for (int j = 0; j < S::NJ; j++)
#pragma unroll
                for (int r = 0; r < 16; r++) acc[i][j][r] = fmaf(d[j], part[i][j][r], acc[i][j][r]);
    }
}
