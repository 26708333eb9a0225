// Prompt-sized linears (more than 16 rows) over GGUF I-quant weights, decoded inside the product: IQ2_XS, IQ2_S, IQ3_XXS, IQ3_S.
//
// A dequantised weight is d * c * I with d the f16 super-block scale, c a power of two and I = (2 ls + 1) * (signed codebook byte) an integer of at
// most 11 bits (IQ3_XXS: 31 * 62), so I is exact in fp16 and the f32 product the reference forms (iq_dequant.cu: db * grid byte, no rounding:
// 11 + 5 + 6 bits) equals (d * c) * I.  C[m, n] = sum_sb (d c)[n, sb] * ( sum_{k in sb} A16[m, k] * I[n, k] ), A16 = the activations as fp16 (bf16
// values convert exactly inside fp16's range): every product is exact, the 256 products of a super-block are added in f32 by the matrix core, and
// the scale is applied once per super-block to the finished sum -- the reference's f32 GEMM on the dequantised weight (IqLinear::forward_inner,
// crates/core/src/quantization/gguf/mod.rs:346-365) up to summation order.
//
// What bounds it.  Dequantising first writes and reads every weight in 16 bits (gate|up of 256 rows x 30720 x 3840: 55 us of writing at 4.3 TB/s,
// then a product that waits for 236 MB).  Here a workgroup of eight waves owns BM rows x 128 columns and walks k in stages of 64:
//   * the raw blocks of its columns (74 .. 110 bytes each, 2-byte aligned) come into LDS by LDS-DMA in whole dwords, (TS + 2) / 4 of them from the
//     dword that holds a block's first byte on: every dword fetched holds a byte of the block;
//   * a thread decodes 16 weights of every stage (four neighbours share a column) in three steps a stage apart, so that none waits for LDS: raw
//     fields, codebook bytes, weights.  Codebook bytes become fp16 pairs by one byte permutation and one fused multiply-add with 2 ls + 1, sign bits
//     move to the sign positions of the pairs; two 16-byte writes into the stage's B tile;
//   * the rows come by LDS-DMA two stages ahead as in tile_gemm.h.  No load of the loop is one the compiler tracks, so none of its waits drains the
//     requests under way; raw blocks are asked for a super-block ahead, between the rows' requests.
// 256 rows x 30720 x 3840 (IQ3_XXS, weights out of HBM): 157 us dequantised first, 72 .. 78 here; of those the products alone take 46 (the clock falls under
// them), no decode 62, no fragment reads 66, no requests 66: LDS pipe (1.7 k clocks a stage), matrix cores (1.0 k) and vector ALU (0.7 k) overlap but not
// wholly, as every wave meets the others' phase at the stage's barrier.
#include <algorithm>
#include "iq_common.h"
#include "tile_gemm.h"
#include "vmx_internal.h"

namespace {

typedef _Float16 iqp_h2 __attribute__((ext_vector_type(2)));
typedef uint32_t iqp_u32x2 __attribute__((ext_vector_type(2)));

constexpr int IQP_BN = 128, IQP_WAVES = 8, IQP_THREADS = 512;

template <int T> struct Iqp {
    static constexpr int TS = IqTraits<T>::TS, ND = (TS + 2) / 4;                              // block bytes; dwords fetched of a block
    static constexpr int REQ = (IQP_BN * ND + 64 * IQP_WAVES - 1) / (64 * IQP_WAVES);          // raw requests of a wave and super-block
    static constexpr int RAW = REQ * IQP_WAVES * 256;                                          // bytes of a raw buffer
    static constexpr bool WIDE = T == 17 || T == 22;                                           // codebook entries of eight weights
    static constexpr int TAB = IqTraits<T>::LDS_WORDS * 4;
    static constexpr float C = WIDE ? 0.125f : T == 18 ? 0.25f : 1.0f;
    static_assert(REQ <= 8, "vmcnt counts 63");
};

template <int WM_, int WN_, int MI_, int NJ_>
struct IqpShape {
    static constexpr int WM = WM_, WN = WN_, MI = MI_, NJ = NJ_, BM = WM * MI * 32, AQ = BM / (8 * IQP_WAVES), A_STAGE = BM * TG_BK * 2;
    static_assert(WM * WN == IQP_WAVES && WN * NJ * 32 == IQP_BN && AQ * 8 * IQP_WAVES == BM, "eight waves, 128 columns, whole requests");
};
constexpr int IQP_B_STAGE = IQP_BN * TG_BK * 2;
template <class S, int T> constexpr int iqp_lds() { return 3 * S::A_STAGE + 2 * IQP_B_STAGE + 2 * Iqp<T>::RAW + Iqp<T>::TAB; }

struct IqpSeg {
    const uint8_t *w;      // raw blocks [n][K / 256] (GEGLU: the gate's)
    int type, n, tile0;    // rows of the weight; first column tile
    int64_t col;           // first output column
};
struct IqpArgs {
    IqpSeg seg[3];
    int nseg;
    const uint8_t *w_up;   // GEGLU
    const uint16_t *A;     // fp16 [M][K]
    float *C;              // [slices][M][ldc]
    uint16_t *act;         // GEGLU: fp16 [M][n]
    int M, K, row_tiles, tiles, per_slice;
    int64_t ldc, slice_stride;
};

// 64 lanes x 4 bytes from each lane's address to the 256 bytes of LDS from byte `at` on (wave-uniform)
__device__ __forceinline__ void iqp_request_dwords(uint32_t at, const uint8_t *src) {
    at = __builtin_amdgcn_readfirstlane(at);
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off" : : "s"(at), "v"(src) : "m0", "memory");
}
template <typename T> __device__ __forceinline__ T iqp_lds_at(uint32_t at) { return *(const __attribute__((address_space(3))) T *)(uintptr_t)at; }
__device__ __forceinline__ void iqp_lds_write(uint32_t at, tg_u32x4 v) { *(__attribute__((address_space(3))) tg_u32x4 *)(uintptr_t)at = v; }

// Codebook into LDS: entries of four (IQ3) or eight (IQ2) bytes, at most 62.  Four-byte entries spread over all banks: as fp16 quadruples of
// eight bytes the gathers of a stage took 2.5 times the clocks of the LDS pipe, which is what bounds the product.
template <int T>
__device__ __forceinline__ void iqp_tables(uint32_t tab) {
    const uint32_t *src = codebook_src<T>();
    for (int i = threadIdx.x; i < IqTraits<T>::LDS_WORDS; i += IQP_THREADS) *(__attribute__((address_space(3))) uint32_t *)(uintptr_t)(tab + 4 * i) = src[i];
}

// What a thread needs of a raw block for its 16 weights (quarter q of the 64 of step u of the super-block): read first, decoded later.
struct IqpRaw { uint32_t lo, hi, a, b, c; };

// row: LDS byte of the block's first byte (2-byte aligned)
template <int T>
__device__ __forceinline__ IqpRaw iqp_fetch(uint32_t row, int u, int q) {
    IqpRaw r = {};
    const int ib = 2 * u + (q >> 1);
    if constexpr (T == 18 || T == 21 || T == 17) {   // four bytes at 2 + 8 ib + 4 (q & 1)
        const uint32_t p = (row + 2 + 16 * u + 4 * q) & ~3u;
        r.lo = iqp_lds_at<uint32_t>(p);
        r.hi = iqp_lds_at<uint32_t>(p + 4);
    } else {
        r.lo = iqp_lds_at<uint16_t>(row + 2 + 4 * ib + 2 * (q & 1));
    }
    if constexpr (T == 18) {
        const uint32_t p = (row + 66 + 4 * ib) & ~3u;
        r.a = iqp_lds_at<uint32_t>(p);
        r.b = iqp_lds_at<uint32_t>(p + 4);
    } else if constexpr (T == 21) {
        r.a = iqp_lds_at<uint16_t>(row + 74 + 4 * ib + 2 * (q & 1));
        r.b = iqp_lds_at<uint8_t>(row + 66 + ib);
        r.c = iqp_lds_at<uint8_t>(row + 106 + u);
    } else if constexpr (T == 22) {
        r.a = iqp_lds_at<uint16_t>(row + 34 + 4 * ib + 2 * (q & 1));
        r.b = iqp_lds_at<uint8_t>(row + 66 + ib);
        r.c = iqp_lds_at<uint8_t>(row + 74 + ib);
    } else {
        r.c = iqp_lds_at<uint8_t>(row + 66 + ib);
    }
    return r;
}

// Codebook bytes of the 16 weights, the signs of either half, 2 ls + 1.
struct IqpCodes { uint32_t g[4], s8[2], scale; };

template <int T>
__device__ __forceinline__ IqpCodes iqp_gather(const IqpRaw &r, uint32_t row, int q, uint32_t tab) {
    IqpCodes o;
    const int h = q & 1;
    const uint32_t sh = (row + 2) & 3;   // 0 or 2
    auto entry4 = [&](int j, uint32_t idx) { o.g[j] = iqp_lds_at<uint32_t>(tab + 4 * idx); };
    auto entry8 = [&](int j, uint32_t idx) {
        const iqp_u32x2 v = iqp_lds_at<iqp_u32x2>(tab + 8 * idx);
        o.g[2 * j] = v[0], o.g[2 * j + 1] = v[1];
    };
    auto parity = [](uint32_t c) { return c | ((__popc(c) & 1u) << 7); };
    if constexpr (T == 18) {
        const uint32_t qs = __builtin_amdgcn_alignbyte(r.hi, r.lo, sh), w = __builtin_amdgcn_alignbyte(r.b, r.a, sh), ws = w >> (14 * h);
#pragma unroll
        for (int j = 0; j < 4; j++) entry4(j, (qs >> (8 * j)) & 0xFFu);
        o.s8[0] = parity(ws & 127u);
        o.s8[1] = parity((ws >> 7) & 127u);
        o.scale = 2 * (w >> 28) + 1;
    } else if constexpr (T == 21) {
        const uint32_t qs = __builtin_amdgcn_alignbyte(r.hi, r.lo, sh), hb = r.b >> (4 * h);
#pragma unroll
        for (int j = 0; j < 4; j++) entry4(j, ((qs >> (8 * j)) & 0xFFu) | ((hb << (8 - j)) & 256u));
        o.s8[0] = r.a & 0xFFu;
        o.s8[1] = r.a >> 8;
        o.scale = 2 * ((r.c >> (4 * (q >> 1))) & 0xFu) + 1;
    } else if constexpr (T == 22) {
        const uint32_t hb = r.b >> (4 * h);
        entry8(0, (r.lo & 0xFFu) | ((hb << 8) & 0x300u));
        entry8(1, (r.lo >> 8) | ((hb << 6) & 0x300u));
        o.s8[0] = r.a & 0xFFu;
        o.s8[1] = r.a >> 8;
        o.scale = 2 * ((r.c >> (4 * h)) & 0xFu) + 1;
    } else {
        const uint32_t w = __builtin_amdgcn_alignbyte(r.hi, r.lo, sh);
        entry8(0, w & 511u);
        entry8(1, (w >> 16) & 511u);
        o.s8[0] = parity((w >> 9) & 127u);
        o.s8[1] = parity(w >> 25);
        o.scale = 2 * ((r.c >> (4 * h)) & 0xFu) + 1;
    }
    return o;
}

// eight fp16 integers of half hf: 1024 + byte as fp16, times 2 ls + 1, less 1024 (2 ls + 1): exact, 1024 * 31 < 65504
__device__ __forceinline__ tg_u32x4 iqp_expand(const IqpCodes &c, int hf) {
    const _Float16 s1 = (_Float16)(float)c.scale;
    const iqp_h2 s = {s1, s1}, off = s * (iqp_h2){(_Float16)-1024.0f, (_Float16)-1024.0f};
    uint32_t t = c.s8[hf] | (c.s8[hf] << 15);
    asm("" : "+v"(t));   // or the compiler makes four multiplications, 16 clocks each, of the four shifts
    tg_u32x4 v;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const uint32_t b = __builtin_amdgcn_perm(c.g[2 * hf + (j >> 1)], 0x64646464u, j & 1 ? 0x00070006u : 0x00050004u);
        const uint32_t pair = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(__builtin_bit_cast(iqp_h2, b), s, off));
        v[j] = pair ^ ((t << (15 - 2 * j)) & 0x80008000u);   // sign bits 2 j and 2 j + 1 to bits 15 and 31
    }
    return v;
}

template <int T, class S, bool GEGLU>
__device__ __forceinline__ void iqp_body(const IqpArgs &p, const IqpSeg &seg, int m0, int ct, uint32_t lds) {
    constexpr int TS = Iqp<T>::TS, ND = Iqp<T>::ND, REQ = Iqp<T>::REQ, MI = S::MI, NJ = S::NJ, AQ = S::AQ;
    constexpr int RA = (REQ + 1) / 2, RB = REQ - RA;   // raw requests in steps 1 and 2 of a super-block
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nsb = p.K >> 8, sb0 = blockIdx.y * p.per_slice, groups = min(p.per_slice, nsb - sb0), steps = 4 * groups;
    const uint32_t a_at = lds, b_at = lds + 3 * S::A_STAGE, raw_at = b_at + 2 * IQP_B_STAGE, tab = raw_at + 2 * Iqp<T>::RAW;
    // tile column -> row of the weight (GEGLU: 16 gate and 16 up columns in every 32)
    auto w_row = [&](int c) { return GEGLU ? min(ct * 64 + (c >> 5) * 16 + (c & 15), seg.n - 1) : min(ct * IQP_BN + c, seg.n - 1); };
    auto w_base = [&](int c) { return GEGLU && (c & 16) ? p.w_up : seg.w; };
    // where a column's block of the slice's first super-block starts
    auto w_start = [&](int c) { return w_base(c) + ((int64_t)w_row(c) * nsb + sb0) * TS; };

    const char *A = (const char *)(p.A + (int64_t)sb0 * 256);
    uint32_t a_src[AQ];
#pragma unroll
    for (int q = 0; q < AQ; q++) a_src[q] = (uint32_t)((int64_t)min(m0 + tg_src_row<AQ>(wave, lane, q), p.M - 1) * p.K * 2) + tg_src_byte(lane);
    auto request_a = [&](int t, int stage, int q) {
        tg_request_1k(a_at + stage * S::A_STAGE + (wave * AQ + q) * (8 * TG_BK * 2), A + (int64_t)t * (2 * TG_BK), a_src[q]);
    };
    // a lane's dword of request q: byte of its block in the weight (GEGLU: bit 0 set for the up weight's; blocks start at even bytes), 4 x the dword
    uint32_t raw_off[REQ], raw_dw[REQ];
#pragma unroll
    for (int q = 0; q < REQ; q++) {
        const int f = min((wave * REQ + q) * 64 + lane, IQP_BN * ND - 1), c = f / ND;
        raw_off[q] = ((uint32_t)w_row(c) * (uint32_t)nsb + (uint32_t)sb0) * TS + (GEGLU && (c & 16) ? 1u : 0u);
        raw_dw[q] = 4 * (f - c * ND);
    }
    auto request_raw = [&](int g, int buf, int q) {
        const uint64_t base = (uint64_t)(uintptr_t)(GEGLU && (raw_off[q] & 1) ? p.w_up : seg.w);
        const uint64_t at = (base + (raw_off[q] & ~1u) + (uint32_t)(g * TS)) & ~(uint64_t)3;
        iqp_request_dwords(raw_at + buf * Iqp<T>::RAW + (wave * REQ + q) * 256, (const uint8_t *)(uintptr_t)(at + raw_dw[q]));
    };
    // the thread's 16 weights of a stage: quarter dq of column dc
    const int dc = tid >> 2, dq = tid & 3;
    const uint32_t d_row = raw_at + dc * (4 * ND), d_odd = (uint32_t)(uintptr_t)w_start(dc) & 2u;
    const uint32_t d_to = b_at + dc * (TG_BK * 2), d_c0 = (uint32_t)((2 * dq) ^ (dc & 7)) << 4, d_c1 = (uint32_t)((2 * dq + 1) ^ (dc & 7)) << 4;
    static_assert((TS & 3) == 2, "block starts alternate between the halves of a dword");
    auto row_of = [&](int g) { return d_row + (g & 1) * Iqp<T>::RAW + (d_odd ^ (2 * (g & 1))); };
    // scales of this lane's columns: the f16 at a block's first byte
    const int wc = wave % S::WN * (NJ * 32) + (lane & 31);
    uint32_t s_row[NJ], s_odd[NJ];
#pragma unroll
    for (int j = 0; j < NJ; j++) {
        s_row[j] = raw_at + (wc + 32 * j) * (4 * ND);
        s_odd[j] = (uint32_t)(uintptr_t)w_start(wc + 32 * j) & 2u;
    }

    // start: raw blocks of two super-blocks, rows of two stages; weights of stage 0 decoded, codes of stage 1 and raw fields of stage 2 in registers
    iqp_tables<T>(tab);
#pragma unroll
    for (int q = 0; q < REQ; q++) request_raw(0, 0, q);
#pragma unroll
    for (int q = 0; q < AQ; q++) request_a(0, 0, q);
#pragma unroll
    for (int q = 0; q < REQ; q++) request_raw(min(1, groups - 1), 1, q);
#pragma unroll
    for (int q = 0; q < AQ; q++) request_a(min(1, steps - 1), 1, q);
    auto arrive = [&](auto left) {
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" : : "n"(decltype(left)::value) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    auto put = [&](const IqpCodes &c, int hf, int par) { iqp_lds_write(d_to + par * IQP_B_STAGE + (hf ? d_c1 : d_c0), iqp_expand(c, hf)); };
    arrive(std::integral_constant<int, AQ + REQ>{});
    IqpCodes codes = iqp_gather<T>(iqp_fetch<T>(row_of(0), 0, dq), row_of(0), dq, tab);
    put(codes, 0, 0);
    put(codes, 1, 0);
    codes = iqp_gather<T>(iqp_fetch<T>(row_of(0), 1, dq), row_of(0), dq, tab);
    IqpRaw raw = iqp_fetch<T>(row_of(0), 2, dq);
    arrive(std::integral_constant<int, AQ>{});

    tg_f32x16 acc[MI][NJ], part[MI][NJ];
    float d[NJ], d_next[NJ];
#pragma unroll
    for (int j = 0; j < NJ; j++) d[j] = d_next[j] = 0.f;
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
        for (int j = 0; j < NJ; j++) acc[i][j] = part[i][j] = tg_f32x16{};
    const int fr = lane & 31;
    const uint32_t first = (((lane >> 5) ^ (fr & 7)) << 4);
    const uint32_t arow = a_at + ((wave / S::WN) * (MI * 32) + fr) * (TG_BK * 2) + first;
    const uint32_t brow = b_at + (wave % S::WN * (NJ * 32) + fr) * (TG_BK * 2) + first;
    tg_u32x4 af[2][MI], bf[2][NJ];
    auto read = [&](int stage, int par, int s, int w) {
#pragma unroll
        for (int i = 0; i < MI; i++) af[w][i] = tg_lds_read(((arow + stage * S::A_STAGE) ^ (32 * s)) + i * (32 * TG_BK * 2));
#pragma unroll
        for (int j = 0; j < NJ; j++) bf[w][j] = tg_lds_read(((brow + par * IQP_B_STAGE) ^ (32 * s)) + j * (32 * TG_BK * 2));
    };
    read(0, 0, 0, 0);
    int cur = 0;
    auto stage = [&](auto step, int g) {
        constexpr int U = decltype(step)::value, RAWS = U == 1 ? RA : U == 2 ? RB : 0, RQ = AQ + RAWS, P = MI * NJ;
        constexpr int LATE = U == 2 ? RA : U == 3 ? RB : 0;   // raw requests of the stage before, behind its rows' requests: out of HBM, they have a stage more
        const int t = 4 * g + U, next = cur == 2 ? 0 : cur + 1, free = cur == 0 ? 2 : cur - 1, ta = min(t + 2, steps - 1), gr = min(g + 2, groups - 1);
        constexpr int PAR = U & 1;
#pragma unroll
        for (int s = 0; s < 4; s++) {
            if (s < 3) {
                read(cur, PAR, s + 1, (s + 1) & 1);
            } else {
                arrive(std::integral_constant<int, RQ + LATE>{});
                read(next, PAR ^ 1, 0, 0);
            }
            // stage t + 1's weights from their codes, t + 2's codes from their raw fields, t + 3's raw fields: each waits for nothing of this stage
            if (s == 0) put(codes, 0, PAR ^ 1);
            if (s == 1) {
                put(codes, 1, PAR ^ 1);
                codes = iqp_gather<T>(raw, row_of(U >= 2 ? g + 1 : g), dq, tab);
            }
            if (s == 2) {
                raw = iqp_fetch<T>(row_of(U >= 1 ? g + 1 : g), (U + 3) & 3, dq);
                if constexpr (U == 0) {
#pragma unroll
                    for (int j = 0; j < NJ; j++)
                        d_next[j] = Iqp<T>::C * vmx_f16_to_f32(iqp_lds_at<uint16_t>(s_row[j] + (g & 1) * Iqp<T>::RAW + (s_odd[j] ^ (2 * (g & 1)))));
                }
            }
#pragma unroll
            for (int i = 0; i < MI; i++)
#pragma unroll
                for (int j = 0; j < NJ; j++) {
                    if constexpr (U == 0) {
                        if (s == 0) {   // the super-block before: its sums take their scales as their registers are needed
#pragma unroll
                            for (int r = 0; r < 16; r++) acc[i][j][r] = fmaf(d[j], part[i][j][r], acc[i][j][r]);
                        }
                        part[i][j] = tg_mfma<true>(af[s & 1][i], bf[s & 1][j], s == 0 ? tg_f32x16{} : part[i][j]);
                    } else {
                        part[i][j] = tg_mfma<true>(af[s & 1][i], bf[s & 1][j], part[i][j]);
                    }
                    const int n = s * P + i * NJ + j;
                    if (s < 3) {
#pragma unroll
                        for (int q = 0; q < RQ; q++)
                            if (q >= (n * RQ + 3 * P - 1) / (3 * P) && q < ((n + 1) * RQ + 3 * P - 1) / (3 * P)) {
                                if (q < AQ) request_a(ta, free, q < AQ ? q : 0);
                                else request_raw(gr, g & 1, (U == 1 ? 0 : RA) + q - AQ);
                            }
                    }
                }
            if constexpr (U == 0) {
                if (s == 3) {
#pragma unroll
                    for (int j = 0; j < NJ; j++) d[j] = d_next[j];
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        cur = next;
    };
    for (int g = 0; g < groups; g++) {
        stage(std::integral_constant<int, 0>{}, g);
        stage(std::integral_constant<int, 1>{}, g);
        stage(std::integral_constant<int, 2>{}, g);
        stage(std::integral_constant<int, 3>{}, g);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // requests past the end are still writing LDS
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
        for (int j = 0; j < NJ; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = fmaf(d[j], part[i][j][r], acc[i][j][r]);

    const int wm = m0 + wave / S::WN * (MI * 32), rows = min(p.M - wm, 32 * MI);   // rows of this wave
    if constexpr (GEGLU) {   // act[m][i] = bf16(bf16(gelu_erf(bf16(gate))) * bf16(up)): lanes with bit 4 clear take one row, the others the next
        const bool hi = lane & 16;
#pragma unroll
        for (int j = 0; j < NJ; j++) {
            const int col = ct * 64 + wave % S::WN * (NJ * 16) + 16 * j + (lane & 15);
#pragma unroll
            for (int i = 0; i < MI; i++)
#pragma unroll
                for (int r = 0; r < 16; r += 2) {
                    const float x = acc[i][j][r], y = acc[i][j][r + 1], got = vmx_lane_xor<16>(hi ? x : y);
                    const float gate = hi ? got : x, up = hi ? y : got;
                    const float g = vmx_bf16_to_f32(vmx_f32_to_bf16(gate)), u = vmx_bf16_to_f32(vmx_f32_to_bf16(up));
                    const float ge = vmx_bf16_to_f32(vmx_f32_to_bf16(0.5f * g * (1.0f + erff(g * 0.70710678118654752f))));
                    const int m = 32 * i + tg_acc_row(lane, r) + (hi ? 1 : 0);
                    if (m < rows && col < seg.n) p.act[(int64_t)(wm + m) * seg.n + col] = bf16_value_to_f16(vmx_f32_to_bf16(ge * u));
                }
        }
    } else {
        float *out = p.C + (int64_t)blockIdx.y * p.slice_stride + seg.col + (int64_t)wm * p.ldc;
#pragma unroll
        for (int i = 0; i < MI; i++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int m = 32 * i + tg_acc_row(lane, r);
                if (m >= rows) continue;
                float *row = out + (int64_t)m * p.ldc;
#pragma unroll
                for (int j = 0; j < NJ; j++) {
                    const int n = ct * IQP_BN + wc + 32 * j;
                    if (n < seg.n) row[n] = acc[i][j][r];
                }
            }
    }
}

// grid (tg_grid(tiles), slices)
template <class S, bool GEGLU>
__global__ __launch_bounds__(IQP_THREADS, 2) void iq_prompt_kernel(const IqpArgs p) {
    extern __shared__ __align__(1024) uint16_t iqp_lds_base[];
    const uint32_t lds = tg_lds_at(iqp_lds_base);
    const int tile = tg_tile(blockIdx.x, p.tiles);
    if (tile < 0) return;
    const int m0 = tile % p.row_tiles * S::BM, ct = tile / p.row_tiles;
    int k = 0;
    while (k + 1 < p.nseg && ct >= p.seg[k + 1].tile0) k++;
    const IqpSeg seg = p.seg[k];
    switch (seg.type) {
        case 17: iqp_body<17, S, GEGLU>(p, seg, m0, ct - seg.tile0, lds); break;
        case 18: iqp_body<18, S, GEGLU>(p, seg, m0, ct - seg.tile0, lds); break;
        case 21: iqp_body<21, S, GEGLU>(p, seg, m0, ct - seg.tile0, lds); break;
        default: iqp_body<22, S, GEGLU>(p, seg, m0, ct - seg.tile0, lds); break;
    }
}

typedef IqpShape<2, 4, 1, 1> Iqp64;
typedef IqpShape<4, 2, 1, 2> Iqp128;
typedef IqpShape<2, 4, 3, 1> Iqp192;
typedef IqpShape<4, 2, 2, 2> Iqp256;

template <class S, bool GEGLU>
int iqp_launch(IqpArgs p, int slices, hipStream_t st) {
    int tiles = 0, bytes = 0;
    for (int i = 0; i < p.nseg; i++) {
        p.seg[i].tile0 = tiles;
        tiles += GEGLU ? (p.seg[i].n + 63) / 64 : (p.seg[i].n + IQP_BN - 1) / IQP_BN;
        const int t = p.seg[i].type;
        bytes = std::max(bytes, t == 17 ? iqp_lds<S, 17>() : t == 18 ? iqp_lds<S, 18>() : t == 21 ? iqp_lds<S, 21>() : iqp_lds<S, 22>());
    }
    p.row_tiles = (p.M + S::BM - 1) / S::BM;
    p.tiles = tiles * p.row_tiles;
    const int nsb = p.K / 256;
    p.per_slice = (nsb + slices - 1) / slices;
    // one kernel serves all types: what it may be given is the most that any of them takes, whichever thread asks
    constexpr int most = std::max({iqp_lds<S, 17>(), iqp_lds<S, 18>(), iqp_lds<S, 21>(), iqp_lds<S, 22>()});
    VMX_CHECK_HIP(hipFuncSetAttribute((const void *)iq_prompt_kernel<S, GEGLU>, hipFuncAttributeMaxDynamicSharedMemorySize, most));
    hipLaunchKernelGGL((iq_prompt_kernel<S, GEGLU>), dim3(tg_grid(p.tiles), (nsb + p.per_slice - 1) / p.per_slice), dim3(IQP_THREADS), bytes, st, p);
    VMX_CHECK_LAUNCH("iq_prompt");
    return VMX_OK;
}

// Estimated ns of a launch: rounds of one workgroup a compute unit, each of `per` super-blocks; what a super-block takes with few and with all units
// at work.  us of IQ3_XXS / IQ3_S products, 64 / 128 / 192 / 256 rows a tile:  64 x 30720 x 3840 42 / - / - / -;  128 79 / 53 / 60 / -;  192 114 / 98 /
// 59 / 68;  256 167 / 105 / 121 / 72;  333 215 / 137 / 112 / 131;  512 284 / 184 / 166 / 133;  256 x 3840 x 15360 in 1, 2, 4, 8 slices of k, without
// their sum: 133, 69, 72, 82 / 166, 87, 51, 58 / 195, 104, 61, 67 / 203, 106, 61, 42.
template <class S>
int64_t iqp_ns(int tiles128, int M, int nsb, int slices, int few, int full) {
    const int units = vmx_num_cus(), per = (nsb + slices - 1) / slices;
    const int64_t wgs = (int64_t)tiles128 * ((M + S::BM - 1) / S::BM) * ((nsb + per - 1) / per), rounds = wgs / units, rest = wgs % units;
    return per * (rounds * full + (rest ? few + (full - few) * rest / units : 0)) + 3000 * (rounds + (rest ? 1 : 0));
}
struct IqpPlan { int rows, slices; int64_t ns; };

// Tile rows and slices of k with the least estimate.  A slice costs its f32 sums written and read again (5 TB/s; where rows are not whole 16 bytes they are read one by one,
// a trip to memory a slice: 107 x 2270 x 6144 in 12 slices 33.5 us, in 6 26), and their addition is one launch more.
IqpPlan iqp_plan(int tiles128, int M, int N, int nsb, int64_t most) {
    IqpPlan best = {0, 0, INT64_MAX};
    for (int s = 1; s <= nsb && (s == 1 || s <= most); s++) {
        const int per = (nsb + s - 1) / s;
        if ((nsb + per - 1) / per != s) continue;
        const int64_t sums = s > 1 ? 2500 + (int64_t)s * M * N * 8 / 5000 + (N % 4 ? 900 * s : 0) : 0;
        const int64_t ns[4] = {iqp_ns<Iqp64>(tiles128, M, nsb, s, 2150, 2600), iqp_ns<Iqp128>(tiles128, M, nsb, s, 2750, 3300),
                               iqp_ns<Iqp192>(tiles128, M, nsb, s, 3200, 3700), iqp_ns<Iqp256>(tiles128, M, nsb, s, 3450, 4700)};
        for (int i = 0; i < 4; i++)
            if (ns[i] + sums < best.ns) best = {64 * (i + 1), s, ns[i] + sums};
        if ((int64_t)tiles128 * ((M + 255) / 256) * s > 2 * vmx_num_cus()) break;
    }
    return best;
}

template <bool GEGLU>
int iqp_launch_rows(const IqpArgs &p, const IqpPlan &plan, hipStream_t st) {
    switch (plan.rows) {
        case 64: return iqp_launch<Iqp64, GEGLU>(p, plan.slices, st);
        case 128: return iqp_launch<Iqp128, GEGLU>(p, plan.slices, st);
        case 192: return iqp_launch<Iqp192, GEGLU>(p, plan.slices, st);
        default: return iqp_launch<Iqp256, GEGLU>(p, plan.slices, st);
    }
}

}  // namespace

// Types with the integer form, operands inside 32-bit byte offsets, blocks at even addresses; and where the other way (vmx_iq_dequant_int, then
// vmx_int_gemm_f32) is not as fast.  IQ3_XXS with the rows' conversion, that way / this one in us:  65 x 30720 x 3840 118 / 46, 256 162 / 76, 600 250 / 195,
// 2048 655 / 515;  200 x 3840 x 15360 75 / 52, 1500 231 / 208;  65 x 8192 x 3840 39 / 23, 2048 135 / 136;  65 x 2048 x 4096 31 / 20, 1000 41 / 40, 2048
// 59 / 63.  Of fewer than 8 M weights the other way writes and reads little and both are a handful of short launches: 65 x 512 x 2048 15 / 13, 400 x
// 1024 x 1024 16 / 15, 800 x 2048 x 2048 28.3 / 28.5, 800 x 512 x 8192 31 / 41.
bool vmx_iq_prompt_ok(const VmxMmvqSeg *segs, int nseg, int M, int K) {
    int64_t total = 0;
    for (int i = 0; i < nseg; i++) {
        if (!vmx_iq_int_form_ok(segs[i].ggml_type) || ((uintptr_t)segs[i].w & 1) || (int64_t)segs[i].n_out * (K / 256) * 128 >= (int64_t)1 << 32) return false;
        total += segs[i].n_out;
    }
    return (int64_t)M * K * 2 < (int64_t)1 << 32 && total * K >= (M < 2048 ? 8 << 20 : 24 << 20);
}

// Estimated ns of the other way on 128 x 128 tiles, two a compute unit: 2.4 bytes a weight at 4.3 TB/s (3.4 where 16 bits a weight are more than the caches
// keep) and a launch, then rounds of 1080 ns a 64-deep step (1280 in products of 280 steps and more, under which the clock falls; 700 with at most one tile a unit)
static int64_t dequantised_ns(int M, int64_t N, int K) {
    const int64_t tiles = (M + 127) / 128 * ((N + 127) / 128), places = 2 * vmx_num_cus(), steps = K / 64;
    const int64_t full = steps * (tiles * steps > 280 * places ? 1280 : 1080), rounds = tiles / places, rest = tiles % places;
    const int64_t last = rest == 0 ? 0 : rounds == 0 ? full * (4 * places + rest) / (5 * places) : full * (2 * places + 3 * rest) / (5 * places);
    return 4000 + N * K * (N * K > 64 << 20 ? 34 : 24) / 43000 + (tiles <= places / 2 ? steps * 700 : rounds * full + last) + M * N * 4 / 18400;
}

// vmx_iq_prompt_ok for a product that is called by itself.  With 128 x 128 tiles for four units of five the dequantised weight costs little and the other way's smaller
// tiles leave less of the last round empty, so the estimates decide (IQ3 codebooks take 4 % more than they say).  IQ3_XXS, weights out of HBM, that way / this one in us:  850 x
// 9216 x 3840 94 / 120, 2000 194 / 216;  1000 x 13862 x 3328 140 / 139, 2400 296 / 347;  1000 x 4096 x 4096 63 / 68, 1500 79 / 76;  2000 x 10240 x 5120 260 / 291;  but 1000 x
// 30720 x 3840 374 / 292, 1000 x 3840 x 15360 173 / 162.  Of 330 calls of 256 .. 4000 rows the estimates lose 0.4 % in the mean against the better way, always this way 1.5 %, always the
// other 10 %.  A model's prompt, whose norms add the slices, is faster without them: Gemma-4-12B (12 layers), 1000 tokens 8.57 ms, with the estimates 9.13; 2000 16.3 / 17.1.
bool vmx_iq_prompt_alone_ok(const VmxMmvqSeg &seg, int M, int K) {
    if (!vmx_iq_prompt_ok(&seg, 1, M, K)) return false;
    const int N = seg.n_out, tiles = (N + IQP_BN - 1) / IQP_BN;
    if (5 * ((int64_t)(M + 127) / 128 * tiles) < 4 * vmx_num_cus()) return true;
    const int64_t slices = (int64_t)(vmx_int_gemm_part_bytes() / ((size_t)M * N * 4));   // as many as the public workspace has room for
    const int64_t inside = iqp_plan(tiles, M, N, K / 256, slices).ns + (int64_t)M * N * 4 / 9200;
    return 100 * inside <= (seg.ggml_type == 18 || seg.ggml_type == 21 ? 96 : 100) * dequantised_ns(M, N, K);
}

// y[:, y_off of a segment ..] (f32, rows ldy apart) = a16 [M][K] times the segments' raw blocks, one product.  The segments' columns lie one behind the
// other from column 0 on.  part: scratch for slices, as many as fit part_bytes.  left: a reader that adds slices itself; *left = their count where they stay in part
// ([*left][M][ldy], rows without gaps), else 1 and the result is in y.
int vmx_iq_prompt_slices(const VmxMmvqSeg *segs, int nseg, const uint16_t *a16, float *y, int M, int K, int64_t ldy, float *part, size_t part_bytes, hipStream_t st,
                         int *left) {
    IqpArgs p = {};
    int tiles = 0, N = 0;
    for (int i = 0; i < nseg; i++) {
        p.seg[i] = IqpSeg{(const uint8_t *)segs[i].w, segs[i].ggml_type, segs[i].n_out, 0, N};
        tiles += (segs[i].n_out + IQP_BN - 1) / IQP_BN;
        N += segs[i].n_out;
    }
    p.nseg = nseg, p.A = a16, p.M = M, p.K = K;
    const IqpPlan plan = iqp_plan(tiles, M, N, K / 256, (int64_t)(part_bytes / ((size_t)M * N * 4)));
    p.C = plan.slices > 1 ? part : y, p.ldc = plan.slices > 1 ? N : ldy, p.slice_stride = (int64_t)M * N;
    if (int rc = iqp_launch_rows<false>(p, plan, st)) return rc;
    if (left) {
        *left = ldy == N ? plan.slices : 1;
        if (*left > 1) return VMX_OK;
    }
    return plan.slices > 1 ? vmx_int_slices(part, y, plan.slices, M, N, ldy, st) : VMX_OK;
}

int vmx_iq_prompt_f32(const VmxMmvqSeg *segs, int nseg, const uint16_t *a16, float *y, int M, int K, int64_t ldy, float *part, size_t part_bytes, hipStream_t st) {
    return vmx_iq_prompt_slices(segs, nseg, a16, y, M, K, ldy, part, part_bytes, st, nullptr);
}

// act16 [M][inter] (fp16) = GeGLU of gate and up, both of one type
int vmx_iq_prompt_geglu(const VmxMmvqSeg &gate, const VmxMmvqSeg &up, const uint16_t *a16, uint16_t *act, int M, int K, hipStream_t st) {
    IqpArgs p = {};
    p.seg[0] = IqpSeg{(const uint8_t *)gate.w, gate.ggml_type, gate.n_out, 0, 0};
    p.nseg = 1, p.w_up = (const uint8_t *)up.w, p.A = a16, p.act = act, p.M = M, p.K = K;
    return iqp_launch_rows<true>(p, iqp_plan((gate.n_out + 63) / 64, M, 2 * gate.n_out, K / 256, 1), st);
}
