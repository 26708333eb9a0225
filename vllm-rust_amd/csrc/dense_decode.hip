// Decode steps (up to 16 rows) of a layer whose projections are plain bf16 matrices W [N][K]: every projection is ONE launch that owns
// both sides of what would be kernel boundaries -- the RMSNorm of the residual stream or the merge of the attention partitions while
// its rows become matrix operands, and behind the sum the residual addition, the gated activation, or the f32 rows the attention reads.
// Such a step is a chain of short launches over weights that are read once (Qwen3-0.6B: 4 .. 13 MB each), so what bounds it is the
// latency of each link: the weights of a workgroup are requested before anything they wait for is computed, and no result is converted
// by a launch of its own.  Qwen3-0.6B at one row, 128 tokens: 12 launches and 43 us a layer as norm, GEMV, widening, activation kernels;
// 5 launches and 22 us now; the whole step 1269 -> 673 us.
#include "vmx_kernels.h"

namespace {

typedef uint32_t dd_u32x4 __attribute__((ext_vector_type(4)));

enum { DD_ROWS = 0, DD_NORM = 1, DD_MERGE = 2, DD_NORM_REG = 3 };   // where the rows come from (DD_NORM_REG: DD_NORM of rows too long for LDS)
enum { DD_F32 = 0, DD_RESID = 1, DD_GLU = 2 };          // what becomes of the sums

struct DenseDecode {
    const uint16_t *W, *x;          // x: bf16 rows [M][K] (DD_ROWS), the residual stream (DD_NORM)
    const uint16_t *norm_w;         // DD_NORM
    const float *ssq;               // DD_NORM: sums of squares of the stream's tiles, [M][tiles]
    float eps;
    int tiles;
    const float *part, *part_max, *part_sum;   // DD_MERGE: [M][K / head][P][head], [M][K / head][P] twice
    int P, head;
    float *y;                       // DD_F32: [M][N]
    uint16_t *h;                    // DD_RESID: stream [M][N], and the tiles' new sums of squares [M][N / CW]
    float *ssq_out;
    uint16_t *act;                  // DD_GLU: [M][N / 2]; rows [0, N / 2) of W are the gate, the others the up projection
    int M, N, K;
};

__device__ __forceinline__ dd_u32x4 dd_pack(const float (&f)[8]) {
    dd_u32x4 v;
#pragma unroll
    for (int e = 0; e < 4; e++) v[e] = (uint32_t)vmx_f32_to_bf16(f[2 * e]) | ((uint32_t)vmx_f32_to_bf16(f[2 * e + 1]) << 16);
    return v;
}
__device__ __forceinline__ void dd_unpack(dd_u32x4 v, float (&f)[8]) {
#pragma unroll
    for (int e = 0; e < 4; e++) {
        f[2 * e] = __uint_as_float(v[e] << 16);
        f[2 * e + 1] = __uint_as_float(v[e] & 0xFFFF0000u);
    }
}

constexpr int DD_STAGE = 16 * 1032;   // values that the norm and the merge stage in LDS at most: rows of K + 8

// A workgroup owns CW columns: 16, or for up to four rows of a narrow product 4 (dd_narrow; DD_GLU: half gate and the same up columns).  Lane
// (c = l & 15, g = l / 16) of v_mfma_f32_16x16x32_bf16 stands for column and row c % CW and for part c / CW of a block's k, so with
// four columns the tile's diagonal 4 x 4 squares are the partial sums of four parts of k and the others are not used: the matrix core
// idles anyway and the product has four times the workgroups (down of Qwen3-0.6B, [1024, 3072] at one row: 8.9 us in 64 workgroups
// of 16 columns, 4.8 in 256 of 4).  A wave takes the blocks w, w + NW, .. of 128 values a part; eight values feed one of four
// products; the four lanes g of a column read 64 consecutive bytes (as 16 bytes of four places 64 apart: gate|up 8.1 us, now 6.4).
// Rows that have to be normed or merged are worked out once per workgroup, spread over its threads, and staged in LDS: computed by
// each lane for its own operands, one live row of sixteen kept four lanes of a wave busy (q|k|v 6.7 -> 5.0 us, gate|up 9.1 -> 8.1).
// Their inputs come from the caches and are requested ahead of the weights of the first DEPTH blocks, because loads return in order.
// What the first requests need comes as arguments of its own, which are in registers when a wave starts (members of a struct are not): a step of Qwen3-0.6B at
// one row, 128 tokens, 821 -> 795 us, 0.2 us a launch.
template <int NW, int CW, int DEPTH, int SRC, int DST, int HELD, int SUMS>
__global__ __launch_bounds__(64 * NW) void dense_decode_kernel(const uint16_t *W, const void *first, const void *second, const void *third, int M, int N, int K,
                                                                int fourth, const DenseDecode rest) {
    DenseDecode p = rest;
    p.W = W, p.M = M, p.N = N, p.K = K;
    if constexpr (SRC == DD_MERGE) p.part = static_cast<const float *>(first), p.part_max = static_cast<const float *>(second), p.part_sum = static_cast<const float *>(third), p.P = fourth;
    else p.x = static_cast<const uint16_t *>(first), p.norm_w = static_cast<const uint16_t *>(second), p.ssq = static_cast<const float *>(third), p.tiles = fourth;
    constexpr int PARTS = 16 / CW, DEEP = 128 * PARTS;
    constexpr bool STAGED = SRC == DD_NORM || SRC == DD_MERGE, NORM = SRC == DD_NORM || SRC == DD_NORM_REG;
    __shared__ float red[NW * SUMS][64][4];
    __shared__ __align__(16) uint16_t rows_lds[STAGED ? DD_STAGE : 8];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), c = lane & (CW - 1), part = (lane & 15) / CW, g = lane >> 4, nt = blockIdx.x;
    const int nblk = (K + DEEP - 1) / DEEP, row = min(c, p.M - 1);
    const uint16_t *wrow = p.W + (int64_t)(DST == DD_GLU ? (c < CW / 2 ? 0 : p.N / 2) + nt * (CW / 2) + (c & (CW / 2 - 1)) : nt * CW + c) * K;
    const uint16_t *idle = p.W + (int64_t)nt * (DST == DD_GLU ? CW / 2 : CW) * K;   // of the workgroup's own rows: a place for all of them is one channel of the L2
    const int k0 = 128 * part + 8 * g;
    // Requests lie behind no condition of a lane (the compiler waits for each before the next) and none that makes them more or fewer before a wait: what lies past K reads
    // the last values again and is cleared before the product, rows past M repeat the last one and are not stored.  A wave without a first or a second block takes a way of
    // its own; where a barrier stands between (staged rows) it reads one place instead, of the workgroup's own weights: the same for all workgroups is one channel of
    // the L2, in which they queue, and one in every lane's own row cost down at 16 rows 8.9 -> 10.9 us.
    // Of several rows what has to be normed and its statistic come ahead of the weights, HELD pieces a thread (dd_launch_norm).
    dd_u32x4 w[DEPTH][4], xr[DEPTH][4], nr[DEPTH][SRC == DD_NORM_REG ? 4 : 1];
    auto load_w = [&](int b, dd_u32x4 (&d)[4]) {
#pragma unroll
        for (int j = 0; j < 4; j++) d[j] = __builtin_nontemporal_load(reinterpret_cast<const dd_u32x4 *>(!STAGED || b < nblk ? wrow + min(DEEP * b + k0 + 32 * j, K - 8) : idle));
    };
    auto load_rows = [&](int b, dd_u32x4 (&x)[4], dd_u32x4 (&n)[SRC == DD_NORM_REG ? 4 : 1]) {
        if constexpr (!STAGED) {
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int k = min(DEEP * b + k0 + 32 * j, K - 8);
                x[j] = *reinterpret_cast<const dd_u32x4 *>(p.x + (int64_t)row * K + k);
                if constexpr (SRC == DD_NORM_REG) n[j] = *reinterpret_cast<const dd_u32x4 *>(p.norm_w + k);
            }
        }
    };
    // staged rows: a thread works out eight consecutive values of a row at a time
    const int chunks = STAGED ? p.M * (K / 8) : 0, chunk0 = min(tid, chunks - 1);
    float4 lo[4], hi[4];
    float most[4], total[4];
    const float per_row = __builtin_amdgcn_rcpf((float)(K / 8));
    auto row_of = [&](int i) { return (int)(((float)i + 0.5f) * per_row); };   // i / (K / 8): of at most DD_STAGE / 8 places and 16 rows, so far closer than half a place
    auto load_parts = [&](int i) {
        const int m = row_of(i), k = (i - m * (K / 8)) * 8;
        const int64_t at = ((int64_t)m * (K / p.head) + k / p.head) * p.P;
#pragma unroll
        for (int q = 0; q < 4; q++) {   // partitions past P read the last one again; their weight is zero below
            const int64_t from = at + min(q, p.P - 1);
            const float4 *src = reinterpret_cast<const float4 *>(p.part + from * p.head + k % p.head);
            lo[q] = src[0], hi[q] = src[1], most[q] = p.part_max[from], total[q] = p.part_sum[from];
        }
    };
    auto merge_parts = [&](int i) {
        float top = -3.402823466e+38f, sum = 0.f, f[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int q = 0; q < 4; q++) top = fmaxf(top, q < p.P ? most[q] : -3.402823466e+38f);
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const float wt = q < p.P ? total[q] * __expf(most[q] - top) : 0.f;
            sum += wt;
            f[0] += lo[q].x * wt, f[1] += lo[q].y * wt, f[2] += lo[q].z * wt, f[3] += lo[q].w * wt;
            f[4] += hi[q].x * wt, f[5] += hi[q].y * wt, f[6] += hi[q].z * wt, f[7] += hi[q].w * wt;
        }
        const float scale = 1.0f / (sum + 1e-6f);
#pragma unroll
        for (int e = 0; e < 8; e++) f[e] *= scale;
        const int m = row_of(i);
        *reinterpret_cast<dd_u32x4 *>(&rows_lds[m * (K + 8) + (i - m * (K / 8)) * 8]) = dd_pack(f);
    };

    // DD_NORM: the wave's lanes share the tiles' sums of its rows out (lane % rows is the row, as it is for c)
    const int row_bits = p.M <= 1 ? 0 : p.M <= 2 ? 1 : p.M <= 4 ? 2 : p.M <= 8 ? 3 : 4, rows = 1 << row_bits, quads = NORM ? p.tiles / 4 : 1;
    const float4 *tile = NORM ? reinterpret_cast<const float4 *>(p.ssq + (int64_t)min(lane & (rows - 1), p.M - 1) * p.tiles) : nullptr;
    float4 t0;
    dd_u32x4 xs[HELD], ns[HELD];
    if constexpr (NORM) t0 = tile[min(lane >> row_bits, quads - 1)];
    float4 tq[HELD];
    if constexpr (SRC == DD_NORM) {
        auto request = [&](int u) {
            const bool some = 64 * NW * u + 64 * wave < chunks;   // of the wave's
            const int at = min(tid + 64 * NW * u, chunks - 1);
            xs[u] = *reinterpret_cast<const dd_u32x4 *>(some ? p.x + (int64_t)at * 8 : p.x);
            ns[u] = *reinterpret_cast<const dd_u32x4 *>(some ? p.norm_w + (at - row_of(at) * (K / 8)) * 8 : p.norm_w);
        };
        request(0);
        if (HELD > 1 && p.M > 1) {   // always where HELD > 1 (dd_launch_norm); as a branch it keeps the compiler from 20 registers more
#pragma unroll
            for (int u = 1; u < HELD; u++) tq[u] = tile[min((lane >> row_bits) + u * (64 >> row_bits), quads - 1)], request(u);
        }
    }
    if constexpr (SRC == DD_MERGE) load_parts(chunk0);
    // DD_RESID: the thread's value of the stream, which the end waits for
    const int om = CW == 16 ? (tid >> 4) & 15 : (tid >> 2) & 3, on = tid & (CW - 1);
    const int64_t out_at = (int64_t)min(om, p.M - 1) * p.N + nt * CW + on;
    uint16_t hold = 0;
    auto request_hold = [&] {
        if constexpr (DST == DD_RESID) hold = p.h[out_at];
    };
    if constexpr (STAGED) {
#pragma unroll
        for (int d = 0; d < DEPTH; d++) load_w(wave + d * NW, w[d]);
        request_hold();
    }
    float inv = 0.f;
    auto statistic = [&] {
        if constexpr (!NORM) return;
        float sq = lane >> row_bits < quads ? (t0.x + t0.y) + (t0.z + t0.w) : 0.f;
#pragma unroll
        for (int u = 1; u < HELD; u++) sq += (lane >> row_bits) + u * (64 >> row_bits) < quads ? (tq[u].x + tq[u].y) + (tq[u].z + tq[u].w) : 0.f;
        for (int i = (lane >> row_bits) + HELD * (64 >> row_bits); i < quads; i += 64 >> row_bits) {
            const float4 v = tile[i];
            sq += (v.x + v.y) + (v.z + v.w);
        }
        if (rows <= 1) sq += vmx_lane_xor<1>(sq);
        if (rows <= 2) sq += vmx_lane_xor<2>(sq);
        if (rows <= 4) sq += vmx_lane_xor<4>(sq);
        if (rows <= 8) sq += vmx_lane_xor<8>(sq);
        sq += vmx_lane_xor<16>(sq);
        sq += vmx_lane_xor<32>(sq);
        inv = rsqrtf(sq / (float)K + p.eps);
    };
    if constexpr (STAGED) statistic();
    auto norm8 = [&](dd_u32x4 x, dd_u32x4 n, float by) {
        float f[8], gain[8];
        dd_unpack(x, f);
        dd_unpack(n, gain);
#pragma unroll
        for (int e = 0; e < 8; e++) f[e] = f[e] * by * gain[e];
        return dd_pack(f);
    };
    if constexpr (SRC == DD_NORM) {
        auto stage = [&](int i, dd_u32x4 x, dd_u32x4 n) {   // whole waves: the statistic of a row is held by the lane of its number
            const int at = min(i, chunks - 1), m = row_of(at);
            const float by = __shfl(inv, m);
            if (i < chunks) *reinterpret_cast<dd_u32x4 *>(&rows_lds[m * (K + 8) + (at - m * (K / 8)) * 8]) = norm8(x, n, by);
        };
#pragma unroll
        for (int u = 0; u < HELD; u++)
            if (64 * NW * u + 64 * wave < chunks) stage(tid + 64 * NW * u, xs[u], ns[u]);
        for (int i = tid + 64 * NW * HELD; i - lane < chunks; i += 64 * NW) {
            const int at = min(i, chunks - 1), m = row_of(at);
            stage(i, *reinterpret_cast<const dd_u32x4 *>(p.x + (int64_t)at * 8), *reinterpret_cast<const dd_u32x4 *>(p.norm_w + (at - m * (K / 8)) * 8));
        }
    }
    if constexpr (SRC == DD_MERGE) {
        if (tid < chunks) merge_parts(tid);
        for (int i = tid + 64 * NW; i < chunks; i += 64 * NW) {
            load_parts(i);
            merge_parts(i);
        }
    }
    if constexpr (STAGED) __syncthreads();
    vmx_f32x4 acc[SUMS];
#pragma unroll
    for (int i = 0; i < SUMS; i++) acc[i] = vmx_f32x4{0.f, 0.f, 0.f, 0.f};
    auto step = [&](int b, dd_u32x4 (&d)[4], dd_u32x4 (&x)[4], dd_u32x4 (&n)[SRC == DD_NORM_REG ? 4 : 1], vmx_f32x4 &sum) {
        const bool past = DEEP * (b + 1) > K;   // the wave's
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int k = DEEP * b + k0 + 32 * j;
            dd_u32x4 a = x[j], v = d[j];
            if constexpr (SRC == DD_NORM_REG) a = norm8(a, n[j], inv);
            else if constexpr (STAGED) a = *reinterpret_cast<const dd_u32x4 *>(&rows_lds[row * (K + 8) + min(k, K - 8)]);
            if (past && k >= K) a = v = dd_u32x4{0, 0, 0, 0};
            sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(vmx_bf16x8, a), __builtin_bit_cast(vmx_bf16x8, v), sum, 0, 0, 0);
        }
    };
    if (DEPTH > 1 && wave + NW < nblk) {
        constexpr int L = DEPTH - 1;
        if constexpr (!STAGED) {
            load_rows(wave, xr[0], nr[0]);
            load_rows(wave + NW, xr[L], nr[L]);
            load_w(wave, w[0]);
            load_w(wave + NW, w[L]);
            if constexpr (SRC == DD_ROWS && HELD > 1) __builtin_amdgcn_sched_barrier(0);
            request_hold();
            statistic();
        }
        for (int b = wave; b < nblk; b += 2 * NW) {
            step(b, w[0], xr[0], nr[0], acc[0]);
            if (b + 2 * NW < nblk) load_w(b + 2 * NW, w[0]), load_rows(b + 2 * NW, xr[0], nr[0]);
            if (b + NW < nblk) step(b + NW, w[L], xr[L], nr[L], acc[SUMS - 1]);
            if (b + 3 * NW < nblk) load_w(b + 3 * NW, w[L]), load_rows(b + 3 * NW, xr[L], nr[L]);
        }
    } else {   // one block or none
        if (!STAGED && wave < nblk) load_rows(wave, xr[0], nr[0]), load_w(wave, w[0]);
        if constexpr (!STAGED) {
            if constexpr (SRC == DD_ROWS && HELD > 1) __builtin_amdgcn_sched_barrier(0);
            request_hold();
            statistic();
        }
        if (wave < nblk) step(wave, w[0], xr[0], nr[0], acc[0]);
    }
#pragma unroll
    for (int i = 0; i < SUMS; i++)
#pragma unroll
        for (int r = 0; r < 4; r++) red[wave + NW * i][lane][r] = acc[i][r];
    __syncthreads();
    if (tid >= (CW == 4 ? 64 : 256)) return;
    // CW 16: thread -> row tid / 16, column tid % 16 (element (4 g + r, c) of a tile sits with lane 16 g + c); CW 4: thread -> part
    // tid / 16, row tid / 4 % 4, column tid % 4, the square of part i at rows and columns 4 i ..
    const int m = om, n = on;
    const int from = CW == 16 ? (m >> 2) * 16 + n : (tid >> 4) * 20 + n, r = m & 3;
    float v = 0.f;
#pragma unroll
    for (int i = 0; i < NW * SUMS; i++) v += red[i][from][r];
    if constexpr (CW == 4) {
        v += vmx_lane_xor<16>(v);
        v += vmx_lane_xor<32>(v);
    }
    const bool keep = m < p.M && (CW == 16 || tid < 16);
    if constexpr (DST == DD_F32) {
        if (keep) p.y[(int64_t)m * p.N + nt * CW + n] = v;
    } else if constexpr (DST == DD_GLU) {
        const float up = vmx_lane_xor<CW / 2>(v);
        if (keep && n < CW / 2) {
            const float gg = vmx_bf16_to_f32(vmx_f32_to_bf16(v)), uu = vmx_bf16_to_f32(vmx_f32_to_bf16(up));
            p.act[(int64_t)m * (p.N / 2) + nt * (CW / 2) + n] = vmx_f32_to_bf16((gg / (1.0f + expf(-gg))) * uu);
        }
    } else {
        const uint16_t hn = vmx_f32_to_bf16(vmx_bf16_to_f32(hold) + vmx_bf16_to_f32(vmx_f32_to_bf16(v)));
        const float f = vmx_bf16_to_f32(hn);
        float s = f * f;
        s += vmx_lane_xor<1>(s);
        s += vmx_lane_xor<2>(s);
        if constexpr (CW == 16) {
            s += vmx_lane_xor<4>(s);
            s += vmx_lane_xor<8>(s);
        }
        if (keep) {
            p.h[out_at] = hn;
            if (n == 0) p.ssq_out[m * (p.N / CW) + nt] = s;
        }
    }
}

template <int CW, int SRC, int DST, int HELD = 1>
int dd_launch(const DenseDecode &p, hipStream_t st) {
    const int nblk = (p.K + 128 * (16 / CW) - 1) / (128 * (16 / CW));
    constexpr bool eight = SRC == DD_NORM || SRC == DD_NORM_REG;   // waves at most
    const dim3 grid((unsigned)(p.N / CW));
    const void *first = p.x, *second = p.norm_w, *third = p.ssq;
    int fourth = p.tiles;
    if (SRC == DD_MERGE) first = p.part, second = p.part_max, third = p.part_sum, fourth = p.P;
    if (nblk <= 4) hipLaunchKernelGGL((dense_decode_kernel<4, CW, 1, SRC, DST, HELD, 1>), grid, dim3(256), 0, st, p.W, first, second, third, p.M, p.N, p.K, fourth, p);
    else if (nblk <= 8) hipLaunchKernelGGL((dense_decode_kernel<8, CW, 1, SRC, DST, HELD, 1>), grid, dim3(512), 0, st, p.W, first, second, third, p.M, p.N, p.K, fourth, p);
    else if (nblk <= 16 || SRC == DD_NORM_REG) hipLaunchKernelGGL((dense_decode_kernel<8, CW, 2, SRC, DST, HELD, 1>), grid, dim3(512), 0, st, p.W, first, second, third, p.M, p.N, p.K, fourth, p);
    else hipLaunchKernelGGL((dense_decode_kernel<eight ? 8 : 16, CW, 2, SRC, DST, HELD, SRC == DD_NORM ? 2 : 1>), grid, dim3(eight ? 512 : 1024), 0, st, p.W, first, second, third, p.M, p.N, p.K, fourth, p);
    VMX_CHECK_LAUNCH("dense_decode");
    return VMX_OK;
}

// The pieces of eight values that a thread of the normed forms requests ahead are registers of every wave: with room for four whatever the rows a compute unit held two
// workgroups (one of 16 waves) where it has LDS for three, and wide products lost by it.  So one and two pieces have forms of their own (72 and 76 registers instead of 93), and
// eight waves walk any K (16 waves of more than 64 registers are one workgroup; beyond 16 blocks a wave keeps the sums of 16 waves' blocks apart: the same bits).  Four pieces: more than two there are, or of many workgroups more than three (steps of
// width 1536, 17920 gate|up columns, 6 / 8 / 10 rows, two or four pieces 604 633 681 / 614 635 669 us; 2048, 12288 columns, 8 rows 552 / 520).
// Steps of 4 .. 12 such layers, 200 tokens, loads behind conditions / four pieces and 16 waves / now, us, 1 2 4 8 16 rows, width (gate|up columns):
//    896 (9728): 320 332 379 468 530 / 312 337 374 474 514 / 279 307 354 441 499;    1024 (6144): 316 337 389 424 488 / 276 312 350 432 461 / 272 308 357 399 453
//    1536 (17920): 443 480 552 638 830 / 464 492 577 637 789 / 436 470 546 636 778;  2048 (12288): 396 432 502 548 694 / 398 407 486 520 663 / 379 414 469 520 659
//    2560 (19456): 424 447 498 613 718 / 455 511 559 568 687 / 411 435 486 567 676;  4096 (24576): 420 445 503 602 722 / 438 485 523 553 658 / 409 430 470 554 656
template <int DST> int dd_launch_norm(const DenseDecode &p, hipStream_t st) {
    if (p.M * (p.K + 8) > DD_STAGE) return dd_launch<16, DD_NORM_REG, DST>(p, st);
    const int threads = p.K <= 512 ? 256 : 512, pieces = (p.M * (p.K / 8) + threads - 1) / threads;
    if (p.M > 1 && pieces > (p.K > 1024 && p.N / 16 > 4 * vmx_num_cus() ? 3 : 2)) return dd_launch<16, DD_NORM, DST, 4>(p, st);
    return pieces == 1 || p.M == 1 ? dd_launch<16, DD_NORM, DST, 1>(p, st) : dd_launch<16, DD_NORM, DST, 2>(p, st);
}

// Four columns a workgroup where sixteen would leave half of the compute units or more without one: each workgroup norms or merges all rows for
// itself, so rows times workgroups is bounded too.  us a layer (300 tokens, 100 for one row), sixteen / four columns for o and down:  hidden size 896, four
// rows 38.1 / 35.7;  1024, one row 31.0 / 27.2, four 37.0 / 35.2;  1536, two 55.1 / 50.7, four 59.8 / 61.2;  2048, one 48.6 / 44.6, two 49.9 / 46.4, four
// 55.1 / 55.7;  2560, one 76.6 / 77.2, two 77.9 / 83.4, four 87.0 / 112.5 (104.7 as twelve launches);  3072, one 73.3 / 77.0, four 82.6 / 106.5;  3584, two
// 115.7 / 135.4, four 128.8 / 180.8.
bool dd_narrow(int M, int N) {
    const int cus = vmx_num_cus(), wide = N / 16;
    return M <= 4 && wide <= cus / 2 && M * wide <= cus;
}

}  // namespace

// A product of N columns over K: whole 16-column tiles, 16-byte rows
bool vmx_dense_decode_ok(int M, int N, int K) { return M >= 1 && M <= 16 && N % 16 == 0 && K % 16 == 0; }

// Sums of squares per row that vmx_dense_decode_resid leaves
int vmx_dense_decode_tiles(int M, int N) { return N / (dd_narrow(M, N) ? 4 : 16); }

int vmx_dense_decode_f32(float *y, const uint16_t *x, const uint16_t *W, int M, int N, int K, hipStream_t st) {
    DenseDecode p{};
    p.W = W, p.x = x, p.y = y, p.M = M, p.N = N, p.K = K;
    // requests all made before the products (HELD > 1), or with the compiler's own order: 16 rows [4096, 1024] 4.2 / 4.4 us, [1024, 2304] 6.5 / 7.1; one 3.8 / 3.6, 5.6 / 5.4
    return M > 8 ? dd_launch<16, DD_ROWS, DD_F32, 2>(p, st) : dd_launch<16, DD_ROWS, DD_F32>(p, st);
}

// y = rms_norm(h) W^T; ssq: what vmx_dense_decode_resid left for h
int vmx_dense_decode_norm_f32(float *y, const uint16_t *h, const uint16_t *norm_w, float eps, const float *ssq, int tiles, const uint16_t *W, int M,
                              int N, int K, hipStream_t st) {
    DenseDecode p{};
    p.W = W, p.x = h, p.norm_w = norm_w, p.eps = eps, p.ssq = ssq, p.tiles = tiles, p.y = y, p.M = M, p.N = N, p.K = K;
    return dd_launch_norm<DD_F32>(p, st);
}

// act [M][N / 2] = silu(gate) * up of rms_norm(h) W^T
int vmx_dense_decode_norm_glu(uint16_t *act, const uint16_t *h, const uint16_t *norm_w, float eps, const float *ssq, int tiles, const uint16_t *W, int M,
                              int N, int K, hipStream_t st) {
    DenseDecode p{};
    p.W = W, p.x = h, p.norm_w = norm_w, p.eps = eps, p.ssq = ssq, p.tiles = tiles, p.act = act, p.M = M, p.N = N, p.K = K;
    return dd_launch_norm<DD_GLU>(p, st);
}

bool vmx_dense_decode_merge_ok(int M, int K, int head_dim, int parts) {
    return M <= 4 && M * (K + 8) <= DD_STAGE && parts >= 1 && parts <= 4 && head_dim % 8 == 0 && K % head_dim == 0;
}

// h += x W^T (x the merged attention partitions if `parts`), ssq [M][vmx_dense_decode_tiles] = sums of squares of the new h's tiles
int vmx_dense_decode_resid(uint16_t *h, float *ssq, const uint16_t *x, const VmxAttnParts *parts, int head_dim, const uint16_t *W, int M, int N, int K,
                           hipStream_t st) {
    DenseDecode p{};
    p.W = W, p.x = x, p.h = h, p.ssq_out = ssq, p.M = M, p.N = N, p.K = K;
    const bool narrow = dd_narrow(M, N);
    if (!parts) return narrow ? dd_launch<4, DD_ROWS, DD_RESID>(p, st) : dd_launch<16, DD_ROWS, DD_RESID>(p, st);
    VMX_REQUIRE(vmx_dense_decode_merge_ok(M, K, head_dim, parts->max_parts), "dense_decode: partitions not covered");
    p.part = parts->tmp_out, p.part_max = parts->max_logits, p.part_sum = parts->exp_sums, p.P = parts->max_parts, p.head = head_dim;
    return narrow ? dd_launch<4, DD_MERGE, DD_RESID>(p, st) : dd_launch<16, DD_MERGE, DD_RESID>(p, st);
}
