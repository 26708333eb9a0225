// Latent attention over a paged cache of compressed keys/values.
//
// A token's cache row is [c | k_rot]: the RMS-normed latent c (kv_rank values) from which every head's unrotated key and value
// are linear maps (k_h = U_h c, v_h = V_h c), and one rotated key part (rot_dim values) shared by all heads.  The up-projections
// are never applied to the cache: with qa_h = U_h^T q_h (done by the caller as a batched product) the score of head h against
// key j is (qa_h . c_j + qr_h . k_rot_j) * scale, and the head's output is V_h (sum_j p_j c_j), so the kernel here works in the
// latent space -- every head reads the same cache rows -- and the caller applies V_h to its result.
//
// Parameters rather than constants: window (position i sees j with 0 <= i - j < window; 0 = unbounded causal), an optional
// per-head sink logit (a key-less term exp(sink_h) in the softmax denominator, not scaled), the rotation (interleaved pairs
// (2i, 2i+1) or halves (i, i + rot_dims / 2) of the first rot_dims dimensions, angle = position * inv_freq[i], cos and sin times a
// constant), queries straight from the input or through an RMS-normed latent of their own, sizes, cache element type (bf16 / f32).
// Layers may attend over another layer's cache: preparation then skips the key/value part.
// Scores, softmax, the weighted sum, norms and angles are f32.  Queries are packed: token t belongs to sequence seq_ids[t] at
// position positions[t], so prompts of different lengths, prompt portions and single decode tokens are the same launch.  A
// token's result depends only on its own query and the cache rows of its window, beyond rounding: how its keys are cut into partitions and tiles, and so the order of
// its sums, depends on how many row tiles the launch has and on whether those beside its own belong to its sequence.  (With fewer than 16 heads a row tile
// holds several tokens; an infinity or a NaN in the cache row of one reaches the others of its tile.)
#include "tile_gemm.h"
#include "vmx_kernels.h"
#include <float.h>
#include <limits.h>

namespace {

template <bool F32> __device__ __forceinline__ float ld_cache(const void *c, int64_t i) {
    if constexpr (F32) return ((const float *)c)[i];
    else return vmx_bf16_to_f32(((const uint16_t *)c)[i]);
}
template <bool F32> __device__ __forceinline__ void st_cache(void *c, int64_t i, float v) {
    if constexpr (F32) ((float *)c)[i] = v;
    else ((uint16_t *)c)[i] = vmx_f32_to_bf16(v);
}

struct LatentPrepareArgs {
    vmx_latent_prepare p;
    const int32_t *positions, *slots;
    void *cache, *q_latent_out;
};

// One workgroup per token, any of three parts (a part without its input pointer is skipped):
//   q_latent: RMS-normed row of the query's latent -> q_latent_out (the element type of the cache);
//   kv:       c = rms_norm(kv[:R]) * w, k_rot = rotate(kv[R:]) -> cache row `slot`;
//   q:        rotate(q_h[dim:]) -> q_rot.
template <bool F32> __global__ __launch_bounds__(256) void latent_prepare_kernel(const LatentPrepareArgs a) {
    __shared__ float red[4];
    __shared__ float2 turn[128];     // cos and sin of the token's angles, shared by all heads
    const vmx_latent_prepare &p = a.p;
    const int t = blockIdx.x, tid = threadIdx.x;
    const float pos = (float)a.positions[t];
    if (p.q_latent) {
        const float *row = p.q_latent + (int64_t)t * p.ldq_latent;
        float ss = 0.f;
        for (int i = tid; i < p.q_rank; i += 256) ss = fmaf(row[i], row[i], ss);
        ss = vmx_block_sum_256(ss, red);
        const float inv = 1.0f / sqrtf(ss / (float)p.q_rank + p.eps);
        for (int i = tid; i < p.q_rank; i += 256)
            st_cache<F32>(a.q_latent_out, (int64_t)t * p.q_rank + i, row[i] * inv * vmx_bf16_to_f32(p.q_latent_norm_bf16[i]));
    }
    const int R = p.kv_rank, rd = p.rot_dim, half = p.rot_dims >> 1, nq = p.q ? p.heads : 0;
    const float *kv = p.kv ? p.kv + (int64_t)t * p.ldkv : nullptr;
    const int64_t slot = kv ? a.slots[t] : -1;
    const int64_t cbase = slot * (R + rd);
    if (kv) {
        float ss = 0.f;
        for (int i = tid; i < R; i += 256) ss += kv[i] * kv[i];
        ss = vmx_block_sum_256(ss, red);
        const float inv = 1.0f / sqrtf(ss / (float)R + p.eps);
        if (slot >= 0)
            for (int i = tid; i < R; i += 256) st_cache<F32>(a.cache, cbase + i, kv[i] * inv * vmx_bf16_to_f32(p.latent_norm_bf16[i]));
    }
    if (!kv && !nq) return;
    auto angle = [&](int i) {
        float sn, cs;
        sincosf(pos * p.inv_freq[i], &sn, &cs);
        return make_float2(cs * p.rot_mul, sn * p.rot_mul);
    };
    for (int i = tid; i < min(half, 128); i += 256) turn[i] = angle(i);
    __syncthreads();
    // rotations: work item = (vector v, pair i); vector 0 is the shared key part, vector 1 + h the rotated part of head h's query
    const int v0 = slot >= 0 ? 0 : 1;
    for (int w = tid + v0 * half; w < (nq + 1) * half; w += 256) {
        const int v = w / half, i = w % half;
        const float2 cs = i < 128 ? turn[i] : angle(i);
        const float *src = v == 0 ? kv + R : p.q + (int64_t)t * p.ldq + (int64_t)(v - 1) * (p.dim + rd) + p.dim;
        const int ia = p.rot_halves ? i : 2 * i, ib = p.rot_halves ? i + half : 2 * i + 1;
        const float x = src[ia], y = src[ib];
        const float rx = x * cs.x - y * cs.y, ry = y * cs.x + x * cs.y;
        if (v == 0) {
            st_cache<F32>(a.cache, cbase + R + ia, rx);
            st_cache<F32>(a.cache, cbase + R + ib, ry);
        } else {
            float *dst = p.q_rot + ((int64_t)t * nq + (v - 1)) * rd;
            dst[ia] = rx;
            dst[ib] = ry;
        }
    }
    // dimensions past rot_dims pass unchanged
    const int rest = rd - p.rot_dims;
    for (int w = tid + v0 * rest; w < (nq + 1) * rest; w += 256) {
        const int v = w / rest, i = p.rot_dims + w % rest;
        if (v == 0) st_cache<F32>(a.cache, cbase + R + i, kv[R + i]);
        else p.q_rot[((int64_t)t * nq + (v - 1)) * rd + i] = p.q[(int64_t)t * p.ldq + (int64_t)(v - 1) * (p.dim + rd) + p.dim + i];
    }
}

// out[h][r][d] = in[h][d][r]: the key up-projection as [head][latent][dim], so that qa_h = U_h^T q_h reads its weights along k
__global__ __launch_bounds__(256) void transpose_heads_kernel(uint16_t *__restrict__ out, const uint16_t *__restrict__ in, int H, int D, int R) {
    const int64_t n = (int64_t)H * D * R;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
        const int64_t h = i / ((int64_t)D * R), rem = i % ((int64_t)D * R);
        const int r = (int)(rem / D), d = (int)(rem % D);
        out[i] = in[(h * D + d) * R + r];
    }
}

// One workgroup per (head, token).  Keys are walked 256 at a time: thread i scores key i of the chunk (a whole cache row against
// the query held in LDS), the chunk's maximum and sum update the running softmax, then wave w adds keys w, w + 4, ... of the chunk
// into its lanes' latent dimensions; the four waves are summed at the end.
template <bool F32>
__global__ __launch_bounds__(256) void latent_attn_kernel(float *__restrict__ out, const float *__restrict__ q_abs,
                                                           const float *__restrict__ q_rot, const void *__restrict__ cache,
                                                           const int32_t *__restrict__ block_tables, int max_blocks,
                                                           const int32_t *__restrict__ seq_ids, const int32_t *__restrict__ positions,
                                                           const uint16_t *__restrict__ sink, float scale, int window, int H, int R, int rd,
                                                           int block_size) {
    extern __shared__ float sm[];
    const int RW = R + rd;
    float *qs = sm;                 // [R + rd]
    float *ps = qs + RW;            // [256]
    int32_t *ks = (int32_t *)(ps + 256);   // [256] cache slots of the chunk's keys
    float *red = (float *)(ks + 256);      // [8]
    float *part = red + 8;          // [4][R]
    const int h = blockIdx.x, t = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int pos = positions[t];
    const int32_t *bt = block_tables + (int64_t)seq_ids[t] * max_blocks;
    const int lo = window > 0 ? max(0, pos - window + 1) : 0;
    const int n = pos - lo + 1;
    for (int i = tid; i < R; i += 256) qs[i] = q_abs[((int64_t)t * H + h) * R + i];
    for (int i = tid; i < rd; i += 256) qs[R + i] = q_rot[((int64_t)t * H + h) * rd + i];
    constexpr int MAXD = 8;         // latent dimensions per lane: R <= 512
    float acc[MAXD];
#pragma unroll
    for (int i = 0; i < MAXD; i++) acc[i] = 0.f;
    // the sink enters as a key-less term: running maximum m = sink, running sum l = exp(sink - m) = 1
    float m = sink ? vmx_bf16_to_f32(sink[h]) : -FLT_MAX, l = sink ? 1.f : 0.f;
    __syncthreads();
    for (int c0 = 0; c0 < n; c0 += 256) {
        const bool valid = c0 + tid < n;
        float s = -FLT_MAX;
        if (valid) {
            const int j = lo + c0 + tid;
            const int slot = bt[j / block_size] * block_size + j % block_size;
            ks[tid] = slot;
            const int64_t base = (int64_t)slot * RW;
            float d = 0.f;
            if constexpr (!F32) {
                if ((RW & 7) == 0) {
                    const uint4 *r8 = reinterpret_cast<const uint4 *>((const uint16_t *)cache + base);
                    for (int i = 0; i < (RW >> 3); i++) {
                        float f[8];
                        vmx_unpack16x8<false>(r8[i], f);
#pragma unroll
                        for (int e = 0; e < 8; e++) d = fmaf(qs[8 * i + e], f[e], d);
                    }
                } else {
                    for (int i = 0; i < RW; i++) d = fmaf(qs[i], ld_cache<F32>(cache, base + i), d);
                }
            } else {
                for (int i = 0; i < RW; i++) d = fmaf(qs[i], ld_cache<F32>(cache, base + i), d);
            }
            s = d * scale;
        }
        float cm = vmx_wave_max(s);
        if (lane == 0) red[wave] = cm;
        __syncthreads();
        cm = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
        const float m_new = fmaxf(m, cm);
        const float p = valid ? expf(s - m_new) : 0.f;
        ps[tid] = p;
        float cs = vmx_wave_sum(p);
        if (lane == 0) red[4 + wave] = cs;
        __syncthreads();
        cs = (red[4] + red[5]) + (red[6] + red[7]);
        const float alpha = expf(m - m_new);   // m == -FLT_MAX only before the first chunk without a sink: l and acc are 0 then
        l = l * alpha + cs;
        m = m_new;
#pragma unroll
        for (int i = 0; i < MAXD; i++) acc[i] *= alpha;
        const int cn = min(256, n - c0);
        for (int kk = wave; kk < cn; kk += 4) {
            const float pk = ps[kk];
            const int64_t base = (int64_t)ks[kk] * RW;
#pragma unroll
            for (int i = 0; i < MAXD; i++) {
                const int d = lane + 64 * i;
                if (d < R) acc[i] = fmaf(pk, ld_cache<F32>(cache, base + d), acc[i]);
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < MAXD; i++) {
        const int d = lane + 64 * i;
        if (d < R) part[wave * R + d] = acc[i];
    }
    __syncthreads();
    const float inv = l > 0.f ? 1.0f / l : 0.f;
    for (int d = tid; d < R; d += 256)
        out[((int64_t)t * H + h) * R + d] = ((part[d] + part[R + d]) + (part[2 * R + d] + part[3 * R + d])) * inv;
}

// ---------------------------------------------------------------------------------------------------------------------------
// Matrix-core form (bf16 cache).  A workgroup owns a ROW TILE: 16 (token, head) rows = TPT consecutive tokens x HPT heads, which
// share their keys because the heads of a token read the same cache rows; with 16 or more heads a tile is one token, so decode
// steps fill the matrix instruction as well as prompts do.  Keys are walked in tiles of 64:
//   S = Q K^T     wave w takes keys 16 w .. 16 w + 15 of the tile: Q fragments (the latent-space query | rotated part, rounded to
//                 bf16) stay in registers, key fragments come straight from the cache rows; v_mfma_f32_16x16x32_bf16 leaves lane
//                 (g, n) the scores of rows 4 g .. 4 g + 3 against key n, so a row's maximum and sum are DPP reductions over 16 lanes
//                 plus one exchange between the four waves through LDS;
//   O += P C      the key fragments a wave already holds also go row-major into LDS (one 16-byte write per fragment; the cache is
//                 read once per tile) and come back as C^T through the transposing LDS read (ds_read_b64_tr_b16); wave w owns a
//                 quarter of the latent dimensions of the output; P goes through LDS as a bf16 pair hi + lo (two products), which
//                 keeps the softmax weights at f32 precision.
// A tile whose tokens belong to several sequences (decode steps of models with fewer than 16 heads) is processed once per
// sequence with the other rows masked.  blockIdx.y splits the key range into partitions for launches with few row tiles; their
// (max, sum, O) triples are merged, with the sink, by latent_attn_merge_kernel.
struct LatentAttnArgs {
    void *out;
    const void *q_abs;   // f32, or (io16) bf16 like out
    const float *q_rot;
    const uint16_t *cache;
    const int32_t *block_tables, *seq_ids, *positions;
    const uint16_t *sink;
    float *part_m, *part_l, *part_o;   // [T][H][NP], [T][H][NP], [T][H][NP][R]
    float scale;
    int max_blocks, window, T, H, R, rd, block_size, HPT, TPT, NHG, NP, io16;
};

// the eight query values from element `at` of the latent-space query on, rounded to bf16
__device__ __forceinline__ uint4 la_query8(const LatentAttnArgs &a, int64_t at) {
    if (a.io16) return *reinterpret_cast<const uint4 *>((const uint16_t *)a.q_abs + at);
    const float4 f0 = *reinterpret_cast<const float4 *>((const float *)a.q_abs + at), f1 = *reinterpret_cast<const float4 *>((const float *)a.q_abs + at + 4);
    const float f[8] = {f0.x, f0.y, f0.z, f0.w, f1.x, f1.y, f1.z, f1.w};
    return vmx_pack16x8<false>(f);
}
__device__ __forceinline__ uint4 la_query8(const float *rot) {
    const float4 f0 = *reinterpret_cast<const float4 *>(rot), f1 = *reinterpret_cast<const float4 *>(rot + 4);
    const float f[8] = {f0.x, f0.y, f0.z, f0.w, f1.x, f1.y, f1.z, f1.w};
    return vmx_pack16x8<false>(f);
}
__device__ __forceinline__ void la_store(void *out, int io16, int64_t at, float v) {
    if (io16) ((uint16_t *)out)[at] = vmx_f32_to_bf16(v);
    else ((float *)out)[at] = v;
}

constexpr int LA_KT = 64, LA_LD = LA_KT + 8;   // keys per tile; row stride of the P tiles
constexpr int LA_PAD = 32;                    // the row-major latent tile pads its rows by 64 bytes: four consecutive rows, four bank groups
typedef uint32_t la_u32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) uint16_t la_lds;
typedef short la_s16x4 __attribute__((ext_vector_type(4)));
typedef short la_s16x8 __attribute__((ext_vector_type(8)));

// WHOLE: rows of exactly 32 KSMAX values with 64 DTW latents (512 + 64).  Every size is then a constant, which leaves the registers for
// requesting a tile's rows while the one before it is worked on; other sizes request a tile's rows when its turn comes.  A partitioned
// launch (decode steps: one workgroup per compute unit, a tile or two each) is mostly setup, so latent_attn_mfma_kernel has no cap on its registers and no
// spills: 16 rows of 1000 tokens 22.3 -> 17.9 us (29.7 with the registers of two workgroups a compute unit, which latent_attn_shared_kernel has).
template <int KSMAX, int DTW, bool WHOLE>
__device__ __forceinline__ void latent_row_tile(const LatentAttnArgs &a, int tb, int hg, int part) {
    extern __shared__ __align__(256) unsigned char la_smem[];
    const int R = WHOLE ? 64 * DTW : a.R, RW = WHOLE ? 32 * KSMAX : a.R + a.rd;
    constexpr int ROWE = 64 * DTW + LA_PAD;   // of the largest latent this form takes, so that offsets are constants
    uint16_t *KT = reinterpret_cast<uint16_t *>(la_smem);            // [LA_KT][ROWE]: the tile's latents, row-major
    uint16_t *Phi = KT + (size_t)LA_KT * ROWE;                        // [16][LA_LD]
    uint16_t *Plo = Phi + 16 * LA_LD;                                 // [16][LA_LD]
    float *red_max = reinterpret_cast<float *>(Plo + 16 * LA_LD);     // [4][16]
    float *red_sum = red_max + 64;                                    // [4][16]
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), fl = lane & 15, fg = lane >> 4;
    const int t0 = tb * a.TPT, t_end = min(t0 + a.TPT, a.T);
    const int ksteps = WHOLE ? KSMAX : (RW + 31) >> 5;
    const int dtiles = WHOLE ? 4 * DTW : (R + 15) >> 4, dt_per_wave = WHOLE ? DTW : (dtiles + 3) >> 2, dt0 = wave * dt_per_wave;
    for (int first = t0; first < t_end;) {
        const int seq = a.seq_ids[first];
        int last = first;
        while (last + 1 < t_end && a.seq_ids[last + 1] == seq) last++;
        const int32_t *bt = a.block_tables + (int64_t)seq * a.max_blocks;
        const int hi = a.positions[last];
        const int lo = a.window > 0 ? max(0, a.positions[first] - a.window + 1) : 0;
        // no keys (a padding token's position -1): no tile, so no row is ever asked for below
        const int ntiles = hi < lo ? 0 : (hi - lo) / LA_KT + 1, tpp = (ntiles + a.NP - 1) / a.NP;
        const int kt_begin = part * tpp, kt_end = min(ntiles, kt_begin + tpp);
        // A operand of S: the query of row fl
        la_u32x4 qf[KSMAX];
        {
            const int tq = t0 + fl / a.HPT, hq = hg * a.HPT + fl % a.HPT;
            const bool act = fl < a.TPT * a.HPT && tq >= first && tq <= last && hq < a.H;
#pragma unroll
            for (int s = 0; s < KSMAX; s++) {
                const int k = 32 * s + 8 * fg;
                la_u32x4 v = {0, 0, 0, 0};
                if (s < ksteps && act && k < RW) {
                    const int64_t row = (int64_t)tq * a.H + hq;
                    v = __builtin_bit_cast(la_u32x4, k < R ? la_query8(a, row * R + k) : la_query8(a.q_rot + row * a.rd + (k - R)));
                }
                qf[s] = v;
            }
        }
        // the rows this lane holds in accumulator layout: 4 fg + r
        int rpos[4], rlo[4], rtok[4], rhead[4];
        bool ract[4];
        float m_r[4], l_r[4];
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int row = 4 * fg + r;
            rtok[r] = t0 + row / a.HPT;
            rhead[r] = hg * a.HPT + row % a.HPT;
            ract[r] = row < a.TPT * a.HPT && rtok[r] >= first && rtok[r] <= last && rhead[r] < a.H;
            rpos[r] = ract[r] ? a.positions[rtok[r]] : -1;
            rlo[r] = a.window > 0 ? max(0, rpos[r] - a.window + 1) : 0;
            m_r[r] = -FLT_MAX;
            l_r[r] = 0.f;
        }
        la_lds *const kt_read = (la_lds *)KT + (8 * fg + (fl >> 2)) * ROWE + 16 * dt0 + 4 * (fl & 3);
        vmx_f32x4 acc[DTW];
#pragma unroll
        for (int d = 0; d < DTW; d++) acc[d] = vmx_f32x4{0.f, 0.f, 0.f, 0.f};
        // this wave's 16 keys of a tile: lane (n, g) reads the 16-byte chunks 32 s + 8 g of key n's cache row.  They are the B operand of
        // the score product and, for the latent part of the row, the tile of the value product: each chunk is also written to
        // KT[key][latent dim], so the cache is read once per tile.  WHOLE: the rows are requested one tile ahead, as soon as the score
        // product has let go of the registers, and their block-table entry two.  Keys past `hi` repeat its row; their weights are 0.
        auto key_row = [&](int kt) {
            const int j = min(lo + LA_KT * kt + 16 * wave + fl, hi);
            return bt[j / a.block_size] * a.block_size + j % a.block_size;
        };
        la_u32x4 kf[KSMAX];
        auto request = [&](int row) {
            const uint16_t *at = a.cache + (int64_t)row * RW + 8 * fg;
#pragma unroll
            for (int s = 0; s < KSMAX; s++) {
                if (!WHOLE) kf[s] = la_u32x4{0, 0, 0, 0};
                if (WHOLE || (s < ksteps && 32 * s + 8 * fg < RW)) kf[s] = *reinterpret_cast<const la_u32x4 *>(at + 32 * s);
            }
        };
        int next_row = 0;
        if (kt_begin < kt_end) {
            if (WHOLE) request(key_row(kt_begin));
            next_row = key_row(kt_begin + (WHOLE ? 1 : 0));
        }
        for (int kt = kt_begin; kt < kt_end; kt++) {
            const int kbase = lo + LA_KT * kt;
            if (!WHOLE) {
                request(next_row);
                next_row = key_row(kt + 1);
            }
            __syncthreads();   // the previous tile's latents and P have been read
            vmx_f32x4 sacc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < KSMAX; s++) {
                const int k = 32 * s + 8 * fg;
                if (s < ksteps && k < R) *reinterpret_cast<la_u32x4 *>(KT + (16 * wave + fl) * ROWE + k) = kf[s];
            }
#pragma unroll
            for (int s = 0; s < KSMAX; s++)
                if (s < ksteps)
                    sacc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(vmx_bf16x8, qf[s]), __builtin_bit_cast(vmx_bf16x8, kf[s]), sacc, 0, 0,
                                                                   0);
            if (WHOLE && kt + 1 < kt_end) {
                request(next_row);
                next_row = key_row(kt + 2);
            }
            const int j = kbase + 16 * wave + fl;
            bool ok[4];
            float sc[4];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                ok[r] = ract[r] && j <= rpos[r] && j >= rlo[r];
                sc[r] = ok[r] ? sacc[r] * a.scale : -FLT_MAX;
                const float mx = vmx_row16_max(sc[r]);
                if (fl == 0) red_max[wave * 16 + 4 * fg + r] = mx;
            }
            __syncthreads();   // maxima and the transposed latents are in LDS
            float alpha[4];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int row = 4 * fg + r;
                const float tm = fmaxf(fmaxf(red_max[row], red_max[16 + row]), fmaxf(red_max[32 + row], red_max[48 + row]));
                const float m_new = fmaxf(m_r[r], tm);
                const float p = ok[r] ? expf(sc[r] - m_new) : 0.f;
                const uint16_t ph = vmx_f32_to_bf16(p);
                Phi[row * LA_LD + 16 * wave + fl] = ph;
                Plo[row * LA_LD + 16 * wave + fl] = vmx_f32_to_bf16(p - vmx_bf16_to_f32(ph));
                const float sm = vmx_row16_sum(p);
                if (fl == 0) red_sum[wave * 16 + row] = sm;
                alpha[r] = expf(m_r[r] - m_new);   // both -FLT_MAX (nothing seen yet): 1, and l and acc are still 0
                m_r[r] = m_new;
            }
            __syncthreads();
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int row = 4 * fg + r;
                l_r[r] = l_r[r] * alpha[r] + ((red_sum[row] + red_sum[16 + row]) + (red_sum[32 + row] + red_sum[48 + row]));
            }
#pragma unroll
            for (int d = 0; d < DTW; d++)
#pragma unroll
                for (int r = 0; r < 4; r++) acc[d][r] *= alpha[r];
#pragma unroll
            for (int ks = 0; ks < LA_KT / 32; ks++) {
                const la_u32x4 ah = *reinterpret_cast<const la_u32x4 *>(Phi + fl * LA_LD + 32 * ks + 8 * fg);
                const la_u32x4 al = *reinterpret_cast<const la_u32x4 *>(Plo + fl * LA_LD + 32 * ks + 8 * fg);
#pragma unroll
                for (int d = 0; d < DTW; d++) {
                    if (WHOLE || (d < dt_per_wave && dt0 + d < dtiles)) {
                        // B operand = C^T: the transposing LDS read hands lane n the values of column 16 dt + n for the four rows
                        // (keys) its 16-lane group addressed; two reads give the eight keys 32 ks + 8 g .. + 7 of this lane's k slots
                        la_lds *const src = kt_read + 32 * ks * ROWE + 16 * d;
                        const la_s16x4 c0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((la_s16x4 __attribute__((address_space(3))) *)src);
                        const la_s16x4 c1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((la_s16x4 __attribute__((address_space(3))) *)(src + 4 * ROWE));
                        const la_s16x8 cf = {c0[0], c0[1], c0[2], c0[3], c1[0], c1[1], c1[2], c1[3]};
                        acc[d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(vmx_bf16x8, ah), __builtin_bit_cast(vmx_bf16x8, cf), acc[d], 0, 0,
                                                                         0);
                        acc[d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(vmx_bf16x8, al), __builtin_bit_cast(vmx_bf16x8, cf), acc[d], 0, 0,
                                                                         0);
                    }
                }
            }
        }
        // results of rows 4 fg + r, latent dimensions 16 (dt0 + d) + fl
#pragma unroll
        for (int r = 0; r < 4; r++) {
            if (!ract[r]) continue;
            const int64_t th = (int64_t)rtok[r] * a.H + rhead[r];
            if (a.NP == 1) {
                const float sk = a.sink ? vmx_bf16_to_f32(a.sink[rhead[r]]) : -FLT_MAX;
                const float M = fmaxf(m_r[r], sk), w = expf(m_r[r] - M);
                const float den = l_r[r] * w + (a.sink ? expf(sk - M) : 0.f);
                const float f = den > 0.f ? w / den : 0.f;
#pragma unroll
                for (int d = 0; d < DTW; d++) {
                    const int dim = 16 * (dt0 + d) + fl;
                    if (d < dt_per_wave && dim < R) la_store(a.out, a.io16, th * R + dim, acc[d][r] * f);
                }
            } else {
                const int64_t tp = th * a.NP + part;
                if (wave == 0 && fl == 0) {
                    a.part_m[tp] = m_r[r];
                    a.part_l[tp] = l_r[r];
                }
#pragma unroll
                for (int d = 0; d < DTW; d++) {
                    const int dim = 16 * (dt0 + d) + fl;
                    if (d < dt_per_wave && dim < R) a.part_o[tp * R + dim] = acc[d][r];
                }
            }
        }
        first = last + 1;
    }
}

template <int KSMAX, int DTW, bool WHOLE>
__global__ __launch_bounds__(256, 1) void latent_attn_mfma_kernel(const LatentAttnArgs a) {
    latent_row_tile<KSMAX, DTW, WHOLE>(a, blockIdx.x / a.NHG, blockIdx.x % a.NHG, blockIdx.y);
}

// ---------------------------------------------------------------------------------------------------------------------------
// Prompts, rows of 512 + 64: FOUR row tiles a workgroup, one a wave, over the same keys.  With one row tile a workgroup the trips of its cache rows to the L2
// are what the time goes into (74 KB a 64-key tile for 16 rows of products); here a tile is fetched once for 64 rows:
//   * 32 keys at a time lie whole (latent | rotated part) in LDS, two tiles deep, filled by LDS-DMA one tile ahead: no registers, one barrier a tile.  Rows are
//     1152 bytes unpadded; 16-byte chunk c of row r sits at c ^ la_swizzle(r), so that neither the 16 rows that a score fragment reads at one chunk nor
//     the eight that a transposing read takes 32 bytes of share a bank group;
//   * S^T = K Q^T leaves a lane the scores of ONE row (fl) against keys 4 fg + r of both 16-key halves: maximum, weights and sum need no LDS, and
//     the weights go straight into the second product O^T = C^T P^T, whose k slots are assigned to the keys a lane already holds;
//   * the 128 accumulators are rescaled only on tiles where a row's maximum grew.  (Leaving it behind by up to 8 saves little and costs precision: the largest
//     weight is then no longer 1, which its two bf16 halves hold exactly.)
// us, 16 heads, one row tile a workgroup -> this: 600 + 500 + 400 tokens packed 177 -> 70, 599 + 501 + 401 173 -> 80, 4000 tokens 1654 -> 466, 130 tokens 29 -> 22, 1500 tokens with a
// window of 200 137 -> 49; 3 heads, 700 + 300 tokens 71 -> 63; 300 decode rows of 700 keys 97 -> 101.  (1 to 4 % of it are the zeros for other tokens' keys.)  Error against 64 bits as before (1.2e-6).
// The queries (72 registers) and the accumulators (128) leave two waves a SIMD, which cap the registers at 256; 85 more (332 bytes a lane of scratch memory) are
// spilled where queries and rows are set up and read back behind the loops; neither loop over key tiles touches scratch.  Blocks are numbered from the last token backwards: later tokens have
// more keys.  A group of row tiles over several sequences (a large decode step) has no keys to share: its tiles go the way above, one a workgroup,
// the first by the group's own workgroup and the others by those behind the groups.
__device__ __forceinline__ int la_swizzle(int r) { return ((((r >> 2) ^ (r >> 3)) & 1) << 2) | (r & 2) | ((r >> 3) & 1); }

__device__ __forceinline__ void la_request_1k(uint32_t at, const char *from) {   // 64 lanes x 16 bytes to the 1 KiB of LDS from byte `at` on
    at = __builtin_amdgcn_readfirstlane(at);
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" : : "s"(at), "v"(from) : "m0", "memory");
}

constexpr int LS_KT = 32, LS_ROW = 1152, LS_TILE = LS_KT * LS_ROW, LS_REQ = LS_TILE / 4096;   // keys a tile; bytes of a row and a tile; requests a wave
constexpr int LS_ZEROS = 1024;                                                                // bytes of zeros: a latent's

__global__ __launch_bounds__(256, 2) void latent_attn_shared_kernel(const LatentAttnArgs a) {
    extern __shared__ __align__(256) unsigned char la_smem[];
    constexpr int R = 512, RD = 64, KS = (R + RD) / 32, DT = R / 16;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), fl = lane & 15, fg = lane >> 4;
    const int row_tiles = (a.T + a.TPT - 1) / a.TPT, groups = (row_tiles + 3) / 4, leaders = groups * a.NHG;
    const bool leader = (int)blockIdx.x < leaders;
    const int id = leader ? leaders - 1 - (int)blockIdx.x : (int)blockIdx.x - leaders;
    const int hg = id % a.NHG, gi = id / a.NHG, group = leader ? gi : gi / 3, which = leader ? 0 : 1 + gi % 3;
    const int t0 = group * 4 * a.TPT, n = min(4 * a.TPT, a.T - t0);   // at most 64 tokens
    const int seq = a.seq_ids[t0];
    if (!__all(a.seq_ids[t0 + min(lane, n - 1)] == seq)) {
        if (4 * group + which < row_tiles) latent_row_tile<KS, R / 64, true>(a, 4 * group + which, hg, 0);
        return;
    }
    if (!leader) return;
    const int32_t *bt = a.block_tables + (int64_t)seq * a.max_blocks;
    int hi = a.positions[t0 + min(lane, n - 1)], lo = hi < 0 ? INT_MAX : a.window > 0 ? max(0, hi - a.window + 1) : 0;
    for (int m = 1; m < 64; m <<= 1) hi = max(hi, __shfl_xor(hi, m)), lo = min(lo, __shfl_xor(lo, m));
    hi = __builtin_amdgcn_readfirstlane(hi), lo = __builtin_amdgcn_readfirstlane(lo);
    // Tiles start at multiples of 32 keys, wherever `lo` lies: a row's sums are cut at the same keys whatever tokens share its workgroup
    const int key0 = lo / LS_KT * LS_KT, ntiles = hi < lo ? 0 : (hi - key0) / LS_KT + 1;
    // the lane's row
    const int tq = t0 + wave * a.TPT + fl / a.HPT, hq = hg * a.HPT + fl % a.HPT;
    const bool act = fl < a.TPT * a.HPT && tq < a.T && hq < a.H;
    const int rpos = act ? a.positions[tq] : -1, rlo = a.window > 0 ? max(0, rpos - a.window + 1) : 0;
    const int64_t th = act ? (int64_t)tq * a.H + hq : 0;
    // the keys of this wave's own tokens
    int own_hi = rpos, own_lo = rpos < 0 ? INT_MAX : rlo;
    for (int m = 1; m < 64; m <<= 1) own_hi = max(own_hi, __shfl_xor(own_hi, m)), own_lo = min(own_lo, __shfl_xor(own_lo, m));
    own_hi = __builtin_amdgcn_readfirstlane(own_hi), own_lo = __builtin_amdgcn_readfirstlane(own_lo);
    tg_u32x4 qf[KS];
#pragma unroll
    for (int s = 0; s < KS; s++) {
        qf[s] = __builtin_bit_cast(tg_u32x4, s < R / 32 ? la_query8(a, th * R + 32 * s + 8 * fg) : la_query8(a.q_rot + th * RD + 32 * s - R + 8 * fg));
    }
    // this wave fetches keys 8 wave .. + 7 of a tile: piece q's lane takes the chunk that belongs at byte 16 (64 q + lane) of those eight rows
    uint32_t piece[LS_REQ];   // byte in the source row | 4 x row << 16
#pragma unroll
    for (int q = 0; q < LS_REQ; q++) {
        const int c = 64 * q + lane, r = c / (LS_ROW / 16), at = c % (LS_ROW / 16);
        piece[q] = (uint32_t)((at ^ la_swizzle(8 * wave + r)) * 16) | (uint32_t)(4 * r) << 16;
    }
    // Key 8 wave + lane % 8 of a tile (keys below `lo` and past `hi`, whose blocks may be another sequence's by now, repeat their rows) and its block's table entry, which is not looked at
    // before the next tile's turn: a wait for it would be one for the rows requested before it
    auto key_of = [&](int kt) { return min(max(key0 + LS_KT * kt + 8 * wave + (lane & 7), lo), hi); };
    auto entry_of = [&](int kt) { return bt[key_of(kt) / a.block_size]; };
    const uint32_t lds = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)la_smem;
    auto request = [&](int kt, int entry, int stage) {
        const int row = entry * a.block_size + key_of(kt) % a.block_size;
#pragma unroll
        for (int q = 0; q < LS_REQ; q++) {
            uint32_t p = piece[q];
            asm volatile("" : "+v"(p));   // or nine 64-bit sums are kept in scratch memory, and each read of one waits for all requests under way
            const int from = __builtin_amdgcn_ds_bpermute((int)(p >> 16), row);
            la_request_1k(lds + stage * LS_TILE + (wave * LS_REQ + q) * 1024, reinterpret_cast<const char *>(a.cache) + (uint64_t)(uint32_t)from * LS_ROW + (p & 0xFFFFu));
        }
    };
    vmx_f32x4 acc[DT];
#pragma unroll
    for (int d = 0; d < DT; d++) acc[d] = vmx_f32x4{0.f, 0.f, 0.f, 0.f};
    float m_r = -FLT_MAX, l_r = 0.f;   // l_r: the lane's own keys
    const uint32_t k_at = lds + fl * LS_ROW + ((fg ^ la_swizzle(fl)) << 4);
    const int vr = 4 * fg + (fl >> 2);   // key of the first half of a tile whose values this lane asks for
    const uint32_t v_at = lds + vr * LS_ROW + ((((fl >> 1) & 1) ^ la_swizzle(vr)) << 4) + 8 * (fl & 1);
    // A wave's second product takes zeros for the keys that none of its own tokens has: their weights are 0, but 0 times an infinity or a NaN in another token's
    // cache row is a NaN.  Its reads of such a key go to a kilobyte of zeros behind the tiles.
    const uint32_t zeros = lds + 2 * LS_TILE;
    if (tid < LS_ZEROS / 16) *(__attribute__((address_space(3))) tg_u32x4 *)(uintptr_t)(zeros + 16 * tid) = tg_u32x4{};
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    int next_entry = 0;
    if (ntiles > 0) {
        request(0, entry_of(0), 0);
        next_entry = entry_of(1);
    }
    for (int kt = 0; kt < ntiles; kt++) {
        const int stage = kt & 1, kbase = key0 + LS_KT * kt;
        asm volatile("s_waitcnt vmcnt(0)" : "+v"(next_entry) : : "memory");
        __builtin_amdgcn_s_barrier();   // this tile is whole, and nobody reads the one before it any more
        asm volatile("" ::: "memory");
        if (kt + 1 < ntiles) {
            request(kt + 1, next_entry, stage ^ 1);
            next_entry = entry_of(kt + 2);
        }
        const uint32_t k_even = k_at + stage * LS_TILE, k_odd = k_even ^ 64;
        vmx_f32x4 sacc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
        // fragments are read AHEAD products before their use; the compiler alone reads each where it is needed and waits for it
        constexpr int AHEAD_K = 4, AHEAD_V = 3;
        tg_u32x4 kf[AHEAD_K];
        auto read_k = [&](int i) { return tg_lds_read((i & 2 ? k_odd : k_even) + (i >> 2) * 128 + (i & 1) * 16 * LS_ROW); };   // step i / 2, keys 16 (i % 2) ..
#pragma unroll
        for (int i = 0; i < AHEAD_K; i++) kf[i] = read_k(i);
#pragma unroll
        for (int i = 0; i < 2 * KS; i++) {
            sacc[i & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(vmx_bf16x8, kf[i % AHEAD_K]), __builtin_bit_cast(vmx_bf16x8, qf[i >> 1]), sacc[i & 1], 0, 0, 0);
            if (i + AHEAD_K < 2 * KS) kf[i % AHEAD_K] = read_k(i + AHEAD_K);
            __builtin_amdgcn_sched_barrier(0);
        }
        float p[8], top = -FLT_MAX;
        bool ok[8];
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const int j = kbase + 16 * (e >> 2) + 4 * fg + (e & 3);
            ok[e] = j <= rpos && j >= rlo;
            p[e] = ok[e] ? sacc[e >> 2][e & 3] * a.scale : -FLT_MAX;
            top = fmaxf(top, p[e]);
        }
        top = fmaxf(top, vmx_lane_xor_m(top, 16));
        top = fmaxf(top, vmx_lane_xor_m(top, 32));
        const bool moves = top > m_r;
        if (__any(moves)) {
            const float alpha = moves ? expf(m_r - top) : 1.f;
            if (moves) m_r = top;
            l_r *= alpha;
#pragma unroll
            for (int d = 0; d < DT; d++)
#pragma unroll
                for (int r = 0; r < 4; r++) acc[d][r] *= alpha;
        }
        float lo8[8];
#pragma unroll
        for (int e = 0; e < 8; e++) {
            p[e] = ok[e] ? expf(p[e] - m_r) : 0.f;
            l_r += p[e];
        }
        const vmx_bf16x8 ph = __builtin_bit_cast(vmx_bf16x8, vmx_pack16x8<false>(p));
#pragma unroll
        for (int e = 0; e < 8; e++) lo8[e] = p[e] - vmx_bf16_to_f32(vmx_f32_to_bf16(p[e]));
        const vmx_bf16x8 pl = __builtin_bit_cast(vmx_bf16x8, vmx_pack16x8<false>(lo8));
        auto v_from = [&](int half) {
            const int j = kbase + 16 * half + vr;
            return j >= own_lo && j <= own_hi ? v_at + stage * LS_TILE + half * 16 * LS_ROW : zeros;
        };
        const uint32_t v_half[2] = {v_from(0), v_from(1)};
        typedef la_s16x4 __attribute__((address_space(3))) *lds_s16x4;
        auto read_v = [&](int d, int half) {   // four keys of latent dimensions 16 d ..
            return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4)(uintptr_t)((v_half[half] ^ (32 * (d & 3))) + (d >> 2) * 128));
        };
        la_s16x4 vf[AHEAD_V][2];
#pragma unroll
        for (int d = 0; d < AHEAD_V; d++) vf[d][0] = read_v(d, 0), vf[d][1] = read_v(d, 1);
#pragma unroll
        for (int d = 0; d < DT; d++) {
            const la_s16x4 c0 = vf[d % AHEAD_V][0], c1 = vf[d % AHEAD_V][1];
            const la_s16x8 cf = {c0[0], c0[1], c0[2], c0[3], c1[0], c1[1], c1[2], c1[3]};
            acc[d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(vmx_bf16x8, cf), ph, acc[d], 0, 0, 0);
            acc[d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(vmx_bf16x8, cf), pl, acc[d], 0, 0, 0);
            if (d + AHEAD_V < DT) vf[d % AHEAD_V][0] = read_v(d + AHEAD_V, 0), vf[d % AHEAD_V][1] = read_v(d + AHEAD_V, 1);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    l_r += vmx_lane_xor_m(l_r, 16);
    l_r += vmx_lane_xor_m(l_r, 32);
    if (!act) return;
    const float sk = a.sink ? vmx_bf16_to_f32(a.sink[hq]) : -FLT_MAX;
    const float M = fmaxf(m_r, sk), w = expf(m_r - M);
    const float den = l_r * w + (a.sink ? expf(sk - M) : 0.f);
    const float f = den > 0.f ? w / den : 0.f;
#pragma unroll
    for (int d = 0; d < DT; d++) {   // latent dimensions 16 d + 4 fg ..
        const int64_t at = th * R + 16 * d + 4 * fg;
        const float4 v = make_float4(acc[d][0] * f, acc[d][1] * f, acc[d][2] * f, acc[d][3] * f);
        if (a.io16)
            *reinterpret_cast<uint2 *>((uint16_t *)a.out + at) = make_uint2(vmx_f32_to_bf16(v.x) | (uint32_t)vmx_f32_to_bf16(v.y) << 16, vmx_f32_to_bf16(v.z) | (uint32_t)vmx_f32_to_bf16(v.w) << 16);
        else *reinterpret_cast<float4 *>((float *)a.out + at) = v;
    }
}

// out[t, h] = sum_p e^(m_p - M) O_p / (sum_p e^(m_p - M) l_p + e^(sink - M)), M = max(sink, max_p m_p); NP <= 64.
// Wave 0 turns the partitions' (m, l) into one weight each (one round trip to memory), then every thread sums its dimensions.
__global__ __launch_bounds__(256) void latent_attn_merge_kernel(void *__restrict__ out, int io16, const float *__restrict__ part_m,
                                                                 const float *__restrict__ part_l, const float *__restrict__ part_o,
                                                                 const uint16_t *__restrict__ sink, int H, int R, int NP) {
    __shared__ float wgt[64];
    const int64_t th = blockIdx.x;
    if (threadIdx.x < 64) {
        const int p = threadIdx.x;
        const float sk = sink ? vmx_bf16_to_f32(sink[th % H]) : -FLT_MAX;
        const float m = p < NP ? part_m[th * NP + p] : -FLT_MAX, l = p < NP ? part_l[th * NP + p] : 0.f;
        const float M = vmx_wave_max(fmaxf(l > 0.f ? m : -FLT_MAX, sk));
        const float e = l > 0.f ? expf(m - M) : 0.f;
        const float den = vmx_wave_sum(e * l) + (sink ? expf(sk - M) : 0.f);
        wgt[p] = den > 0.f ? e / den : 0.f;
    }
    __syncthreads();
    for (int d = threadIdx.x; d < R; d += 256) {
        float v = 0.f;
        for (int p = 0; p < NP; p++) v = fmaf(wgt[p], part_o[(th * NP + p) * R + d], v);
        la_store(out, io16, th * R + d, v);
    }
}

}  // namespace

extern "C" int vmx_latent_prepare_rows(const vmx_latent_prepare *prep, const int32_t *positions, const int32_t *slots, void *cache,
                                       int cache_dtype, void *q_latent_out, int tokens, void *stream) {
    VMX_REQUIRE(prep && positions, "latent_prepare: null pointer");
    const vmx_latent_prepare &p = *prep;
    VMX_REQUIRE(cache_dtype == VMX_F32 || cache_dtype == VMX_BF16, "latent_prepare: the cache holds f32 or bf16");
    VMX_REQUIRE(!p.kv || (slots && cache && p.latent_norm_bf16 && p.kv_rank >= 1 && p.ldkv >= p.kv_rank + p.rot_dim), "latent_prepare: bad key/value rows");
    VMX_REQUIRE(!p.q || (p.heads >= 1 && p.dim >= 0 && p.rot_dim >= 0 && p.ldq >= (int64_t)p.heads * (p.dim + p.rot_dim) && (p.q_rot || p.rot_dim == 0)),
                "latent_prepare: bad query rows");
    VMX_REQUIRE(!p.q_latent || (q_latent_out && p.q_latent_norm_bf16 && p.q_rank >= 1 && p.ldq_latent >= p.q_rank), "latent_prepare: bad query latents");
    VMX_REQUIRE(!(p.kv || p.q) || (p.rot_dims >= 0 && p.rot_dims <= p.rot_dim && p.rot_dims % 2 == 0 && (p.inv_freq || p.rot_dims == 0)),
                "latent_prepare: rot_dims (%d) must be even and at most rot_dim (%d)", p.rot_dims, p.rot_dim);
    if (tokens <= 0) return VMX_OK;
    LatentPrepareArgs a{p, positions, slots, cache, q_latent_out};
    if (a.p.rot_mul == 0.f) a.p.rot_mul = 1.f;
    if (cache_dtype == VMX_F32) hipLaunchKernelGGL(latent_prepare_kernel<true>, dim3(tokens), dim3(256), 0, vmx_stream(stream), a);
    else hipLaunchKernelGGL(latent_prepare_kernel<false>, dim3(tokens), dim3(256), 0, vmx_stream(stream), a);
    VMX_CHECK_LAUNCH("latent_prepare");
    return VMX_OK;
}

extern "C" int vmx_latent_kv_prepare(const float *fused, int64_t ld_fused, int q_offset, int dkv_offset, const uint16_t *latent_norm_w,
                                     float eps, const float *inv_freq, int rot_dims, const int32_t *positions, const int32_t *slots,
                                     void *cache, int cache_dtype, float *q_rot, int tokens, int heads, int dim, int rot_dim, int kv_rank,
                                     void *stream) {
    VMX_REQUIRE(fused && latent_norm_w && inv_freq && positions && slots && cache && q_rot, "latent_kv_prepare: null pointer");
    vmx_latent_prepare p = {};
    p.kv = fused + dkv_offset, p.ldkv = ld_fused, p.kv_rank = kv_rank, p.latent_norm_bf16 = latent_norm_w, p.eps = eps;
    p.q = fused + q_offset, p.ldq = ld_fused, p.heads = heads, p.dim = dim, p.rot_dim = rot_dim, p.q_rot = q_rot;
    p.inv_freq = inv_freq, p.rot_dims = rot_dims, p.rot_mul = 1.0f;
    return vmx_latent_prepare_rows(&p, positions, slots, cache, cache_dtype, nullptr, tokens, stream);
}

int vmx_latent_transpose_heads(uint16_t *out, const uint16_t *in, int heads, int dim, int kv_rank, hipStream_t st) {
    hipLaunchKernelGGL(transpose_heads_kernel, dim3(512), dim3(256), 0, st, out, in, heads, dim, kv_rank);
    VMX_CHECK_LAUNCH("latent transpose");
    return VMX_OK;
}

// Partition count of the matrix-core form for a launch (host arithmetic only): one workgroup fits a compute unit at the largest
// latent size, so the launch is given at most one workgroup per compute unit -- row tiles x partitions <= compute units -- and a
// launch with that many row tiles or more is not split at all.
static int latent_attn_partitions(int tokens, int heads, int window, int max_blocks_per_seq, int block_size) {
    const int hpt = heads < 16 ? heads : 16, tpt = 16 / hpt, nhg = (heads + hpt - 1) / hpt;
    const int64_t tiles = (int64_t)((tokens + tpt - 1) / tpt) * nhg;
    int64_t max_keys = (int64_t)max_blocks_per_seq * block_size;
    if (window > 0 && window < max_keys) max_keys = window;
    const int64_t key_tiles = max_keys / LA_KT + 1;
    int64_t np = vmx_num_cus() / tiles;
    if (np > key_tiles) np = key_tiles;
    if (np > 64) np = 64;
    return np < 1 ? 1 : (int)np;
}

extern "C" size_t vmx_latent_attention_workspace_bytes(int tokens, int heads, int kv_rank, int window, int max_blocks_per_seq,
                                                       int block_size) {
    if (tokens <= 0 || heads <= 0 || kv_rank <= 0 || max_blocks_per_seq <= 0 || block_size <= 0) return 0;
    const int np = latent_attn_partitions(tokens, heads, window, max_blocks_per_seq, block_size);
    return np == 1 ? 0 : (size_t)tokens * heads * np * (kv_rank + 2) * sizeof(float);
}

// The matrix-core form: 16-byte chunks of a cache row must not straddle the latent / rotated boundary
static bool latent_on_matrix_cores(int cache_dtype, int kv_rank, int rot_dim) {
    return cache_dtype == VMX_BF16 && kv_rank % 8 == 0 && rot_dim % 8 == 0 && kv_rank + rot_dim <= 576;
}

bool vmx_latent_attention_takes_bf16(int cache_dtype, int kv_rank, int rot_dim) { return latent_on_matrix_cores(cache_dtype, kv_rank, rot_dim); }

int vmx_latent_attention_launch(void *out_latent, const void *q_abs, int io_bf16, const float *q_rot, const void *cache, int cache_dtype,
                                const int32_t *block_tables, int max_blocks_per_seq, const int32_t *seq_ids, const int32_t *positions,
                                const uint16_t *sink_bf16, float scale, int window, int tokens, int heads, int kv_rank, int rot_dim, int block_size,
                                void *workspace, size_t workspace_bytes, hipStream_t st) {
    VMX_REQUIRE(out_latent && q_abs && q_rot && cache && block_tables && seq_ids && positions, "latent_attention: null pointer");
    VMX_REQUIRE(cache_dtype == VMX_F32 || cache_dtype == VMX_BF16, "latent_attention: the cache holds f32 or bf16");
    VMX_REQUIRE(kv_rank >= 1 && kv_rank <= 512, "latent_attention: kv_rank (%d) must be in 1..512", kv_rank);
    VMX_REQUIRE(heads >= 1 && rot_dim >= 0 && block_size >= 1 && max_blocks_per_seq >= 1 && window >= 0, "latent_attention: bad sizes");
    VMX_REQUIRE(!io_bf16 || latent_on_matrix_cores(cache_dtype, kv_rank, rot_dim), "latent_attention: bf16 queries need the matrix-core form");
    if (tokens <= 0) return VMX_OK;
    const int RW = kv_rank + rot_dim;
    if (latent_on_matrix_cores(cache_dtype, kv_rank, rot_dim)) {
        LatentAttnArgs a;
        a.out = out_latent, a.q_abs = q_abs, a.io16 = io_bf16, a.q_rot = q_rot, a.cache = (const uint16_t *)cache;
        a.block_tables = block_tables, a.seq_ids = seq_ids, a.positions = positions, a.sink = sink_bf16;
        a.scale = scale, a.max_blocks = max_blocks_per_seq, a.window = window, a.T = tokens, a.H = heads, a.R = kv_rank, a.rd = rot_dim;
        a.block_size = block_size;
        a.HPT = heads < 16 ? heads : 16, a.TPT = 16 / a.HPT, a.NHG = (heads + a.HPT - 1) / a.HPT;
        a.NP = latent_attn_partitions(tokens, heads, window, max_blocks_per_seq, block_size);
        const size_t need = a.NP == 1 ? 0 : (size_t)tokens * heads * a.NP * (kv_rank + 2) * sizeof(float);
        if (need > workspace_bytes || (need && !workspace)) a.NP = 1;   // no room for partitions: one workgroup walks all keys
        a.part_m = (float *)workspace;
        a.part_l = a.part_m + (size_t)tokens * heads * a.NP;
        a.part_o = a.part_l + (size_t)tokens * heads * a.NP;
        dim3 grid((unsigned)(((tokens + a.TPT - 1) / a.TPT) * a.NHG), a.NP);
        const bool small = RW <= 160 && kv_rank <= 128;
        const size_t lds = ((size_t)LA_KT * ((small ? 128 : 512) + LA_PAD) + 2 * 16 * LA_LD) * 2 + (64 + 64) * 4;
        static_assert(2 * LS_TILE + LS_ZEROS <= (LA_KT * (512 + LA_PAD) + 2 * 16 * LA_LD) * 2 + (64 + 64) * 4, "the shared form fits the row tiles' memory");
        const bool whole = kv_rank == 512 && rot_dim == 64;
        const void *fn = small              ? (const void *)latent_attn_mfma_kernel<5, 2, false>
                         : !whole           ? (const void *)latent_attn_mfma_kernel<18, 8, false>
                         : a.NP > 1         ? (const void *)latent_attn_mfma_kernel<18, 8, true>
                                            : (const void *)latent_attn_shared_kernel;
        if (lds > 64 * 1024) VMX_CHECK_HIP(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        if (small) hipLaunchKernelGGL((latent_attn_mfma_kernel<5, 2, false>), grid, dim3(256), lds, st, a);
        else if (!whole) hipLaunchKernelGGL((latent_attn_mfma_kernel<18, 8, false>), grid, dim3(256), lds, st, a);
        else if (a.NP > 1) hipLaunchKernelGGL((latent_attn_mfma_kernel<18, 8, true>), grid, dim3(256), lds, st, a);
        else hipLaunchKernelGGL(latent_attn_shared_kernel, dim3((unsigned)(((tokens + a.TPT - 1) / a.TPT + 3) / 4 * 4 * a.NHG)), dim3(256), lds, st, a);
        VMX_CHECK_LAUNCH("latent_attention (matrix cores)");
        if (a.NP > 1) {
            hipLaunchKernelGGL(latent_attn_merge_kernel, dim3(tokens * heads), dim3(256), 0, st, out_latent, io_bf16, a.part_m, a.part_l, a.part_o, sink_bf16,
                               heads, kv_rank, a.NP);
            VMX_CHECK_LAUNCH("latent_attention (merge)");
        }
        return VMX_OK;
    }
    const size_t lds = (size_t)(kv_rank + rot_dim + 256 + 256 + 8 + 4 * kv_rank) * 4;
    dim3 grid(heads, tokens);
    if (cache_dtype == VMX_F32)
        hipLaunchKernelGGL(latent_attn_kernel<true>, grid, dim3(256), lds, st, (float *)out_latent, (const float *)q_abs, q_rot, cache, block_tables,
                           max_blocks_per_seq, seq_ids, positions, sink_bf16, scale, window, heads, kv_rank, rot_dim, block_size);
    else
        hipLaunchKernelGGL(latent_attn_kernel<false>, grid, dim3(256), lds, st, (float *)out_latent, (const float *)q_abs, q_rot, cache, block_tables,
                           max_blocks_per_seq, seq_ids, positions, sink_bf16, scale, window, heads, kv_rank, rot_dim, block_size);
    VMX_CHECK_LAUNCH("latent_attention");
    return VMX_OK;
}

extern "C" int vmx_latent_attention(float *out_latent, const float *q_abs, const float *q_rot, const void *cache, int cache_dtype,
                                    const int32_t *block_tables, int max_blocks_per_seq, const int32_t *seq_ids, const int32_t *positions,
                                    const uint16_t *sink_bf16, float scale, int window, int tokens, int heads, int kv_rank, int rot_dim,
                                    int block_size, void *workspace, size_t workspace_bytes, void *stream) {
    return vmx_latent_attention_launch(out_latent, q_abs, 0, q_rot, cache, cache_dtype, block_tables, max_blocks_per_seq, seq_ids, positions, sink_bf16, scale,
                                       window, tokens, heads, kv_rank, rot_dim, block_size, workspace, workspace_bytes, vmx_stream(stream));
}
