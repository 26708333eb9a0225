// Linear layers over UNQUANTIZED bf16 weights for any shape: C[m, n] (op)= sum_k A[m, k] * W(n, k), f32 accumulation in ascending k.
// One argument block (VmxLinear, vmx_kernels.h) describes every variant the executors need:
//   * activations in f32 or bf16, output in f32 or bf16; weights addressed with two strides, so [N, K] (y = W x) and [K, N]
//     (y = W^T x, the absorbed key up-projection of latent attention) are the same kernel;
//   * blockIdx.z batches with element strides (one product per attention head);
//   * gathered activation rows and per-row-block weight matrices (experts of a mixture whose (token, slot) pairs were sorted into
//     blocks by vmx_moe_align_block_size);
//   * an optional bf16 bias per output column, then an epilogue: plain store, squared ReLU, tanh-form GELU, accumulate into an
//     f32 residual stream, multiply by sigmoid(gate), or both of the last two (a gated residual update); a range of output columns
//     may go through SiLU, so that one product serves readers that want it and readers that do not.
// Kernels: `linear_tile_kernel` (prompts and 64-row expert blocks in whole 64-deep stages), `linear_mfma_kernel` (the same
// for unaligned rows and other depths; a staged 16-row form for shapes the streaming kernel does not take) and `linear_skinny_kernel` (up to 16
// rows: decode steps and 16-row expert blocks, weights streamed once) round the activations to bf16 and multiply on the matrix cores;
// `linear_fma_kernel` multiplies in true f32 on the vector ALU (the 32-bit mode of a model), `linear_fewcols_f32_kernel` does the
// same for a few output columns (router logits) with one kernel for every row count.  A row's result never depends on the other rows of the call: within a kernel a row is summed in
// the same order whatever M is; between the streaming and the tiled kernels the order differs (rounding-level differences).
#include <algorithm>
#include "tile_gemm.h"

namespace {

__device__ __forceinline__ float ld_act(const void *A, int a_f32, int64_t i) {
    return a_f32 ? ((const float *)A)[i] : vmx_bf16_to_f32(((const uint16_t *)A)[i]);
}

__device__ __forceinline__ void linear_store(const VmxLinear &p, int z, int m, int n, float v) {
    if (p.bias) v += vmx_bf16_to_f32(p.bias[n + z * p.bias_bs]);
    if (p.epilogue == VMX_EP_RELU2) {
        const float r = fmaxf(v, 0.f);
        v = r * r;
    } else if (p.epilogue == VMX_EP_GELU_TANH) {
        v = 0.5f * v * (1.0f + tanhf(0.7978845608028654f * (v + 0.044715f * v * v * v)));
    } else if (p.epilogue == VMX_EP_MUL_SIGMOID || p.epilogue == VMX_EP_ADD_MUL_SIGMOID) {
        const float g = p.aux[(int64_t)m * p.ldaux + (int64_t)n * p.aux_sn + z * p.aux_bs];
        v *= 1.0f / (1.0f + expf(-g));
    }
    if (n >= p.silu_begin && n < p.silu_end) v /= 1.0f + expf(-v);
    v *= p.out_scale;
    const int64_t o = (int64_t)m * p.ldc + n + z * p.c_bs;
    if (p.epilogue == VMX_EP_ADD_F32 || p.epilogue == VMX_EP_ADD_MUL_SIGMOID) ((float *)p.C)[o] += v;
    else if (p.c_f32) ((float *)p.C)[o] = v;
    else ((uint16_t *)p.C)[o] = vmx_f32_to_bf16(v);
}

// source row of output row m, or -1 for padding / out of range
__device__ __forceinline__ int64_t linear_src_row(const VmxLinear &p, int m) {
    if (m >= p.M) return -1;
    if (!p.row_ids) return m;
    const int r = p.row_ids[m];
    return (r < 0 || r >= p.row_limit) ? -1 : r / p.row_div;
}

// BM x 64 output tile per workgroup, 16 x 16 threads, (BM / 16) x 4 outputs per thread, 16-deep k steps through LDS.
template <int BM>
__global__ __launch_bounds__(256) void linear_fma_kernel(const VmxLinear p) {
    constexpr int BN = 64, BK = 16, TM = BM / 16, TN = 4;
    __shared__ float As[BK][BM + 1];
    __shared__ float Ws[BK][BN + 1];
    __shared__ int64_t rows[BM];
    const int tid = threadIdx.x, tx = tid & 15, ty = tid >> 4;
    const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN, z = blockIdx.z;
    if (p.total_rows && m0 >= *p.total_rows) return;
    const uint16_t *W = p.W + z * p.w_bs;
    if (p.block_expert) W += (int64_t)p.block_expert[m0 / p.block_rows] * p.expert_stride;
    const int64_t a_off = z * p.a_bs;
    for (int i = tid; i < BM; i += 256) rows[i] = linear_src_row(p, m0 + i);
    __syncthreads();
    float acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] = 0.f;
    const bool wk_fast = p.w_sk == 1;
    for (int k0 = 0; k0 < p.K; k0 += BK) {
        for (int i = tid; i < BM * BK; i += 256) {
            const int m = i / BK, k = i % BK;
            const int64_t r = rows[m];
            As[k][m] = (r >= 0 && k0 + k < p.K) ? ld_act(p.A, p.a_f32, a_off + r * p.lda + k0 + k) : 0.f;
        }
        for (int i = tid; i < BN * BK; i += 256) {
            const int n = wk_fast ? i / BK : i % BN, k = wk_fast ? i % BK : i / BN;
            Ws[k][n] = (n0 + n < p.N && k0 + k < p.K) ? vmx_bf16_to_f32(W[(int64_t)(n0 + n) * p.w_sn + (int64_t)(k0 + k) * p.w_sk]) : 0.f;
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < BK; k++) {
            float a[TM], w[TN];
#pragma unroll
            for (int i = 0; i < TM; i++) a[i] = As[k][ty * TM + i];
#pragma unroll
            for (int j = 0; j < TN; j++) w[j] = Ws[k][tx + 16 * j];
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++) acc[i][j] = fmaf(a[i], w[j], acc[i][j]);
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < TM; i++) {
        const int m = m0 + ty * TM + i;
        if (m >= p.M || (p.row_ids && rows[ty * TM + i] < 0)) continue;
#pragma unroll
        for (int j = 0; j < TN; j++) {
            const int n = n0 + tx + 16 * j;
            if (n < p.N) linear_store(p, z, m, n, acc[i][j]);
        }
    }
}

// Matrix-core form: BM x 64 output tile, 64-deep k stages of bf16 in LDS (rows padded by 16 bytes), v_mfma_f32_16x16x32_bf16.
// BM = 64: wave w owns the 32 x 32 quadrant (w >> 1, w & 1) as 2 x 2 instruction tiles; BM = 16: wave w owns columns 16 w .. + 16.
// The next stage is requested into registers before the current one is multiplied.  An output element sums its k in the same
// order in both shapes, so a row's result does not depend on which shape its call took.
template <int BM>
__global__ __launch_bounds__(256) void linear_mfma_kernel(const VmxLinear p) {
    constexpr int BN = 64, BK = 64, LD = BK + 8, CH = BK / 8;   // CH: 8-element chunks per staged row
    constexpr int TI = BM == 64 ? 2 : 1, TJ = BM == 64 ? 2 : 1;
    constexpr int ACH = (BM * CH + 255) / 256, WCH = BN * CH / 256;
    __shared__ __align__(16) uint16_t As[BM * LD];
    __shared__ __align__(16) uint16_t Ws[BN * LD];
    __shared__ int64_t rows[BM];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN, z = blockIdx.z;
    if (p.total_rows && m0 >= *p.total_rows) return;
    const uint16_t *W = p.W + z * p.w_bs;
    if (p.block_expert) W += (int64_t)p.block_expert[m0 / p.block_rows] * p.expert_stride;
    const int64_t a_off = z * p.a_bs;
    for (int i = tid; i < BM; i += 256) rows[i] = linear_src_row(p, m0 + i);
    __syncthreads();
    // 16-byte loads need aligned rows: every row start and every chunk a multiple of 8 (bf16) elements
    const bool a_vec = (p.K & 7) == 0 && (p.lda & 7) == 0 && (a_off & 7) == 0 && ((uintptr_t)p.A & 31) == 0;
    const bool w_vec = p.w_sk == 1 && (p.K & 7) == 0 && (p.w_sn & 7) == 0 && (((uintptr_t)W) & 15) == 0;
    uint4 ar[ACH], wr[WCH];
    auto fetch = [&](int k0) {
#pragma unroll
        for (int c = 0; c < ACH; c++) {
            const int idx = tid + 256 * c, m = idx / CH, k = k0 + 8 * (idx % CH);
            uint4 v = make_uint4(0, 0, 0, 0);
            if (idx < BM * CH) {
                const int64_t r = rows[m];
                if (r >= 0 && k < p.K) {
                    const int64_t at = a_off + r * p.lda + k;
                    if (a_vec) {
                        if (p.a_f32) {
                            const float4 f0 = *reinterpret_cast<const float4 *>((const float *)p.A + at);
                            const float4 f1 = *reinterpret_cast<const float4 *>((const float *)p.A + at + 4);
                            const float f[8] = {f0.x, f0.y, f0.z, f0.w, f1.x, f1.y, f1.z, f1.w};
                            v = vmx_pack16x8<false>(f);
                        } else {
                            v = *reinterpret_cast<const uint4 *>((const uint16_t *)p.A + at);
                        }
                    } else {
                        float f[8];
#pragma unroll
                        for (int e = 0; e < 8; e++) f[e] = k + e < p.K ? ld_act(p.A, p.a_f32, at + e) : 0.f;
                        v = vmx_pack16x8<false>(f);
                    }
                }
            }
            ar[c] = v;
        }
#pragma unroll
        for (int c = 0; c < WCH; c++) {
            const int idx = tid + 256 * c, n = n0 + idx / CH, k = k0 + 8 * (idx % CH);
            uint4 v = make_uint4(0, 0, 0, 0);
            if (n < p.N && k < p.K) {
                if (w_vec) {
                    v = *reinterpret_cast<const uint4 *>(W + (int64_t)n * p.w_sn + k);
                } else {
                    uint32_t h[8];
#pragma unroll
                    for (int e = 0; e < 8; e++) h[e] = k + e < p.K ? W[(int64_t)n * p.w_sn + (int64_t)(k + e) * p.w_sk] : 0;
                    v = make_uint4(h[0] | (h[1] << 16), h[2] | (h[3] << 16), h[4] | (h[5] << 16), h[6] | (h[7] << 16));
                }
            }
            wr[c] = v;
        }
    };
    auto stash = [&]() {
#pragma unroll
        for (int c = 0; c < ACH; c++) {
            const int idx = tid + 256 * c;
            if (idx < BM * CH) *reinterpret_cast<uint4 *>(As + (idx / CH) * LD + 8 * (idx % CH)) = ar[c];
        }
#pragma unroll
        for (int c = 0; c < WCH; c++) {
            const int idx = tid + 256 * c;
            *reinterpret_cast<uint4 *>(Ws + (idx / CH) * LD + 8 * (idx % CH)) = wr[c];
        }
    };
    vmx_f32x4 acc[TI][TJ];
#pragma unroll
    for (int i = 0; i < TI; i++)
#pragma unroll
        for (int j = 0; j < TJ; j++) acc[i][j] = vmx_f32x4{0.f, 0.f, 0.f, 0.f};
    const int wm = BM == 64 ? (wave >> 1) * 32 : 0, wn = BM == 64 ? (wave & 1) * 32 : wave * 16;
    const int fl = lane & 15, fg = lane >> 4;
    fetch(0);
    stash();
    __syncthreads();
    for (int k0 = 0; k0 < p.K; k0 += BK) {
        if (k0 + BK < p.K) fetch(k0 + BK);
#pragma unroll
        for (int s = 0; s < BK / 32; s++) {
            uint4 af[TI], wf[TJ];
#pragma unroll
            for (int i = 0; i < TI; i++) af[i] = *reinterpret_cast<const uint4 *>(As + (wm + 16 * i + fl) * LD + 32 * s + 8 * fg);
#pragma unroll
            for (int j = 0; j < TJ; j++) wf[j] = *reinterpret_cast<const uint4 *>(Ws + (wn + 16 * j + fl) * LD + 32 * s + 8 * fg);
#pragma unroll
            for (int i = 0; i < TI; i++)
#pragma unroll
                for (int j = 0; j < TJ; j++)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(vmx_bf16x8, af[i]), __builtin_bit_cast(vmx_bf16x8, wf[j]),
                                                                        acc[i][j], 0, 0, 0);
        }
        __syncthreads();
        if (k0 + BK < p.K) {
            stash();
            __syncthreads();
        }
    }
#pragma unroll
    for (int i = 0; i < TI; i++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int ml = wm + 16 * i + 4 * fg + r, m = m0 + ml;
            if (m >= p.M || (p.row_ids && rows[ml] < 0)) continue;
#pragma unroll
            for (int j = 0; j < TJ; j++) {
                const int n = n0 + wn + 16 * j + fl;
                if (n < p.N) linear_store(p, z, m, n, acc[i][j][r]);
            }
        }
}

// The accumulators to rows wm .., columns wn .. of C.  A tile inside C goes out without a look at each row: the choices and 64-bit
// addresses of the general form cost a 192 x 128 tile 6 us, a fifth of its products 2048 deep (1500 x 12288 x 2048: 105 -> 86 us).  bf16 columns go out in
// pairs: lane c even takes columns c, c + 1 of one row, its neighbour the same of the next row.
template <class S, typename T>
__device__ __forceinline__ void linear_tile_store(const VmxLinear &p, int z, int wm, int wn, int lane, tg_f32x16 (&acc)[S::MI][S::NJ]) {
    const int col = lane & 31;
    T *C = (T *)p.C + z * p.c_bs;
    if (!p.row_ids && wm + 32 * S::MI <= p.M && wn + 32 * S::NJ <= p.N) {
        constexpr bool PAIRS = sizeof(T) == 2;
        const bool odd = lane & 1, pairs = PAIRS && (((uintptr_t)C | (2 * p.ldc) | (2 * wn)) & 3) == 0;
        T *at = C + (int64_t)wm * p.ldc + wn;                                               // uniform
        const uint32_t off = (uint32_t)(4 * (lane >> 5)) * (uint32_t)p.ldc;                 // elements
#pragma unroll
        for (int i = 0; i < S::MI; i++)
#pragma unroll
            for (int r = 0; r < 16; r += 2) {
                T *row = at + (int64_t)(32 * i + 8 * (r >> 2) + (r & 3)) * p.ldc;
#pragma unroll
                for (int j = 0; j < S::NJ; j++) {
                    const float a = acc[i][j][r], b = acc[i][j][r + 1];
                    if constexpr (!PAIRS) {
                        row[32 * j + off + col] = a;
                        row[32 * j + p.ldc + off + col] = b;
                    } else if (pairs) {
                        const float got = vmx_dpp<VMX_DPP_XOR1>(odd ? a : b);
                        const uint32_t two = odd ? (uint32_t)vmx_f32_to_bf16(got) | (uint32_t)vmx_f32_to_bf16(b) << 16
                                                 : (uint32_t)vmx_f32_to_bf16(a) | (uint32_t)vmx_f32_to_bf16(got) << 16;
                        *reinterpret_cast<uint32_t *>(row + 32 * j + (off + (odd ? (uint32_t)p.ldc : 0u) + (col & 30))) = two;
                    } else {
                        row[32 * j + off + col] = vmx_f32_to_bf16(a);
                        row[32 * j + p.ldc + off + col] = vmx_f32_to_bf16(b);
                    }
                }
            }
        return;
    }
#pragma unroll
    for (int i = 0; i < S::MI; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int m = wm + 32 * i + tg_acc_row(lane, r);
            if (m >= p.M || (p.row_ids && linear_src_row(p, m) < 0)) continue;
            T *row = C + (int64_t)m * p.ldc + wn + col;
#pragma unroll
            for (int j = 0; j < S::NJ; j++) {
                if (wn + 32 * j + col >= p.N) continue;
                if constexpr (sizeof(T) == 4) row[32 * j] = acc[i][j][r];
                else row[32 * j] = vmx_f32_to_bf16(acc[i][j][r]);
            }
        }
}

// Prompt-sized bf16 products on the core of tile_gemm.h: plain, batched, gathered rows and 64-row expert blocks alike.  EP: the
// finished sums are stored as they are, with a bias and a SiLU range, times the sigmoids of a gate, or through linear_store (whose run-time choices per
// element cost a 1500 x 12288 output as much as half of its product: 159 against 101 us; gates read there wait for the store before them, each in
// turn: 16 products of 1500 x 128 x 512 33 -> 27 us).
// TILE_GLU: of a wave's pairs of 32 columns the first are gate columns and the second the up columns that belong to them, so a lane holds both.
enum { TILE_PLAIN, TILE_BIAS_SILU, TILE_GATE, TILE_ANY, TILE_GLU };
template <class S> struct HalfColumns { static constexpr int MI = S::MI, NJ = S::NJ / 2; };
struct GluLinear : VmxLinear { float slope, limit; };   // vmx_linear_glu
__device__ __forceinline__ float linear_glu(const GluLinear &p, float g, float u) {
    g = fminf(g, p.limit);
    return g / (1.0f + expf(-p.slope * g)) * (fminf(fmaxf(u, -p.limit), p.limit) + 1.0f);
}
template <class S, int EP, class P = VmxLinear>
__global__ __launch_bounds__(S::THREADS, S::PER_SIMD) void linear_tile_kernel(const P p, int row_tiles, int tiles) {
    extern __shared__ __align__(1024) uint16_t tg_lds[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int tile = tg_tile(blockIdx.x, tiles), z = blockIdx.y;
    if (tile < 0) return;
    const int m0 = tile % row_tiles * S::BM, n0 = tile / row_tiles * S::BN;
    if (p.total_rows && m0 >= *p.total_rows) return;
    const uint16_t *W = p.W + z * p.w_bs;
    if (p.block_expert) W += (int64_t)p.block_expert[m0 / p.block_rows] * p.expert_stride;
    // rows and columns past the end (and padding rows) fetch a row that exists; what they give is not stored
    uint32_t a_src[S::AQ], b_src[S::BQ];
#pragma unroll
    for (int q = 0; q < S::AQ; q++) {
        const int row = S::A32 ? tg_src_row32<S::AQ>(wave, lane, q) : tg_src_row<S::AQ>(wave, lane, q);
        const int64_t r = linear_src_row(p, m0 + row);
        a_src[q] = (uint32_t)((r < 0 ? 0 : r) * p.lda * (S::A32 ? 4 : 2)) + (S::A32 ? tg_src_byte32(lane, row) : tg_src_byte(lane));
    }
#pragma unroll
    for (int q = 0; q < S::BQ; q++)
    {
        const int c = tg_src_row<S::BQ>(wave, lane, q);   // column of the tile
        int n = min(n0 + c, p.N - 1);
        if constexpr (EP == TILE_GLU) {
            const int half = p.N / 2, j = c / 32 % S::NJ;
            n = (j & 1 ? half : 0) + min(n0 / 2 + c / (32 * S::NJ) * (16 * S::NJ) + j / 2 * 32 + (c & 31), half - 1);
        }
        b_src[q] = (uint32_t)((int64_t)n * p.w_sn * 2) + tg_src_byte(lane);
    }
    tg_f32x16 acc[S::MI][S::NJ];
#pragma unroll
    for (int i = 0; i < S::MI; i++)
#pragma unroll
        for (int j = 0; j < S::NJ; j++) acc[i][j] = tg_f32x16{};
    const TgCore<false, S> core{(const char *)p.A + z * p.a_bs * (S::A32 ? 4 : 2), (const char *)W, a_src, b_src, tg_lds_at(tg_lds), wave, lane};
    tg_product(core, p.K, acc);
    const int wm = m0 + wave / S::WN * (S::MI * 32), wn = n0 + wave % S::WN * (S::NJ * 32), col = lane & 31;
    if constexpr (EP == TILE_ANY) {
#pragma unroll
        for (int i = 0; i < S::MI; i++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int m = wm + 32 * i + tg_acc_row(lane, r);
                if (m >= p.M || (p.row_ids && linear_src_row(p, m) < 0)) continue;
#pragma unroll
                for (int j = 0; j < S::NJ; j++)
                    if (wn + 32 * j + col < p.N) linear_store(p, z, m, wn + 32 * j + col, acc[i][j][r]);
            }
        return;
    }
    if constexpr (EP == TILE_BIAS_SILU) {
#pragma unroll
        for (int j = 0; j < S::NJ; j++) {
            const int n = wn + 32 * j + col;
            const float bias = p.bias && n < p.N ? vmx_bf16_to_f32(p.bias[n + z * p.bias_bs]) : 0.f;
            const bool silu = n >= p.silu_begin && n < p.silu_end;
#pragma unroll
            for (int i = 0; i < S::MI; i++)
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    float v = acc[i][j][r] + bias;
                    if (silu) v /= 1.0f + expf(-v);
                    acc[i][j][r] = v;
                }
        }
    }
    if constexpr (EP == TILE_GATE) {
#pragma unroll
        for (int i = 0; i < S::MI; i++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const float *gate = p.aux + (int64_t)min(wm + 32 * i + tg_acc_row(lane, r), p.M - 1) * p.ldaux + z * p.aux_bs;
#pragma unroll
                for (int j = 0; j < S::NJ; j++) acc[i][j][r] *= 1.0f / (1.0f + expf(-gate[(int64_t)min(wn + 32 * j + col, p.N - 1) * p.aux_sn]));
            }
    }
    if constexpr (EP == TILE_GLU) {
        tg_f32x16 act[S::MI][S::NJ / 2];
#pragma unroll
        for (int i = 0; i < S::MI; i++)
#pragma unroll
            for (int j = 0; j < S::NJ / 2; j++)
#pragma unroll
                for (int r = 0; r < 16; r++) act[i][j][r] = linear_glu(p, acc[i][2 * j][r], acc[i][2 * j + 1][r]);
        VmxLinear out = p;
        out.N = p.N / 2;
        if (p.c_f32) linear_tile_store<HalfColumns<S>, float>(out, z, wm, wn / 2, lane, act);
        else linear_tile_store<HalfColumns<S>, uint16_t>(out, z, wm, wn / 2, lane, act);
        return;
    }
    if (p.c_f32) linear_tile_store<S, float>(p, z, wm, wn, lane, acc);
    else linear_tile_store<S, uint16_t>(p, z, wm, wn, lane, acc);
}

// Up to 16 rows (decode steps, 16-row expert blocks): the product is a stream over the weights.  A workgroup owns 16 output columns, or
// with PARTS = 2 eight columns whose k is halved over the two halves of a tile's columns: each weight fragment then meets two
// activation fragments, and of either product the half that belongs to its part is kept.  Its NW waves take the blocks w, w + NW, ..
// of 128 values a part.  Lane (c, g) reads 16 of the 64 consecutive bytes that the four lanes g share of a column, straight from memory
// and DEPTH blocks ahead, and the activation fragment at the same k from the (cache-resident) rows.  The waves' tiles are added in
// wave order through LDS.
// GluLinear: the sixteen columns are eight gate columns and the up columns that belong to them.
// What the first requests need comes as arguments of its own (in registers when a wave starts; `plain`: no row list, no blocks, one product).  Requests lie behind no
// condition of a lane, or the compiler waits for each before the next (dense_decode.hip): what lies past K reads the last values again and is cleared before the product,
// rows that do not exist read row 0 and are not stored.  A wave without a first or a second block takes a way of its own (as requests of one place, the same for every
// workgroup, they made shallow products slower than behind conditions: below).  f32 rows (A32) are rounded to bf16 as they are multiplied.
// HOLD: a block's requests are all made before its products, which the compiler else moves between them where a wave has one block: 16 rows of bf16, without / with,
// [2048, 2048] 5.9 / 5.7 us, [3664, 2048] 9.3 / 8.4, [32000, 512] 12.8 / 11.2, [12288, 512] 6.2 / 5.6; of one row 3.2 / 3.3 [4096, 512], and f32 rows 3 % slower with.
// 16 rows, us a launch, requests behind conditions / now:  gate and up [12288, 2048] 16.4 / 14.9, [32000, 2048] 36.9 / 34.3, [11264, 2048] 16.1 / 14.7, [3664, 2048] 9.2 / 8.4,
// [2048, 6144] 13.5 / 11.8, [2048, 2048] 6.5 / 5.7; a step of Larolorn's four layers with 1 / 4 / 16 rows 362 / 383 / 468 -> 354 / 367 / 450.
template <int NW, int PARTS, int DEPTH, bool A32, bool HOLD, class P = VmxLinear>
__global__ __launch_bounds__(64 * NW) void linear_skinny_kernel(const uint16_t *W, const void *A, int M, int N, int K, int lda, int w_sn, int plain, const P p) {
    constexpr bool GLU = std::is_same<P, GluLinear>::value;
    static_assert(!GLU || PARTS == 1, "eight gate and eight up columns a workgroup");
    constexpr int CW = 16 / PARTS, DEEP = 128 * PARTS, AV = A32 ? 2 : 1;   // 16-byte pieces that hold eight values of a row
    __shared__ float red[NW][64][4];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), fl = lane & 15, c = fl & (CW - 1), part = fl / CW, fg = lane >> 4;
    const int m0 = blockIdx.y * 16, n0 = blockIdx.x * CW, z = blockIdx.z;
    int64_t ar = min(fl, M - 1), row_len = lda, col_len = w_sn;
    if (!plain) {
        if (p.total_rows && m0 >= *p.total_rows) return;
        W += z * p.w_bs;
        if (p.block_expert) W += (int64_t)p.block_expert[m0 / p.block_rows] * p.expert_stride;
        A = (const char *)A + z * p.a_bs * (A32 ? 4 : 2);
        ar = max(linear_src_row(p, m0 + fl), (int64_t)0), row_len = p.lda, col_len = p.w_sn;
    }
    const int wn = GLU ? (c < 8 ? 0 : N / 2) + min(n0 / 2 + (c & 7), N / 2 - 1) : min(n0 + c, N - 1);
    const uint16_t *wrow = W + wn * col_len;
    const char *arow = (const char *)A + ar * row_len * (A32 ? 4 : 2);
    const int nblk = (K + DEEP - 1) / DEEP;
    tg_u32x4 w[DEPTH][4], a[DEPTH][PARTS][4][AV];
    auto load_w = [&](int b, tg_u32x4 (&d)[4]) {
#pragma unroll
        for (int j = 0; j < 4; j++) d[j] = *reinterpret_cast<const tg_u32x4 *>(wrow + min(DEEP * b + 128 * part + 32 * j + 8 * fg, K - 8));
    };
    auto load_a = [&](int b, tg_u32x4 (&d)[PARTS][4][AV]) {
#pragma unroll
        for (int q = 0; q < PARTS; q++)
#pragma unroll
            for (int j = 0; j < 4; j++)
#pragma unroll
                for (int e = 0; e < AV; e++)
                    d[q][j][e] = *reinterpret_cast<const tg_u32x4 *>(arow + min(DEEP * b + 128 * q + 32 * j + 8 * fg, K - 8) * (A32 ? 4 : 2) + 16 * e);
    };
    vmx_f32x4 acc[PARTS];
#pragma unroll
    for (int q = 0; q < PARTS; q++) acc[q] = vmx_f32x4{0.f, 0.f, 0.f, 0.f};
    auto step = [&](int b, tg_u32x4 (&wv)[4], tg_u32x4 (&av)[PARTS][4][AV]) {
        const bool past = DEEP * (b + 1) > K;   // the wave's
#pragma unroll
        for (int j = 0; j < 4; j++) {
            tg_u32x4 x = wv[j];
            if (past && DEEP * b + 128 * part + 32 * j + 8 * fg >= K) x = tg_u32x4{0, 0, 0, 0};
#pragma unroll
            for (int q = 0; q < PARTS; q++) {
                tg_u32x4 v = av[q][j][0];
                if constexpr (A32) {
                    const tg_u32x4 u = av[q][j][1];
                    const float f[8] = {__uint_as_float(v[0]), __uint_as_float(v[1]), __uint_as_float(v[2]), __uint_as_float(v[3]),
                                        __uint_as_float(u[0]), __uint_as_float(u[1]), __uint_as_float(u[2]), __uint_as_float(u[3])};
                    v = __builtin_bit_cast(tg_u32x4, vmx_pack16x8<false>(f));
                }
                if (past && DEEP * b + 128 * q + 32 * j + 8 * fg >= K) v = tg_u32x4{0, 0, 0, 0};
                acc[q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(vmx_bf16x8, v), __builtin_bit_cast(vmx_bf16x8, x), acc[q], 0, 0, 0);
            }
        }
    };
    auto load = [&](int b, tg_u32x4 (&wv)[4], tg_u32x4 (&av)[PARTS][4][AV]) {
        load_w(b, wv);
        load_a(b, av);
        if constexpr (HOLD) __builtin_amdgcn_sched_barrier(0);
    };
    if (DEPTH > 1 && wave + NW < nblk) {
        constexpr int L = DEPTH - 1;
        load(wave, w[0], a[0]);
        load(wave + NW, w[L], a[L]);
        for (int b = wave; b < nblk; b += 2 * NW) {
            step(b, w[0], a[0]);
            if (b + 2 * NW < nblk) load(b + 2 * NW, w[0], a[0]);
            if (b + NW < nblk) step(b + NW, w[L], a[L]);
            if (b + 3 * NW < nblk) load(b + 3 * NW, w[L], a[L]);
        }
    } else if (wave < nblk) {   // one block, or none: no requests in their place
        load(wave, w[0], a[0]);
        step(wave, w[0], a[0]);
    }
    // the product of a column's own part
    vmx_f32x4 own = acc[0];
    if constexpr (PARTS == 2) {
#pragma unroll
        for (int r = 0; r < 4; r++) own[r] = part ? acc[1][r] : acc[0][r];
    }
#pragma unroll
    for (int r = 0; r < 4; r++) red[wave][lane][r] = own[r];
    __syncthreads();
    if (tid >= 16 * CW) return;
    const int ml = tid / CW, nl = tid & (CW - 1), m = m0 + ml;   // element (4 g + r, c) of a tile sits with lane 16 g + c
    float v = 0.f;
#pragma unroll
    for (int q = 0; q < PARTS; q++)
#pragma unroll
        for (int i = 0; i < NW; i++) v += red[i][(ml >> 2) * 16 + CW * q + nl][ml & 3];
    if constexpr (GLU) {
        const float up = vmx_lane_xor<8>(v);
        const int n = n0 / 2 + nl;
        if (m < p.M && nl < 8 && n < p.N / 2) {
            const float y = linear_glu(p, v, up);
            if (p.c_f32) ((float *)p.C)[(int64_t)m * p.ldc + n] = y;
            else ((uint16_t *)p.C)[(int64_t)m * p.ldc + n] = vmx_f32_to_bf16(y);
        }
        return;
    }
    if (m < p.M && n0 + nl < p.N && !(p.row_ids && linear_src_row(p, m) < 0)) linear_store(p, z, m, n0 + nl, v);
}

template <int NW, int PARTS, int DEPTH, class P>
void launch_skinny_as(const P &p, hipStream_t st) {
    constexpr int CW = 16 / PARTS;
    const dim3 grid((p.N + CW - 1) / CW, (p.M + 15) / 16, p.batch);
    const int64_t most = 0x7fffffff;
    const int plain = p.M <= 16 && p.batch == 1 && !p.row_ids && !p.block_expert && !p.total_rows && p.lda >= 0 && p.lda <= most && p.w_sn >= 0 && p.w_sn <= most;
#define SKINNY(A32, HOLD) \
    hipLaunchKernelGGL((linear_skinny_kernel<NW, PARTS, DEPTH, A32, HOLD, P>), grid, dim3(64 * NW), 0, st, p.W, p.A, p.M, p.N, p.K, (int)p.lda, (int)p.w_sn, plain, p)
    if (p.a_f32) SKINNY(true, false);
    else if (DEPTH == 1 && (PARTS == 2 || p.M > 8)) SKINNY(false, DEPTH == 1);
    else SKINNY(false, DEPTH == 1 && PARTS == 2);
#undef SKINNY
}

// What bounds these is the number of requests under way, so the split follows the number of 16-column groups (and K, never M: a row's
// sums do not depend on its neighbours).  16 rows, before (one form: 4 waves, 16 columns, a lane's 64 bytes in a row) and now:
//   [12288, 2048], two groups a compute unit or more: 21.3 -> 16.6 us (the 64 bytes across lanes; 8 waves: 16.8); [32000, 2048]: 46.6 -> 36.7
//   [11264, 2048]: 21.2 -> 16.4;  [3664, 2048], fewer groups than compute units: 10.4 -> 8.4
//   [2048, 2048] and [2048, 6144], 128 groups: 12.4 on average -> 6.4 and 12.7
// Up to 512 deep a wave has one block of 16 columns: with eight columns and k halved it loads twice the rows for the same chain, which one f32 row paid
// for.  1 / 16 f32 rows, before / eight columns / now: [256, 256] 3.7 / 3.9 / 3.2 and 4.6 / 4.3 / 3.3, [4000, 512] 4.1 / 4.5 / 3.5 and 5.3 / 4.8 / 3.8
// Expert blocks bring row blocks of their own and keep four waves.
void launch_skinny(const VmxLinear &p, hipStream_t st) {
    const int cols = (p.N + 15) / 16 * p.batch, cus = vmx_num_cus();
    if (p.K > 512 && (p.block_expert || cols >= 2 * cus)) return launch_skinny_as<4, 1, 2>(p, st);
    if (cols >= cus || p.K <= 512) {
        const int nblk = (p.K + 127) / 128;
        return nblk <= 4 ? launch_skinny_as<4, 1, 1>(p, st) : nblk <= 8 ? launch_skinny_as<8, 1, 1>(p, st) : launch_skinny_as<8, 1, 2>(p, st);
    }
    const int nblk = (p.K + 255) / 256;
    if (nblk <= 4) return launch_skinny_as<4, 2, 1>(p, st);
    if (nblk <= 8) return launch_skinny_as<8, 2, 1>(p, st);
    launch_skinny_as<8, 2, 2>(p, st);
}
void launch_skinny_glu(const GluLinear &p, hipStream_t st) {   // sixteen columns a workgroup
    const int nblk = (p.K + 127) / 128;
    if (nblk > 4 && p.N / 16 >= 2 * vmx_num_cus()) return launch_skinny_as<4, 1, 2>(p, st);
    return nblk <= 4 ? launch_skinny_as<4, 1, 1>(p, st) : nblk <= 8 ? launch_skinny_as<8, 1, 1>(p, st) : launch_skinny_as<8, 1, 2>(p, st);
}

// A few output columns in true f32 (router logits): one workgroup per row and group of 16 columns; a thread walks its k with
// stride 256 over all 16 weight rows, then lanes, then waves are added in a fixed order.  Every row count takes this kernel, so
// a row's logits have the same bits in a prompt and in a decode step.
__global__ __launch_bounds__(256) void linear_fewcols_f32_kernel(const VmxLinear p) {
    __shared__ float red[4][16];
    const int m = blockIdx.x, n0 = blockIdx.y * 16, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    float acc[16];
#pragma unroll
    for (int e = 0; e < 16; e++) acc[e] = 0.f;
    for (int k = tid; k < p.K; k += 256) {
        const float x = ld_act(p.A, p.a_f32, (int64_t)m * p.lda + k);
#pragma unroll
        for (int e = 0; e < 16; e++) {
            const int n = min(n0 + e, p.N - 1);
            acc[e] = fmaf(x, vmx_bf16_to_f32(p.W[(int64_t)n * p.w_sn + k]), acc[e]);
        }
    }
#pragma unroll
    for (int e = 0; e < 16; e++) {
        const float v = vmx_wave_sum(acc[e]);
        if (lane == 0) red[wave][e] = v;
    }
    __syncthreads();
    if (tid < 16 && n0 + tid < p.N) linear_store(p, 0, m, n0 + tid, (red[0][tid] + red[1][tid]) + (red[2][tid] + red[3][tid]));
}

// What linear_tile_kernel takes: rows in 16-byte chunks, whole 64-deep stages, operands (one batch) inside 32-bit byte offsets.
bool tile_ok(const VmxLinear &p, bool direct) {
    const int64_t a_rows = p.row_ids ? (p.row_limit + p.row_div - 1) / p.row_div : p.M;
    return direct && p.K % TG_BK == 0 && a_rows * p.lda * (p.a_f32 ? 4 : 2) < (int64_t)1 << 32 && (int64_t)p.N * p.w_sn * 2 < (int64_t)1 << 32 &&
           p.lda >= 0 && p.w_sn >= 0;
}

template <class S, int EP, class P>
int launch_tile_as(const P &p, hipStream_t st) {
    const int row_tiles = (p.M + S::BM - 1) / S::BM, tiles = row_tiles * ((p.N + S::BN - 1) / S::BN);
    VMX_CHECK_HIP(hipFuncSetAttribute((const void *)linear_tile_kernel<S, EP, P>, hipFuncAttributeMaxDynamicSharedMemorySize, S::LDS));
    hipLaunchKernelGGL((linear_tile_kernel<S, EP, P>), dim3(tg_grid(tiles), p.batch), dim3(S::THREADS), S::LDS, st, p, row_tiles, tiles);
    return VMX_OK;
}

template <class S>
int launch_tile_shape(const VmxLinear &p, hipStream_t st) {
    const bool plain = !p.bias && p.silu_end <= p.silu_begin;
    if (p.epilogue == VMX_EP_MUL_SIGMOID && plain && p.out_scale == 1.0f) return launch_tile_as<S, TILE_GATE>(p, st);
    if (p.epilogue != VMX_EP_STORE || p.out_scale != 1.0f) return launch_tile_as<S, TILE_ANY>(p, st);
    if (!plain) return launch_tile_as<S, TILE_BIAS_SILU>(p, st);
    return launch_tile_as<S, TILE_PLAIN>(p, st);
}

// Every shape adds an element's k in the same order.
typedef TgShape<2, 2, 1, 1, 5> Tile64;       // 64 x 64, two workgroups a compute unit
typedef TgShape<2, 2, 1, 2, 3> Tile64w;      // 64 x 128, two
typedef TgShape<2, 2, 2, 2, 2> Tile128two;   // 128 x 128, two
typedef TgShape<2, 4, 2, 1, 4> Tile128;      // 128 x 128, one
typedef TgShape<2, 2, 3, 2, 3> Tile192;      // 192 x 128, one
typedef TgShape<4, 2, 2, 2, 3> Tile256;      // 256 x 128, one
// f32 rows: 64 x 128, two a unit (64 x 64, 128 x 64, 128 x 128 one a unit: 16 products of 1500 x 512 x 128 in 30 / 31 / 27 us against 22).  us, linear_mfma_kernel
// -> this: those products 53 -> 22; 17 x 64 x 512 12 -> 8, 64 x 256 x 2048 42 -> 21, 500 x 8192 x 128 19 -> 8, 1500 x 12288 x 2048 337 -> 160, 2000 x 2048 x 6144 304 -> 95.
typedef TgShape<2, 2, 1, 2, 2, true> Tile64f;

// Estimated ns of a launch.  It runs in rounds of one tile for every place; a 64-deep step of a full round takes `full`, one with at most a
// workgroup for every second place `few` (shapes with two places a unit), and a last round is shorter, the emptier it is (least so where it is the
// only one of a shape with two places).  The results leave at 9.2 TB/s (into the L2), half of that time under the products of the unit's other
// workgroup where it has one.
template <class S>
int64_t tile_ns(const VmxLinear &p, int full, int few) {
    const int64_t tiles = (int64_t)((p.M + S::BM - 1) / S::BM) * ((p.N + S::BN - 1) / S::BN) * p.batch, places = (int64_t)vmx_num_cus() * S::PER_UNIT;
    const int64_t rounds = tiles / places, rest = tiles % places, out = (int64_t)p.M * p.N * p.batch * (p.c_f32 ? 4 : 2) / (S::PER_UNIT > 1 ? 18400 : 9200);
    if (S::PER_UNIT > 1 && tiles <= places / 2) return p.K / TG_BK * (int64_t)few + out;
    const int64_t last = rest == 0 ? 0 : S::PER_UNIT == 1 ? full * (3 * places + rest) / (4 * places)
                                       : rounds == 0 ? full * (4 * places + rest) / (5 * places) : full * (2 * places + 3 * rest) / (5 * places);
    return p.K / TG_BK * (rounds * full + last) + out;
}

// The shape with the least estimate.  Fitted to bf16 products of 17 .. 2000 rows on 256 units, weights out of HBM.  us, 64 x 64 / 64 x 128 / 128 x 128
// two / one a unit / 192 / 256 x 128 (rows x columns x depth, bf16 results):  100 x 12288 x 2048 19 / 19 / 31 / 21 / 25 / 25;  200 24 / 25 / 33 / 21 /
// 26 / 29;  500 49 / 42 / 38 / 42 / 51 / 32;  700 67 / 59 / 64 / 57 / 53 / 59;  1000 94 / 77 / 68 / 64 / 75 / 62;  1500 139 / 107 / 99 / 99 / 83 / 90;
// 1500 x 11264 x 2048 129 / 99 / 89 / 92 / 83 / 81;  1500 x 3664 x 2048 47 / 38 / 33 / 41 / 28 / 30;  1000 x 2048 x 6144 48 / 47 / 79 / 53 / 57 / 73;
// 1500 x 2048 x 6144 74 / 61 / 81 / 53 / 65 / 73.  The call before (128 x 128 two a unit, or 64 x 64 in two or three stages, requests at the head of a
// stage, results element by element) and now:  1500 x 12288 x 2048 107 -> 85, 1500 x 3664 x 2048 36 -> 28, 1500 x 2048 x 6144 72 -> 53, 500 x 12288 x
// 2048 42 -> 33, 333 x 2048 x 6144 35 -> 25, 100 x 3664 x 2048 14.6 -> 11.2.  Expert blocks bring 64 rows each.
int64_t ns64(const VmxLinear &p) { return tile_ns<Tile64>(p, 490, 280); }
int64_t ns64w(const VmxLinear &p) { return tile_ns<Tile64w>(p, 700, 450); }
int64_t ns128two(const VmxLinear &p) { return tile_ns<Tile128two>(p, 1130, 800); }
int64_t ns128(const VmxLinear &p) { return tile_ns<Tile128>(p, 640, 0); }
int64_t ns192(const VmxLinear &p) { return tile_ns<Tile192>(p, 850, 0); }
int64_t ns256(const VmxLinear &p) { return tile_ns<Tile256>(p, 1000, 0); }
int launch_tile(const VmxLinear &p, hipStream_t st) {
    if (p.a_f32) return launch_tile_shape<Tile64f>(p, st);
    const int64_t t64 = ns64(p), t64w = ns64w(p);
    if (p.block_expert) return t64 <= t64w ? launch_tile_shape<Tile64>(p, st) : launch_tile_shape<Tile64w>(p, st);
    const int64_t two = ns128two(p), t128 = ns128(p), t192 = ns192(p), t256 = ns256(p), least = std::min({t64, t64w, two, t128, t192, t256});
    if (least == t64) return launch_tile_shape<Tile64>(p, st);
    if (least == t64w) return launch_tile_shape<Tile64w>(p, st);
    if (least == t128) return launch_tile_shape<Tile128>(p, st);
    if (least == t192) return launch_tile_shape<Tile192>(p, st);
    return least == t256 ? launch_tile_shape<Tile256>(p, st) : launch_tile_shape<Tile128two>(p, st);
}
// ... of those whose waves own pairs of 32 columns
int launch_tile_glu(const GluLinear &p, hipStream_t st) {
    const int64_t t64w = ns64w(p), two = ns128two(p), t192 = ns192(p), t256 = ns256(p), least = std::min({t64w, two, t192, t256});
    if (least == t64w) return launch_tile_as<Tile64w, TILE_GLU>(p, st);
    if (least == t192) return launch_tile_as<Tile192, TILE_GLU>(p, st);
    return least == t256 ? launch_tile_as<Tile256, TILE_GLU>(p, st) : launch_tile_as<Tile128two, TILE_GLU>(p, st);
}

// 16-byte loads straight from the operands: whole 8-element chunks, aligned rows
bool direct_ok(const VmxLinear &p) {
    return p.w_sk == 1 && p.K % 8 == 0 && p.w_sn % 8 == 0 && p.lda % 8 == 0 && p.a_bs % 8 == 0 && p.w_bs % 8 == 0 && p.expert_stride % 8 == 0 &&
           ((uintptr_t)p.W & 15) == 0 && ((uintptr_t)p.A & 31) == 0;
}

}  // namespace

// A plain product with bf16 rows (a few rows: f32 as well) whose kernel ends in TILE_GLU or its counterpart for up to 16 rows.  Against f32 rows of gate and up
// and a kernel of its own for the activation (the same bits): 1500 x 12288 x 2048 89.5 + 17.8 -> 91.6 us, 16 rows 17.0 + 4.6 -> 16.2.
bool vmx_linear_glu_ok(const VmxLinear &p) {
    const bool plain = !p.exact && p.batch == 1 && !p.row_ids && !p.block_expert && !p.bias && p.silu_end <= p.silu_begin && p.epilogue == VMX_EP_STORE &&
                       p.out_scale == 1.0f;
    if (!plain || p.M < 1 || p.N % 16 || !direct_ok(p)) return false;
    return p.M <= 16 || (!p.a_f32 && tile_ok(p, true));
}

// Whether that is faster than a plain product into f32 rows and a kernel of its own for the activation.  Up to 16 rows it is.  Tiles: pairs of columns leave out the
// shapes of 64 x 64 and of 128 x 128 with one workgroup a unit, and where those are the plain product's, two launches can be done first.  Both sides by
// the shapes' estimates and what these leave out: shapes with two workgroups a unit wait for weights out of memory (the bytes at 8 TB/s); the activation's launch, and its
// rows at 4.5 TB/s.  us, two launches / this, weights out of memory:  12288 x 2048, 17 rows 15.8 / 20.2, 64 17.1 / 20.8, 65 21.1 / 19.8, 128 23.1 / 20.6, 129 22.6 / 26.9,
// 256 28.1 / 30.3, 257 33.0 / 28.1, 1500 102 / 87;  16384 x 3072, 64 24.8 / 31.8, 65 30.7 / 28.9, 192 38.1 / 47.0, 257 46.3 / 41.5;  24576 x 4096, 64 50.7 / 47.5, 128 58.8 /
// 62.6, 129 60.0 / 56.5;  6144 x 1024, 128 10.8 / 11.8, 129 13.1 / 11.4;  2816 x 2048, 300 14.8 / 18.5, 400 20.3 / 18.2.  Of six widths at 27 counts of 17 .. 2000 rows all but
// one (2816 x 2048, 333 rows: 16.1 / 18.3) take the faster side or are within 3 % of it.
int vmx_linear_glu_pays(const VmxLinear &p) {
    if (p.M <= 16) return 1;
    VmxLinear rows = p;   // of gate and up
    rows.c_f32 = 1;
    const int64_t fetch = (int64_t)p.N * p.K * 2 / 8000, activation = 800 + (int64_t)p.M * p.N / 2 * 10 / 4500;
    auto least = [&](int64_t two_a_unit, int64_t one_a_unit) { return two_a_unit <= one_a_unit ? two_a_unit + fetch : one_a_unit; };
    const int64_t apart = least(std::min({ns64(rows), ns64w(rows), ns128two(rows)}), std::min({ns128(rows), ns192(rows), ns256(rows)}));
    return least(std::min(ns64w(p), ns128two(p)), std::min(ns192(p), ns256(p))) <= apart + activation;
}

int vmx_linear_glu(const VmxLinear &p, float slope, float limit, hipStream_t st) {
    VMX_REQUIRE(p.A && p.W && p.C && p.N > 0 && p.K > 0 && vmx_linear_glu_ok(p), "linear_glu: no gated epilogue for %d rows, [%d, %d]", p.M, p.N, p.K);
    GluLinear g;
    static_cast<VmxLinear &>(g) = p;
    g.slope = slope, g.limit = limit;
    if (p.M <= 16) launch_skinny_glu(g, st);
    else if (int rc = launch_tile_glu(g, st)) return rc;
    VMX_CHECK_LAUNCH("linear (gated)");
    return VMX_OK;
}

int vmx_linear_launch(const VmxLinear &p, hipStream_t st) {
    VMX_REQUIRE(p.A && p.W && p.C, "linear: null pointer");
    VMX_REQUIRE(p.M >= 0 && p.N > 0 && p.K > 0 && p.batch >= 1, "linear: bad shape M %d N %d K %d batch %d", p.M, p.N, p.K, p.batch);
    VMX_REQUIRE((p.epilogue != VMX_EP_ADD_F32 && p.epilogue != VMX_EP_ADD_MUL_SIGMOID) || p.c_f32, "linear: the accumulating epilogues need an f32 output");
    VMX_REQUIRE((p.epilogue != VMX_EP_MUL_SIGMOID && p.epilogue != VMX_EP_ADD_MUL_SIGMOID) || p.aux, "linear: the gate epilogues need their gate rows");
    VMX_REQUIRE(!p.block_expert || (p.total_rows && (p.block_rows == 16 || p.block_rows == 64)), "linear: expert blocks are 16 or 64 rows");
    VMX_REQUIRE(!p.row_ids || p.row_div >= 1, "linear: row_div must be positive");
    if (p.M == 0) return VMX_OK;
    const bool plain = !p.row_ids && !p.block_expert && p.batch == 1 && p.w_sk == 1;
    if (p.exact && plain && p.N <= 256) {
        hipLaunchKernelGGL(linear_fewcols_f32_kernel, dim3(p.M, (p.N + 15) / 16), dim3(256), 0, st, p);
        VMX_CHECK_LAUNCH("linear (few columns)");
        return VMX_OK;
    }
    const int bm = p.block_expert ? p.block_rows : (p.M <= 16 ? 16 : 64);
    dim3 grid((p.N + 63) / 64, (p.M + bm - 1) / bm, p.batch);
    if (p.exact) {
        if (bm == 16) hipLaunchKernelGGL(linear_fma_kernel<16>, grid, dim3(256), 0, st, p);
        else hipLaunchKernelGGL(linear_fma_kernel<64>, grid, dim3(256), 0, st, p);
    } else {
        const bool direct = direct_ok(p);
        if (bm == 64 && tile_ok(p, direct)) {
            if (int rc = launch_tile(p, st)) return rc;
        } else if (bm == 16 && direct) {
            launch_skinny(p, st);
        } else if (bm == 16) hipLaunchKernelGGL(linear_mfma_kernel<16>, grid, dim3(256), 0, st, p);
        else hipLaunchKernelGGL(linear_mfma_kernel<64>, grid, dim3(256), 0, st, p);
    }
    VMX_CHECK_LAUNCH("linear");
    return VMX_OK;
}

extern "C" int vmx_linear_bf16w(void *y, int y_dtype, const void *x, int x_dtype, const uint16_t *w, int M, int N, int K, int exact,
                                void *stream) {
    VMX_REQUIRE((y_dtype == VMX_F32 || y_dtype == VMX_BF16) && (x_dtype == VMX_F32 || x_dtype == VMX_BF16), "linear_bf16w: f32 or bf16 rows");
    VmxLinear p;
    p.A = x, p.a_f32 = x_dtype == VMX_F32, p.lda = K;
    p.W = w, p.w_sn = K, p.w_sk = 1;
    p.C = y, p.c_f32 = y_dtype == VMX_F32, p.ldc = N;
    p.M = M, p.N = N, p.K = K, p.exact = exact;
    return vmx_linear_launch(p, vmx_stream(stream));
}
