// Prompt-sized linears over GGUF I-quant weights.  Beyond IQ_GEMV_MAX_M = 16 rows the reference dequantises the whole weight to
// dense f32 and runs one f32 GEMM on the f32 activations (IqLinear::forward_inner, crates/core/src/quantization/gguf/mod.rs:346-365):
// no q8_1 rounding of the activations on that path.  gfx950 has no fast f32 matrix instruction, but the activations are bf16 values
// and a dequantised weight w = d * scale * grid needs at most ~16 mantissa bits, so w is split as hi = bf16(w), lo = bf16(w - hi) and
// the product is two bf16 MFMA passes into one f32 accumulator: x * hi and x * lo are exact in f32, and hi + lo reproduces w to
// 2^-17 relative -- below the f32 summation noise of a dot over thousands of terms.
#include <algorithm>
#include "vmx_internal.h"
#include "tile_gemm.h"

namespace {

typedef float sg_f32x4 __attribute__((ext_vector_type(4)));

// C[m, n] (f32, row stride ldc) = sum_k A[m,k] * (Bhi[n,k] + Blo[n,k]);  A [M, K] bf16, Bhi / Blo [N, K] bf16, K % 32 == 0.
// Workgroup = 4 waves side by side on a 64 x 256 tile of C; a wave owns 64 rows x 64 columns = 4 x 4 accumulators of
// v_mfma_f32_16x16x32_bf16.  Lane (i = lane & 15, g = lane >> 4) feeds row i of a 16-row block with the 8 values k0 + 8 g .. + 7,
// read straight from global memory as one 16-byte load per operand block (the four waves of a workgroup re-read the A rows
// through the vector L1).  No LDS, no barriers: out-of-range rows and columns read a clamped address and are not stored.
// KSPLIT: few output tiles (down_proj, o_proj: N = hidden) would leave most compute units idle, so the four waves of a workgroup
// share ONE 64 x 64 tile and take a quarter of K each; the quarters are added through LDS in wave order (deterministic).
template <bool LO, bool KSPLIT>
__global__ __launch_bounds__(256) void split_gemm_kernel(const uint16_t *__restrict__ A, const uint16_t *__restrict__ Bhi,
                                                          const uint16_t *__restrict__ Blo, float *__restrict__ C, int M, int N, int K,
                                                          int ldc) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int i = lane & 15, g = lane >> 4;
    const int m0 = blockIdx.y * 64, n0 = KSPLIT ? blockIdx.x * 64 : blockIdx.x * 256 + wave * 64;
    if (!KSPLIT && n0 >= N) return;
    const int kq = K / 4;   // KSPLIT: K % 128 == 0
    const int k_begin = KSPLIT ? wave * kq : 0, k_end = KSPLIT ? k_begin + kq : K;
    int64_t arow[4], brow[4];
#pragma unroll
    for (int b = 0; b < 4; b++) {
        arow[b] = (int64_t)min(m0 + b * 16 + i, M - 1) * K + 8 * g;
        brow[b] = (int64_t)min(n0 + b * 16 + i, N - 1) * K + 8 * g;
    }
    sg_f32x4 acc[4][4];
#pragma unroll
    for (int rb = 0; rb < 4; rb++)
#pragma unroll
        for (int cb = 0; cb < 4; cb++) acc[rb][cb] = sg_f32x4{0.f, 0.f, 0.f, 0.f};
    for (int k0 = k_begin; k0 < k_end; k0 += 32) {
        uint4 a[4], bh[4], bl[4];
#pragma unroll
        for (int b = 0; b < 4; b++) {
            a[b] = *reinterpret_cast<const uint4 *>(A + arow[b] + k0);
            bh[b] = *reinterpret_cast<const uint4 *>(Bhi + brow[b] + k0);
            if (LO) bl[b] = *reinterpret_cast<const uint4 *>(Blo + brow[b] + k0);
        }
#pragma unroll
        for (int cb = 0; cb < 4; cb++)
#pragma unroll
            for (int rb = 0; rb < 4; rb++) {
                acc[rb][cb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(vmx_bf16x8, a[rb]), __builtin_bit_cast(vmx_bf16x8, bh[cb]),
                                                                      acc[rb][cb], 0, 0, 0);
                if (LO)
                    acc[rb][cb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(vmx_bf16x8, a[rb]),
                                                                          __builtin_bit_cast(vmx_bf16x8, bl[cb]), acc[rb][cb], 0, 0, 0);
            }
    }
    if constexpr (KSPLIT) {
        // wave w keeps row block w: it adds the four waves' sums of that block in wave order
        __shared__ sg_f32x4 red[4][4][4][64];   // [source wave][row block][column block][lane]: 64 KiB
#pragma unroll
        for (int rb = 0; rb < 4; rb++)
#pragma unroll
            for (int cb = 0; cb < 4; cb++) red[wave][rb][cb][lane] = acc[rb][cb];
        __syncthreads();
#pragma unroll
        for (int cb = 0; cb < 4; cb++) {
            sg_f32x4 t = red[0][wave][cb][lane];
#pragma unroll
            for (int w = 1; w < 4; w++) {
                const sg_f32x4 o = red[w][wave][cb][lane];
                t[0] += o[0]; t[1] += o[1]; t[2] += o[2]; t[3] += o[3];
            }
            const int col = n0 + cb * 16 + i;
            if (col >= N) continue;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int row = m0 + wave * 16 + 4 * g + j;
                if (row < M) C[(int64_t)row * ldc + col] = t[j];
            }
        }
        return;
    }
#pragma unroll
    for (int rb = 0; rb < 4; rb++)
#pragma unroll
        for (int cb = 0; cb < 4; cb++) {
            const int col = n0 + cb * 16 + i;
            if (col >= N) continue;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int row = m0 + rb * 16 + 4 * g + j;
                if (row < M) C[(int64_t)row * ldc + col] = acc[rb][cb][j];
            }
        }
}

// The one-pass form for weights that are (f32 scale per super-block) x (small integer), see iq_dequant_int_kernel:
// C[m, n] = sum_sb Dt[sb][n] * ( sum_{k in sb} A16[m, k] * Q[n, k] ), A16 = the activations as fp16 (bf16 values convert exactly
// inside fp16's range), Q fp16 integers: every product is exact, the 256 products of a super-block are added in f32 by the matrix
// core, and the scale is applied once per super-block to the finished sum -- the reference's f32 GEMM on the dequantised
// weight up to summation order.  On the tiles of tile_gemm.h; blockIdx.y = slice of super-blocks (few tiles: down_proj, o_proj, short
// prompts), whose sums go to slices [M][N] of their own and are added in slice order by int_slices_kernel.
// GEGLU: Q holds `inter` gate rows, then `inter` up rows; a tile takes 64 of each, side by side in every wave, and stores
// act[m][i] = bf16(bf16(gelu_erf(bf16(gate))) * bf16(up)) as the fp16 operand of the next product (one slice).
// Against one 16-byte operand load per lane straight from global memory (no LDS), 256 rows x 30720 x 3840 (gate|up): 222 -> 107 us (566 TFLOP/s).
template <class S, bool GEGLU>
__global__ __launch_bounds__(S::THREADS) void int_tile_kernel(const uint16_t *__restrict__ A, const uint16_t *__restrict__ Q,
                                                               const float *__restrict__ Dt, float *__restrict__ C, uint16_t *__restrict__ act,
                                                               int M, int N, int K, int64_t ldc, int row_tiles, int tiles, int per_slice) {
    extern __shared__ __align__(1024) uint16_t tg_lds[];
    static_assert(!GEGLU || (S::WN == 2 && S::NJ == 2), "a wave holds 32 gate columns and the same 32 up columns");
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int tile = tg_tile(blockIdx.x, tiles);
    if (tile < 0) return;
    const int m0 = tile % row_tiles * S::BM, ct = tile / row_tiles, nsb = K >> 8, inter = N >> 1;
    const int sb0 = blockIdx.y * per_slice, groups = min(per_slice, nsb - sb0);
    // tile column -> row of Q
    auto q_row = [&](int c) {
        if constexpr (GEGLU) return (c & 32 ? inter : 0) + min(ct * 64 + (c >> 6) * 32 + (c & 31), inter - 1);
        else return min(ct * S::BN + c, N - 1);
    };
    uint32_t a_src[S::AQ], b_src[S::BQ];
#pragma unroll
    for (int q = 0; q < S::AQ; q++) a_src[q] = (uint32_t)((int64_t)min(m0 + tg_src_row<S::AQ>(wave, lane, q), M - 1) * K * 2) + tg_src_byte(lane);
#pragma unroll
    for (int q = 0; q < S::BQ; q++) b_src[q] = (uint32_t)((int64_t)q_row(tg_src_row<S::BQ>(wave, lane, q)) * K * 2) + tg_src_byte(lane);
    const int wc = wave % S::WN * (S::NJ * 32) + (lane & 31);   // this lane's column of the tile (and 32 j further on)
    int dcol[S::NJ];
#pragma unroll
    for (int j = 0; j < S::NJ; j++) dcol[j] = q_row(wc + 32 * j);
    tg_f32x16 acc[S::MI][S::NJ];
#pragma unroll
    for (int i = 0; i < S::MI; i++)
#pragma unroll
        for (int j = 0; j < S::NJ; j++) acc[i][j] = tg_f32x16{};
    const TgCore<true, S> core{(const char *)(A + sb0 * 256), (const char *)(Q + sb0 * 256), a_src, b_src, tg_lds_at(tg_lds), wave, lane};
    tg_product_scaled(core, groups, acc, [&](int g, float (&d)[S::NJ]) {
#pragma unroll
        for (int j = 0; j < S::NJ; j++) d[j] = Dt[(int64_t)(sb0 + g) * N + dcol[j]];
    });
    const int wm = m0 + wave / S::WN * (S::MI * 32);
    if constexpr (GEGLU) {
        const int col = ct * 64 + wave % S::WN * 32 + (lane & 31);
        if (col >= inter) return;
#pragma unroll
        for (int i = 0; i < S::MI; i++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int m = wm + 32 * i + tg_acc_row(lane, r);
                if (m >= M) continue;
                const float g = vmx_bf16_to_f32(vmx_f32_to_bf16(acc[i][0][r])), u = vmx_bf16_to_f32(vmx_f32_to_bf16(acc[i][1][r]));
                const float ge = vmx_bf16_to_f32(vmx_f32_to_bf16(0.5f * g * (1.0f + erff(g * 0.70710678118654752f))));
                act[(int64_t)m * inter + col] = bf16_value_to_f16(vmx_f32_to_bf16(ge * u));
            }
    } else {
        float *out = C + (int64_t)blockIdx.y * M * ldc;
#pragma unroll
        for (int j = 0; j < S::NJ; j++) {
            const int n = ct * S::BN + wc + 32 * j;
            if (n >= N) continue;
#pragma unroll
            for (int i = 0; i < S::MI; i++)
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const int m = wm + 32 * i + tg_acc_row(lane, r);
                    if (m < M) out[(int64_t)m * ldc + n] = acc[i][j][r];
                }
        }
    }
}

// y[m][n] (rows ldy apart) = the slices [slices][M][N] added in slice order, V elements a thread.  V = 4: N % 4 == 0, y and its rows on 16 bytes
// (a caller's output may be a view that starts anywhere).
template <int V>
__global__ __launch_bounds__(256) void int_slices_kernel(const float *__restrict__ part, float *__restrict__ y, int slices, int M, int N, int64_t ldy) {
    typedef float Vec __attribute__((ext_vector_type(V)));
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x, n_vec = (int64_t)M * N / V;
    if (i >= n_vec) return;
    Vec v = reinterpret_cast<const Vec *>(part)[i];
    for (int s = 1; s < slices; s++) v += reinterpret_cast<const Vec *>(part)[i + s * n_vec];
    const int64_t m = V * i / N, n = V * i - m * N;
    *reinterpret_cast<Vec *>(y + m * ldy + n) = v;
}

__global__ __launch_bounds__(256) void bf16_to_f16_kernel(uint16_t *__restrict__ out, const uint16_t *__restrict__ in, int64_t n8) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n8; i += (int64_t)gridDim.x * 256) {
        const uint4 v = reinterpret_cast<const uint4 *>(in)[i];
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
        uint32_t o[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            o[j] = (uint32_t)bf16_value_to_f16((uint16_t)w[j]) | ((uint32_t)bf16_value_to_f16((uint16_t)(w[j] >> 16)) << 16);
        }
        reinterpret_cast<uint4 *>(out)[i] = make_uint4(o[0], o[1], o[2], o[3]);
    }
}

// f32 rows [rows, K] -> bf16 rows [rows, 3K]: v = hi + lo with hi = bf16(v), lo = bf16(v - hi).  WEIGHT rows are laid out
// hi | hi | lo and ACTIVATION rows hi | lo | hi, so that one bf16 GEMM over 3K computes xhi.whi + xlo.whi + xhi.wlo: the
// f32 product short of the lo.lo term (2^-16 relative per factor pair, below the f32 summation noise of a long dot).
template <bool WEIGHT>
__global__ __launch_bounds__(256) void split3_rows_kernel(uint16_t *__restrict__ out, const float *__restrict__ in, int64_t rows, int K) {
    const int64_t n = rows * K;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
        const int64_t r = i / K;
        const int k = (int)(i - r * K);
        const float v = in[i];
        const uint16_t hi = vmx_f32_to_bf16(v), lo = vmx_f32_to_bf16(v - vmx_bf16_to_f32(hi));
        uint16_t *o = out + r * 3 * K;
        o[k] = hi;
        o[K + k] = WEIGHT ? hi : lo;
        o[2 * K + k] = WEIGHT ? lo : hi;
    }
}

}  // namespace

// QMatMul::forward beyond the 8-row vector kernels (candle's dequantize-and-matmul path behind QuantizedLinear,
// crates/core/src/quantization/gguf/mod.rs): the K-quant / legacy-block weight dequantised to dense f32, times f32 activations.
// workspace: f32 weight [N*K] | bf16 weight thirds [N, 3K] | bf16 activation thirds [M, 3K]
extern "C" size_t vmx_kquant_gemm_workspace_bytes(int m, int n_out, int n_in) {
    if (m <= 0 || n_out <= 0 || n_in <= 0) return 0;
    return (size_t)n_out * n_in * 4 + (size_t)n_out * n_in * 6 + (size_t)m * n_in * 6;
}

extern "C" int vmx_kquant_gemm_f32(int ggml_type, const void *w, const float *x, float *y, int m, int n_out, int n_in, void *workspace,
                                   size_t workspace_bytes, void *stream) {
    VMX_REQUIRE(w && x && y && workspace, "kquant_gemm: null pointer");
    VMX_REQUIRE(vmx_ggml_type_size(ggml_type) > 0 && vmx_iq_type_size(ggml_type) <= 0, "kquant_gemm: ggml type %d is not a K-quant / legacy block type",
                ggml_type);
    VMX_REQUIRE(m >= 0 && n_out > 0 && n_in > 0 && n_in % vmx_ggml_block_elems(ggml_type) == 0,
                "kquant_gemm: n_in (%d) must be a positive multiple of the block size", n_in);
    if (m == 0) return VMX_OK;
    VMX_REQUIRE(workspace_bytes >= vmx_kquant_gemm_workspace_bytes(m, n_out, n_in), "kquant_gemm: workspace of %zu bytes, need %zu",
                workspace_bytes, vmx_kquant_gemm_workspace_bytes(m, n_out, n_in));
    hipStream_t st = vmx_stream(stream);
    const int64_t nk = (int64_t)n_out * n_in;
    float *wf = (float *)workspace;
    uint16_t *w3 = (uint16_t *)(wf + nk), *x3 = w3 + 3 * nk;
    if (int rc = vmx_kquant_dequantize_f32(ggml_type, w, wf, nk / vmx_ggml_block_elems(ggml_type), stream)) return rc;
    const int gw = (int)std::min<int64_t>((nk + 255) / 256, 16384), gx = (int)std::min<int64_t>(((int64_t)m * n_in + 255) / 256, 16384);
    hipLaunchKernelGGL((split3_rows_kernel<true>), dim3(gw), dim3(256), 0, st, w3, wf, (int64_t)n_out, n_in);
    hipLaunchKernelGGL((split3_rows_kernel<false>), dim3(gx), dim3(256), 0, st, x3, x, (int64_t)m, n_in);
    const int K3 = 3 * n_in;
    const int wide_wgs = ((n_out + 255) / 256) * ((m + 63) / 64);
    if (wide_wgs < 2 * vmx_num_cus() && K3 % 128 == 0)
        hipLaunchKernelGGL((split_gemm_kernel<false, true>), dim3((n_out + 63) / 64, (m + 63) / 64), dim3(256), 0, st, x3, w3, w3, y, m, n_out, K3, n_out);
    else
        hipLaunchKernelGGL((split_gemm_kernel<false, false>), dim3((n_out + 255) / 256, (m + 63) / 64), dim3(256), 0, st, x3, w3, w3, y, m, n_out, K3, n_out);
    VMX_CHECK_LAUNCH("kquant_gemm");
    return VMX_OK;
}

size_t vmx_iq_gemm_workspace(int N, int K) { return (size_t)N * K * 4; }   // the two bf16 halves

// workspace -> (hi bf16 [N*K], lo bf16 [N*K])
int vmx_iq_dequant_split(int ggml_type, const void *blocks, void *workspace, int N, int K, hipStream_t st) {
    const int64_t n = (int64_t)N * K;
    uint16_t *hi = (uint16_t *)workspace, *lo = hi + n;
    return vmx_iq_dequantize_split_bf16(ggml_type, blocks, hi, lo, n / 256, st);
}

// C[:, 0..N) (row stride ldc) = A @ (hi + lo)^T with the halves a previous vmx_iq_dequant_split left in `workspace`
int vmx_split_gemm_f32(const uint16_t *A, const void *workspace, float *C, int M, int N, int K, int ldc, hipStream_t st) {
    const int64_t n = (int64_t)N * K;
    const uint16_t *hi = (const uint16_t *)workspace, *lo = hi + n;
    // under about two workgroups per compute unit the four waves of a workgroup split K over one 64 x 64 tile instead
    const int wide_wgs = ((N + 255) / 256) * ((M + 63) / 64);
    if (wide_wgs < 2 * vmx_num_cus() && K % 128 == 0 && K >= 1024)
        hipLaunchKernelGGL((split_gemm_kernel<true, true>), dim3((N + 63) / 64, (M + 63) / 64), dim3(256), 0, st, A, hi, lo, C, M, N, K, ldc);
    else
        hipLaunchKernelGGL((split_gemm_kernel<true, false>), dim3((N + 255) / 256, (M + 63) / 64), dim3(256), 0, st, A, hi, lo, C, M, N, K, ldc);
    VMX_CHECK_LAUNCH("split_gemm");
    return VMX_OK;
}

// ---- the integer form: workspace = Q fp16 [N*K] | Dt f32 [K/256][N] | A16 fp16 [M*K]
size_t vmx_iq_gemm_int_weight_bytes(int N, int K) { return (size_t)N * K * 2 + (((size_t)N * (K / 256) * 4 + 255) & ~(size_t)255); }
size_t vmx_iq_gemm_int_workspace(int M, int N, int K) { return vmx_iq_gemm_int_weight_bytes(N, K) + (size_t)M * K * 2; }

// rows [row0, row0 + rows) of the integer form of N rows
int vmx_iq_dequant_int(int ggml_type, const void *blocks, void *workspace, int row0, int rows, int N, int K, hipStream_t st) {
    uint16_t *Q = (uint16_t *)workspace;
    float *Dt = (float *)(Q + (int64_t)N * K);
    return vmx_iq_dequantize_int_f16(ggml_type, blocks, Q + (int64_t)row0 * K, Dt + row0, rows, N, K / 256, st);
}

// a16: fp16 copy of the activations (vmx_bf16_rows_to_f16), shared by the linears that read the same rows
int vmx_bf16_rows_to_f16(const uint16_t *A, uint16_t *a16, int64_t n, hipStream_t st) {
    const int64_t n8 = n / 8;
    if (n8 <= 0) return VMX_OK;
    hipLaunchKernelGGL(bf16_to_f16_kernel, dim3((unsigned)std::min<int64_t>((n8 + 255) / 256, 4096)), dim3(256), 0, st, a16, A, n8);
    VMX_CHECK_LAUNCH("bf16_to_f16");
    return VMX_OK;
}

namespace {
typedef TgShape<2, 2, 2, 2, 2> IntWide;     // 128 x 128
typedef TgShape<2, 2, 1, 2, 2> IntMid;      // 64 x 128
typedef TgShape<2, 2, 1, 1, 2> IntSmall;    // 64 x 64

template <class S, bool GEGLU>
void launch_int_tile(const uint16_t *a16, const uint16_t *Q, const float *Dt, float *C, uint16_t *act, int M, int N, int K, int64_t ldc, int slices,
                     hipStream_t st) {
    const int row_tiles = (M + S::BM - 1) / S::BM, tiles = row_tiles * (GEGLU ? (N / 2 + 63) / 64 : (N + S::BN - 1) / S::BN);
    const int nsb = K / 256, per_slice = (nsb + slices - 1) / slices;
    hipLaunchKernelGGL((int_tile_kernel<S, GEGLU>), dim3(tg_grid(tiles), (nsb + per_slice - 1) / per_slice), dim3(S::THREADS), S::LDS, st, a16, Q, Dt, C,
                       act, M, N, K, ldc, row_tiles, tiles, per_slice);
}

// Rows of a tile: 128 where there are more than 32 such tiles.  Whole call in us, 128 / 64 rows (slices as below): 4096 columns x 2048, 100 rows
// 33.2 / 32.0, 200 rows 26.8 / 31.0;  2048 x 3840, 65 rows 33.6 / 31.8, 400 rows 30.5 / 31.7;  3840 x 15360, 128 rows 62.6 / 59.7, 256 rows
// 73.3 / 75.5, 400 rows 102 / 109.
int int_rows(int M, int N) { return M > 64 && (int64_t)((M + 127) / 128) * ((N + 127) / 128) > 32 ? 128 : 64; }

// Slices of super-blocks, at most `most`, that give every compute unit about two workgroups.  Without them a product with few tiles walks its K
// alone (one / all slices: 3840 x 3840, 100 rows 56 / 30 us, 2048 x 3840 50 / 32, 512 x 2048 25 / 15).
int int_slices(int M, int N, int K, int64_t most) {
    const int rows = int_rows(M, N), nsb = K / 256;
    const int64_t tiles = (int64_t)((M + rows - 1) / rows) * ((N + 127) / 128), want = std::min(2 * (int64_t)vmx_num_cus() / tiles, most);
    if (want <= 1) return 1;
    const int per = (int)((nsb + want - 1) / want);
    return (nsb + per - 1) / per;
}

// A short K is a chain of few stages whose latency the tile's size decides: below eight super-blocks tiles are 64 x 64, up to four a compute unit.
// us, 128- or 64-row tiles as above uncut / 64 x 64 tiles with the slices below: 17 x 512 x 1024 17.9 / 13.3, 65 x 8192 x 1024 31.3 / 26.7, 200 x 4096 x
// 1024 25.2 / 20.7, 600 x 4096 x 1024 26.9 / 23.3, 400 x 2048 x 1280 29.8 / 21.2, 1000 x 2048 x 512 18.7 / 15.9; six tiles a unit no longer, 1200 x 8192 x
// 1024 45.8 / 47.2.  From eight super-blocks on slices hide the latency: 200 x 4096 x 2048 28.5 / 30.9, 400 x 4096 x 4096 41.9 / 43.6.
bool int_short(int M, int N, int K) { return K < 8 * 256 && (int64_t)((M + 63) / 64) * ((N + 63) / 64) <= 4 * vmx_num_cus(); }

// Its slices: the count with the least estimated time of 1.6 us a super-block (1.9 with two workgroups a unit) and, for more than one, of a
// launch and the f32 sums written and read.  1024 deep, one / two / four slices in us: 17 x 512 16.0 / 14.5 / 13.3, 200 x 1024 17.1 / 16.0 / 15.5,
// 65 x 4096 20.1 / 19.6 / 19.8, 400 x 2048 18.8 / 20.7 / 24.1; 512 deep, 17 x 2048 12.9 / 13.2.
int int_short_slices(int M, int N, int K, int64_t most) {
    const int nsb = K / 256, tiles = ((M + 63) / 64) * ((N + 63) / 64), cus = vmx_num_cus();
    int best = 1;
    int64_t least = nsb * (tiles > cus ? 1900 : 1600);
    for (int s = 2; s <= nsb && s <= most && tiles * s <= 2 * cus; s++) {
        const int per = (nsb + s - 1) / s;
        const int64_t ns = per * (tiles * s > cus ? 1900 : 1600) + 1700 + (int64_t)s * M * N * 8 / 5000;
        if ((nsb + per - 1) / per == s && ns < least) least = ns, best = s;
    }
    return best;
}
}  // namespace

// most bytes of slice sums any call can want: int_slices gives at most two tiles a compute unit, of at most 128 x 128 sums
size_t vmx_int_gemm_part_bytes() { return (size_t)2 * vmx_num_cus() * 128 * 128 * 4; }

bool vmx_int_gemm_ok(int M, int N, int K) { return (int64_t)M * K * 2 < (int64_t)1 << 32 && (int64_t)N * K * 2 < (int64_t)1 << 32; }

int vmx_int_slices(const float *part, float *y, int slices, int M, int N, int64_t ldy, hipStream_t st) {
    const bool wide = N % 4 == 0 && ldy % 4 == 0 && ((uintptr_t)y & 15) == 0;
    const dim3 grid((unsigned)(((int64_t)M * N / (wide ? 4 : 1) + 255) / 256));
    if (wide) hipLaunchKernelGGL(int_slices_kernel<4>, grid, dim3(256), 0, st, part, y, slices, M, N, ldy);
    else hipLaunchKernelGGL(int_slices_kernel<1>, grid, dim3(256), 0, st, part, y, slices, M, N, ldy);
    VMX_CHECK_LAUNCH("int_slices");
    return VMX_OK;
}

// part: scratch for slices, as many as fit part_bytes; vmx_int_gemm_part_bytes() hold all that are wanted
int vmx_int_gemm_f32(const uint16_t *a16, const void *workspace, float *C, int M, int N, int K, int ldc, float *part, size_t part_bytes, hipStream_t st) {
    const uint16_t *Q = (const uint16_t *)workspace;
    const float *Dt = (const float *)(Q + (int64_t)N * K);
    const int64_t fit = (int64_t)(part_bytes / ((size_t)M * N * 4));
    const bool brief = int_short(M, N, K);
    const int slices = brief ? int_short_slices(M, N, K, fit) : int_slices(M, N, K, fit);
    float *to = slices > 1 ? part : C;
    const int64_t ld = slices > 1 ? N : ldc;
    if (brief) launch_int_tile<IntSmall, false>(a16, Q, Dt, to, nullptr, M, N, K, ld, slices, st);
    else if (int_rows(M, N) == 128) launch_int_tile<IntWide, false>(a16, Q, Dt, to, nullptr, M, N, K, ld, slices, st);
    else launch_int_tile<IntMid, false>(a16, Q, Dt, to, nullptr, M, N, K, ld, slices, st);
    if (slices > 1)
        if (int rc = vmx_int_slices(part, C, slices, M, N, ldc, st)) return rc;
    VMX_CHECK_LAUNCH("int_gemm");
    return VMX_OK;
}

// act16 [M][inter] (fp16) of the gate rows and up rows that `workspace` holds one behind the other (N = 2 inter)
int vmx_int_gemm_geglu(const uint16_t *a16, const void *workspace, uint16_t *act, int M, int inter, int K, hipStream_t st) {
    const int N = 2 * inter;
    const uint16_t *Q = (const uint16_t *)workspace;
    const float *Dt = (const float *)(Q + (int64_t)N * K);
    if (int_rows(M, N) == 128) launch_int_tile<IntWide, true>(a16, Q, Dt, nullptr, act, M, N, K, 0, 1, st);
    else launch_int_tile<IntMid, true>(a16, Q, Dt, nullptr, act, M, N, K, 0, 1, st);
    VMX_CHECK_LAUNCH("int_gemm(geglu)");
    return VMX_OK;
}

extern "C" size_t vmx_iq_gemm_workspace_bytes(int n_out, int n_in) {
    if (n_out <= 0 || n_in <= 0) return 0;
    // what the product must have, and room for the slices of one with few tiles
    const size_t least = vmx_iq_gemm_workspace(n_out, n_in);
    return least + std::min(least, vmx_int_gemm_part_bytes());
}

extern "C" int vmx_iq_gemm_f32(int ggml_type, const void *blocks, const uint16_t *x, float *y, int m, int n_out, int n_in, void *workspace,
                               size_t workspace_bytes, void *stream) {
    VMX_REQUIRE(blocks && x && y && workspace, "iq_gemm: null pointer");
    VMX_REQUIRE(vmx_iq_type_size(ggml_type) > 0, "iq_gemm: ggml type %d is not a supported I-quant", ggml_type);
    VMX_REQUIRE(m >= 0 && n_out > 0 && n_in > 0 && n_in % 256 == 0, "iq_gemm: n_in (%d) must be a positive multiple of 256", n_in);
    VMX_REQUIRE(workspace_bytes >= vmx_iq_gemm_workspace(n_out, n_in), "iq_gemm: workspace of %zu bytes, need %zu", workspace_bytes,
                vmx_iq_gemm_workspace(n_out, n_in));
    if (m == 0) return VMX_OK;
    hipStream_t st = vmx_stream(stream);
    // Activations go to fp16 (which saturates and loses small values) only where the workspace has always allowed it, whichever of the two products then runs
    const bool int_form = vmx_iq_int_form_ok(ggml_type) && workspace_bytes >= vmx_iq_gemm_int_workspace(m, n_out, n_in) && vmx_int_gemm_ok(m, n_out, n_in);
    const VmxMmvqSeg seg = {blocks, ggml_type, n_out, 0};
    if (int_form && vmx_iq_prompt_alone_ok(seg, m, n_in)) {   // decoded inside the product: the workspace holds the rows, then slice sums
        const size_t rows = ((size_t)m * n_in * 2 + 255) & ~(size_t)255;   // fewer than the weights' integer form takes, besides these rows
        if (int rc = vmx_bf16_rows_to_f16(x, (uint16_t *)workspace, (int64_t)m * n_in, st)) return rc;
        return vmx_iq_prompt_f32(&seg, 1, (const uint16_t *)workspace, y, m, n_in, n_out, (float *)((char *)workspace + rows), workspace_bytes - rows, st);
    }
    if (int_form) {
        // exact one-pass form: integer weights in fp16, one f32 scale per super-block; slice sums where the workspace has room for them
        uint16_t *a16 = (uint16_t *)((char *)workspace + vmx_iq_gemm_int_workspace(0, n_out, n_in));
        const size_t used = (vmx_iq_gemm_int_workspace(m, n_out, n_in) + 255) & ~(size_t)255;
        const size_t room = workspace_bytes > used ? workspace_bytes - used : 0;
        if (int rc = vmx_iq_dequant_int(ggml_type, blocks, workspace, 0, n_out, n_out, n_in, st)) return rc;
        if (int rc = vmx_bf16_rows_to_f16(x, a16, (int64_t)m * n_in, st)) return rc;
        return vmx_int_gemm_f32(a16, workspace, y, m, n_out, n_in, n_out, (float *)((char *)workspace + used), room, st);
    }
    if (int rc = vmx_iq_dequant_split(ggml_type, blocks, workspace, n_out, n_in, st)) return rc;
    return vmx_split_gemm_f32(x, workspace, y, m, n_out, n_in, n_out, st);
}
