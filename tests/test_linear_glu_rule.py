"""When a gated product takes its activation behind its sums and when it takes two launches (host arithmetic, no GPU): vmx_linear_glu_pays."""
import ctypes as C

import pytest


# [rows, gate and up columns, depth]: us of two launches and of one, weights out of memory, on 256 compute units
@pytest.mark.parametrize("M,N,K,two,one", [
    (1, 12288, 2048, 16.7, 12.2), (16, 24576, 4096, 55.0, 52.8), (16, 2048, 512, 6.8, 3.7),
    (17, 12288, 2048, 15.8, 20.2), (64, 12288, 2048, 17.1, 20.8), (65, 12288, 2048, 21.1, 19.8), (128, 12288, 2048, 23.1, 20.6), (129, 12288, 2048, 22.6, 26.9),
    (256, 12288, 2048, 28.1, 30.3), (257, 12288, 2048, 33.0, 28.1), (1500, 12288, 2048, 102.0, 87.4), (2000, 12288, 2048, 122.6, 102.9),
    (17, 16384, 3072, 22.4, 29.3), (65, 16384, 3072, 30.7, 28.9), (192, 16384, 3072, 38.1, 47.0), (257, 16384, 3072, 46.3, 41.5),
    (64, 24576, 4096, 50.7, 47.5), (128, 24576, 4096, 58.8, 62.6), (129, 24576, 4096, 60.0, 56.5),
    (17, 6144, 1024, 9.6, 11.7), (128, 6144, 1024, 10.8, 11.8), (129, 6144, 1024, 13.1, 11.4), (333, 6144, 1024, 18.3, 12.9),
    (64, 2816, 2048, 14.3, 18.7), (300, 2816, 2048, 14.8, 18.5), (400, 2816, 2048, 20.3, 18.2), (850, 2816, 2048, 24.6, 21.0),
])
def test_the_faster_side(M, N, K, two, one):
    from tests.test_gpu_tile_gemm import _Linear
    from vllm_rust_amd._lib import lib
    p = _Linear(lda=K, w_sn=K, w_sk=1, ldc=N // 2, M=M, N=N, K=K, batch=1, row_div=1, aux_sn=1, out_scale=1.0)
    assert lib.vmx_linear_glu_pays(C.byref(p)) == (one < two)
