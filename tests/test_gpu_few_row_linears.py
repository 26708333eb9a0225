"""Linears of up to 16 rows whose waves have no block of K, one, two or more, with columns below and above two groups of 16 a compute unit; against float64."""
import ctypes as C

import pytest

pytestmark = pytest.mark.gpu


def _launch(torch, x, w, y):
    from tests.helpers import launched_kernels
    from tests.test_gpu_tile_gemm import _Linear
    from vllm_rust_amd._lib import check, lib
    B, M, K = x.shape
    N = w.shape[1]
    rows, out = x.transpose(0, 1).reshape(M, B * K).contiguous(), y
    p = _Linear(A=rows.data_ptr(), a_f32=x.dtype == torch.float32, lda=B * K, a_bs=K, W=w.data_ptr(), w_sn=K, w_sk=1, w_bs=N * K, C=out.data_ptr(), c_f32=1, ldc=B * N, c_bs=N,
                M=M, N=N, K=K, batch=B, row_div=1, aux_sn=1, out_scale=1.0)
    run = lambda: check(lib.vmx_linear_launch(C.byref(p), C.c_void_p(torch.cuda.current_stream().cuda_stream)))   # noqa: E731
    (name,) = [k for k, *_ in launched_kernels(torch, run)]
    run()
    torch.cuda.synchronize()
    return name


@pytest.mark.parametrize("M", [1, 9, 16])
@pytest.mark.parametrize("rows", ["f32", "bf16"])
@pytest.mark.parametrize("B,N,K", [
    (1, 40, 8), (1, 8200, 64), (32, 512, 96), (1, 8208, 320), (3, 3000, 512),           # at most a block of 128 for each of four waves
    (1, 8208, 520), (1, 8192, 576), (1, 8192, 1024), (1, 8200, 1160), (2, 4100, 2112),  # two and more, many columns
    (1, 4096, 1032), (1, 4100, 2200), (1, 4096, 640),                                   # one to two groups of columns a unit: up to eight waves
    (1, 2048, 1000), (1, 2000, 1048), (1, 300, 2112), (1, 2048, 4104), (1, 130, 6144),  # eight columns a workgroup, k in halves
])
def test_matches_float64(B, N, K, rows, M):
    """Products of bf16 are exact in f32; an f32 sum of K of them is off by at most (K + 8) 2^-24 of the sum of magnitudes.  What lies behind the last row and column of a
    product is not written."""
    import torch
    import vllm_rust_amd as vmx
    vmx.init(0)
    g = torch.Generator(device="cuda").manual_seed(N + K + M)
    x = torch.randn((B, M, K), device="cuda", generator=g)
    x = x if rows == "f32" else x.to(torch.bfloat16)
    w = torch.randn((B, N, K), device="cuda", generator=g).to(torch.bfloat16)
    guard = torch.full((M + 1, B * N), 3.0, device="cuda")
    _launch(torch, x, w, guard)
    xd, wd = x.to(torch.bfloat16).double(), w.double().transpose(1, 2).contiguous()
    want, size = torch.bmm(xd, wd), torch.bmm(xd.abs(), wd.abs())
    got = guard[:M].reshape(M, B, N).transpose(0, 1).double()
    assert bool(((got - want).abs() <= (K + 8) * 2.0 ** -24 * size).all())
    assert bool((guard[M] == 3.0).all())


@pytest.mark.parametrize("B,N,K,deep", [(1, 12288, 64, False), (32, 512, 320, False), (1, 32000, 512, False), (1, 12288, 520, True)])
def test_shallow_products_take_the_form_of_one_block_a_wave(B, N, K, deep):
    """Up to four blocks of 128 are one for each of four waves, whatever the columns: a second block's registers and requests cost products of many columns up to a third."""
    import torch
    import vllm_rust_amd as vmx
    vmx.init(0)
    x, w = torch.zeros((B, 2, K), device="cuda", dtype=torch.bfloat16), torch.zeros((B, N, K), device="cuda", dtype=torch.bfloat16)
    name = _launch(torch, x, w, torch.empty((2, B * N), device="cuda"))
    assert ("linear_skinny_kernelILi4ELi1ELi2E" if deep else "linear_skinny_kernelILi4ELi1ELi1E") in name, name
