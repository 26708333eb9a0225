"""Normed unquantised products of up to 16 rows in every form they have: one, two and up to four pieces of the rows a thread requests ahead, few and many workgroups, one
block of weights a wave, two, more and none, rows too long for LDS; against float64."""
import ctypes as C

import pytest

pytestmark = pytest.mark.gpu


# pieces are M K / 8 over 512 threads (K <= 512: 256), rounded up; above 1024 workgroups of 16 columns three pieces take the form of two; M (K + 8) > 16512: rows not staged
@pytest.mark.parametrize("glu", [False, True])
@pytest.mark.parametrize("M,N,K", [
    (1, 32, 192), (16, 32, 512), (9, 48, 320), (4, 32, 1024), (5, 32, 896), (8, 32, 1024), (16, 48, 1024), (13, 32, 960),          # four or eight waves of a block
    (1, 32, 1152), (2, 4096, 1536), (6, 64, 1536), (8, 32, 2048), (8, 16416, 1536), (6, 16400, 2048), (8, 16416, 2048), (7, 16400, 1280),   # eight waves, nine to 16 blocks
    (1, 32, 2112), (1, 48, 16448), (2, 32, 2560), (3, 16400, 4096), (4, 48, 4096), (1, 16, 5184),                                                 # more than two blocks a wave
    (16, 32, 1152), (8, 32, 2112), (9, 64, 4096), (16, 32, 2048),                                                                 # rows not staged
])
def test_matches_float64(M, N, K, glu):
    """A normed value is rounded to bf16 (2^-9 of itself, or one more step where the f32 statistic moves it over a boundary), so the result is off by about 2^-9 / sqrt(3) of
    its norm, at most by 2^-8 of the sum of magnitudes; the sums' own rounding is K 2^-24 of that.  Bounds: 2^-8 of the norm, 2^-8 + K 2^-24 of the magnitudes; the gated
    product's three roundings to bf16 add 3 2^-8 of the result, and its slopes are at most 1.1 max(1, |up|)."""
    import torch
    import vllm_rust_amd as vmx
    from vllm_rust_amd._lib import check, lib
    vmx.init(0)
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    h = (torch.randn(M, K, device="cuda", generator=g) * 2).bfloat16()
    gain = (1 + 0.1 * torch.randn(K, device="cuda", generator=g)).bfloat16()
    w = (torch.randn(N, K, device="cuda", generator=g) * K ** -0.5).bfloat16()
    ssq = (h.float() ** 2).reshape(M, K // 16, 16).sum(-1).contiguous()   # of tiles of 16, as the product before leaves them
    guard = torch.full((M + 2, N // 2 if glu else N), 3.0, device="cuda", dtype=torch.bfloat16 if glu else torch.float32)
    y = guard[1:M + 1]
    f = lib._Z25vmx_dense_decode_norm_gluPtPKtS1_fPKfiS1_iiiP12ihipStream_t if glu else lib._Z25vmx_dense_decode_norm_f32PfPKtS1_fPKfiS1_iiiP12ihipStream_t
    f.argtypes, f.restype = [C.c_void_p] * 3 + [C.c_float, C.c_void_p, C.c_int, C.c_void_p] + [C.c_int] * 3 + [C.c_void_p], C.c_int
    check(f(y.data_ptr(), h.data_ptr(), gain.data_ptr(), 1e-6, ssq.data_ptr(), K // 16, w.data_ptr(), M, N, K, torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    hd = h.double()
    x = hd / torch.sqrt((hd * hd).mean(-1, keepdim=True) + 1e-6) * gain.double()
    want, size = x @ w.double().T.contiguous(), x.abs() @ w.double().abs().T.contiguous()
    off = (2.0 ** -8 + K * 2.0 ** -24) * size
    if glu:
        gate, up = want[:, :N // 2], want[:, N // 2:]
        off = 1.1 * (off[:, :N // 2] * up.abs() + off[:, N // 2:] * (gate.abs() + 1))
        want = gate * torch.sigmoid(gate) * up
        off = off + 3 * 2.0 ** -8 * (want.abs() + off)
    d = (y.double() - want).abs()
    assert bool((d <= off).all())
    assert d.norm().item() <= (4 if glu else 1) * 2.0 ** -8 * want.norm().item()
    assert bool((guard[0] == 3.0).all()) and bool((guard[M + 1] == 3.0).all())
