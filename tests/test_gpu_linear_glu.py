"""Products with a clamped gated activation behind their sums against the same sums stored as f32 and the activation in float64: the sums of a column do not
depend on the form, so what may differ is the f32 activation and a rounding to bf16."""
import ctypes as C

import pytest

pytestmark = pytest.mark.gpu


# one and sixteen rows, one above, around the tiles of 64 .. 256 rows; F below, at and above the columns of a workgroup (8) and of a tile (64), many
@pytest.mark.parametrize("rows", ["bf16", "f32"])
@pytest.mark.parametrize("out", ["f32", "bf16"])
@pytest.mark.parametrize("M,F,K", [(1, 8, 64), (16, 24, 200), (5, 4104, 256), (16, 6144, 2048), (16, 64, 1032), (17, 8, 64), (63, 72, 128), (65, 56, 192), (129, 1000, 64),
                                   (193, 3072, 320), (300, 6144, 64), (1025, 2056, 128)])
def test_linear_glu(M, F, K, out, rows):
    import torch
    import vllm_rust_amd as vmx
    from tests.test_gpu_tile_gemm import _Linear
    from vllm_rust_amd._lib import VmxError, check, lib
    vmx.init(0)
    slope, limit = 1.702, 7.0
    g = torch.Generator(device="cuda").manual_seed(M * 31 + F + K)
    x = (torch.randn((M, K), device="cuda", generator=g) * 4).to(torch.float32 if rows == "f32" else torch.bfloat16)   # sums beyond the limits on both sides
    w = (torch.randn((2 * F, K), device="cuda", generator=g) * K ** -0.5).to(torch.bfloat16)
    guard = torch.full((M + 2, F), 3.0, device="cuda", dtype=torch.float32 if out == "f32" else torch.bfloat16)
    y = guard[1:M + 1]
    p = _Linear(A=x.data_ptr(), a_f32=rows == "f32", lda=K, W=w.data_ptr(), w_sn=K, w_sk=1, C=y.data_ptr(), c_f32=out == "f32", ldc=F, M=M, N=2 * F, K=K, batch=1,
                row_div=1, aux_sn=1, out_scale=1.0)
    lib.vmx_linear_glu.argtypes, lib.vmx_linear_glu.restype = [C.c_void_p, C.c_float, C.c_float, C.c_void_p], C.c_int
    run = lambda: check(lib.vmx_linear_glu(C.byref(p), slope, limit, C.c_void_p(torch.cuda.current_stream().cuda_stream)))   # noqa: E731
    if M > 16 and rows == "f32":   # no such tiles: refused, the caller takes two launches
        with pytest.raises(VmxError, match="no gated epilogue"):
            run()
        return
    run()
    sums = torch.empty((M, 2 * F), device="cuda")
    check(lib.vmx_linear_bf16w(sums.data_ptr(), 0, x.data_ptr(), 0 if rows == "f32" else 1, w.data_ptr(), M, 2 * F, K, 0, torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    a, b = sums[:, :F].double().clamp(max=limit), sums[:, F:].double().clamp(-limit, limit)
    ref = a * torch.sigmoid(slope * a) * (b + 1)
    # sums of up to 16 rows come from forms with other orders of k: their f32 rounding, through slopes of at most 2 (limit + 1)
    loose = (K + 8) * 2.0 ** -24 * 4 * K ** 0.5 * 2 * (limit + 1) if M <= 16 else 0.0
    # f32 activation: the exponent's product is off by |slope a| 2^-24, which is that much of the exponential, and exponential, sum, quotient and the two products
    # by a few 2^-24 each; u + 1 by 2^-24 of its size before it cancels
    act = 2.0 ** -22 * ((2 + slope * a.abs()) * ref.abs() + (a * torch.sigmoid(slope * a)).abs() * (1 + b.abs()))
    bound = loose + act + (2.0 ** -8 * ref.abs() if out == "bf16" else 0) + 2.0 ** -40
    assert bool(((y.double() - ref).abs() <= bound).all())
    assert bool((guard[0] == 3.0).all()) and bool((guard[M + 1] == 3.0).all())
