"""Unquantised products of 5 .. 16 rows on the matrix cores, activations staged 1024 deep: one block of 128, a pass and a block, whole passes, odd numbers of
columns; an infinite weight stays in its column; against float64."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K", [(5, 17, 128), (16, 33, 256), (7, 100, 896), (16, 64, 1024), (9, 65, 1152), (16, 1000, 2048), (6, 250, 2560), (16, 47, 4096), (13, 130, 5248)])
def test_matches_float64(M, N, K):
    """Products are exact in f32 and each of the K sums rounds once, so the sum is off by at most K 2^-24 of the sum of magnitudes, and storing it rounds by less than 2^-8 of it."""
    import torch
    import vllm_rust_amd as vmx
    vmx.init(0)
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x, W = torch.randn(M, K, device="cuda", generator=g).bfloat16(), torch.randn(N, K, device="cuda", generator=g).bfloat16()
    if N > 20:
        W[3, K - 1] = float("inf")   # one column's: the others stay finite, also those behind the last block
    y = vmx.dense_gemv(x, W)
    exact = x.double() @ W.double().T.contiguous()
    bound = K * 2.0 ** -24 * (x.double().abs() @ W.double().abs().T.contiguous()) + 2.0 ** -8 * exact.abs()
    keep = torch.ones(N, dtype=torch.bool, device="cuda")
    if N > 20:
        keep[3] = False
        assert torch.equal(y[:, 3].double(), exact[:, 3])
    assert torch.isfinite(y[:, keep]).all()
    assert ((y.double() - exact).abs() <= bound)[:, keep].all()


# up to 16384 columns are one workgroup a compute unit at most; one column more and it is the other kernel: last tiles and workgroups that are part empty, odd and even
# rows, one pass, a pass and some blocks, several
@pytest.mark.parametrize("M,N,K", [(16, 16384, 256), (5, 16385, 128), (16, 16385, 1024), (8, 16447, 1152), (13, 20001, 896), (7, 33000, 640), (6, 16448, 4096), (11, 270001, 128)])
def test_more_workgroups_than_compute_units(M, N, K):
    """As above, with its bound."""
    test_matches_float64(M, N, K)
