"""int4 products that only models call, each against float64 on the operands it multiplies: the pass of a few rows behind the last whole prompt tile, and the linears
of 5 .. 16 rows that end in the residual stream and those that read it.

Bounds.  Weights are s (q - z) with q and z of 4 bits.  A k-block of 128 is summed in f32 from terms of up to 31 |x| (16 + q), the zero's share likewise, then scaled; K / 128
blocks, waves and slices are added: a sum is off by at most (128 + K / 128 + 16) 2^-24 64 s |x| summed over k."""
import ctypes as C

import pytest

pytestmark = pytest.mark.gpu
GROUP = 128


@pytest.fixture(scope="module")
def gpu():
    import torch
    import vllm_rust_amd as vmx
    vmx.init(0)
    return vmx, torch


class _Weights:
    """[K, N] in both forms; paired: columns in the order of a merged gate | up linear, eight of each in turn."""

    def __init__(self, vmx, torch, K, N, seed, paired=False):
        g = torch.Generator(device="cuda").manual_seed(seed)
        q = torch.randint(0, 16, (K, N), device="cuda", generator=g)
        z = torch.randint(0, 16, (K // GROUP, N), device="cuda", generator=g)
        s = ((0.5 + torch.rand((K // GROUP, N), device="cuda", generator=g)) / (8 * K ** 0.5)).to(torch.bfloat16)
        self.K, self.N, self.torch = K, N, torch
        self.w = ((q - z.repeat_interleave(GROUP, 0)).double() * s.double().repeat_interleave(GROUP, 0)).T.contiguous()   # [N, K]
        self.s = s.double().repeat_interleave(GROUP, 0).T.contiguous()
        if paired:
            order = torch.arange(N, device="cuda").reshape(2, N // 16, 8).transpose(0, 1).reshape(-1)
            q, z, s = q[:, order], z[:, order], s[:, order]
        shift = 4 * torch.arange(8, device="cuda")

        def words(nibbles):   # [.., 8] -> int32
            v = (nibbles << shift).sum(-1)
            return torch.where(v >= 2 ** 31, v - 2 ** 32, v).to(torch.int32).contiguous()
        qw = words(q.reshape(K // 8, 8, N).transpose(1, 2))
        qz = words(z.reshape(K // GROUP, N // 8, 8))
        self.packed = vmx.int4_pack(qw, s.view(torch.int16).contiguous(), qz, K, N, GROUP)

    def product(self, x):
        """x W and how far an f32 sum may be from it."""
        y = x.double() @ self.w.T
        return y, (128 + self.K / 128 + 16) * 2.0 ** -24 * 64 * (x.double().abs() @ self.s.T)


def _rows(torch, M, K, seed):
    """Rows of different sizes, some with a few large elements."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn((M, K), device="cuda", generator=g) * torch.exp2(torch.randint(-3, 4, (M, 1), device="cuda", generator=g).float())
    x[:, 7::509] *= 30
    return x.to(torch.bfloat16)


def _glu(torch, gu, err):
    """bf16(silu(bf16 gate) bf16 up) and its bound: an f32 sum may fall on the other side of a rounding (2^-8 of it), two products are rounded."""
    F = gu.shape[1] // 2
    g, u, eg, eu = gu[:, :F], gu[:, F:], err[:, :F] + 2.0 ** -8 * gu[:, :F].abs(), err[:, F:] + 2.0 ** -8 * gu[:, F:].abs()
    silu = g * torch.sigmoid(g)
    ref = silu * u
    return ref, 1.1 * eg * (u.abs() + eu) + silu.abs() * eu + 2.0 ** -7 * ref.abs() + 2.0 ** -30


def _p(t):
    return C.c_void_p(t.data_ptr())


@pytest.mark.parametrize("tail", [1, 4, 5, 16, 17])
@pytest.mark.parametrize("full,N,K,slices", [(512, 7424, 2048, 2), (512, 4864, 6144, 3)])
def test_tail_in_slices(gpu, tail, full, N, K, slices):
    """Tiles alone would leave one slice less: as many as the plan has says that the tail took a pass of its own, 17 rows take none."""
    vmx, torch = gpu
    from vllm_rust_amd._lib import check, lib
    M = full + tail
    assert lib._Z20vmx_int4_splits_rowsiii(M, N, K) == (slices if tail <= 16 else slices - 1)
    slices -= tail > 16
    w, x = _Weights(vmx, torch, K, N, tail + N), _rows(torch, M, K, tail)
    out = torch.full((slices * M + 1, N), float("nan"), device="cuda")
    check(lib._Z21vmx_int4_gemm_partialPKvPKtPfiiiiP12ihipStream_t(_p(w.packed), _p(x), _p(out), M, N, K, GROUP, None))
    torch.cuda.synchronize()
    ref, err = w.product(x)
    assert bool(((out[:-1].double().reshape(slices, M, N).sum(0) - ref).abs() <= err).all())
    assert bool(out[-1].isnan().all())


@pytest.mark.parametrize("tail", [1, 4, 5, 16, 17])
@pytest.mark.parametrize("full,N,K", [(320, 12288, 2048), (320, 12288, 4096)])
def test_tail_of_gate_and_up(gpu, tail, full, N, K):
    vmx, torch = gpu
    from vllm_rust_amd._lib import check, lib
    M = full + tail
    lib._Z18vmx_int4_gemm_y_okiii.restype = C.c_bool
    assert lib._Z18vmx_int4_gemm_y_okiii(M, N, K) == (tail > 16)   # one slice and no pass of its own for the tail
    w, x = _Weights(vmx, torch, K, N, tail + K, paired=True), _rows(torch, M, K, tail)
    out = torch.full((M + 1, N // 2), float("nan"), device="cuda", dtype=torch.bfloat16)
    check(lib._Z17vmx_int4_gemm_gluPKvPKtPtiiiiP12ihipStream_t(_p(w.packed), _p(x), _p(out), M, N, K, GROUP, None))
    torch.cuda.synchronize()
    ref, bound = _glu(torch, *w.product(x))
    assert bool(((out[:-1].double() - ref).abs() <= bound).all())
    assert bool(out[-1].isnan().all())


@pytest.mark.parametrize("M", [5, 11, 16])
@pytest.mark.parametrize("K", [2048, 4096, 6144, 8192, 12288])
@pytest.mark.parametrize("N", [16, 1040])
def test_residual(gpu, M, K, N):
    """h = bf16(h + bf16(x W)), the sums of squares of its 16-column tiles and bf16(h gain): every depth that has a form."""
    vmx, torch = gpu
    from vllm_rust_amd._lib import check, lib
    w, x = _Weights(vmx, torch, K, N, M + K + N), _rows(torch, M, K, M)
    g = torch.Generator(device="cuda").manual_seed(K)
    before = torch.randn((M, N), device="cuda", generator=g).to(torch.bfloat16)
    gain = (1 + 0.1 * torch.randn(N, device="cuda", generator=g)).to(torch.bfloat16)
    h, hg = (torch.full((M + 1, N), float("nan"), device="cuda", dtype=torch.bfloat16) for _ in range(2))
    h[:M] = before
    ssq = torch.full((M + 1, N // 16), float("nan"), device="cuda")
    check(lib._Z19vmx_int4_ring_residPKvPKtPtS3_S2_PfiiiiP12ihipStream_t(_p(w.packed), _p(x), _p(h), _p(hg), _p(gain), _p(ssq), M, N, K, GROUP, None))
    torch.cuda.synchronize()
    y, err = w.product(x)
    err = err + 2.0 ** -8 * (y.abs() + err)   # eight significant bits: rounding to bf16 moves a value by at most 2^-8 of it
    ref = before.double() + y
    assert bool(((h[:M].double() - ref).abs() <= err + 2.0 ** -8 * (ref.abs() + err)).all())
    assert torch.equal(hg[:M], (h[:M].float() * gain.float()).to(torch.bfloat16))
    squares = h[:M].double().square().reshape(M, N // 16, 16).sum(2)
    assert bool(((ssq[:M].double() - squares).abs() <= 20 * 2.0 ** -24 * squares).all())
    assert bool(h[M].isnan().all()) and bool(hg[M].isnan().all()) and bool(ssq[M].isnan().all())


@pytest.mark.parametrize("M", [5, 11, 16])
@pytest.mark.parametrize("K,N,glu", [(2048, 6144, False), (4096, 6144, False), (8192, 10240, False), (2048, 12288, True), (4096, 24576, True)])
def test_behind_the_residual(gpu, M, K, N, glu):
    """The linear of rms_norm(h) from h's rows times the gains and the sums of squares; the factor of a row is right to a few 2^-24."""
    vmx, torch = gpu
    from vllm_rust_amd._lib import check, lib
    slices = lib._Z25vmx_int4_ring_norm_splitsiiii(M, N, K, int(glu))
    assert slices == (1 if glu else 2)
    w, hg = _Weights(vmx, torch, K, N, M + K + N, paired=glu), _rows(torch, M, K, M)
    eps = 1e-6
    ssq = hg.float().square().reshape(M, K // 16, 16).sum(2).contiguous()   # as of gains of one
    factor = torch.rsqrt(ssq.double().sum(1, keepdim=True) / K + eps)
    ref, err = w.product(hg)
    ref, err = ref * factor, err * factor
    err = err + 2.0 ** -18 * ref.abs()
    call = lib._Z18vmx_int4_ring_normPKvPKtPKffPfPtiiiiP12ihipStream_t
    if glu:
        out = torch.full((M + 1, N // 2), float("nan"), device="cuda", dtype=torch.bfloat16)
        check(call(_p(w.packed), _p(hg), _p(ssq), C.c_float(eps), None, _p(out), M, N, K, GROUP, None))
        torch.cuda.synchronize()
        ref, err = _glu(torch, ref, err)
        got = out[:-1].double()
    else:
        out = torch.full((slices * M + 1, N), float("nan"), device="cuda")
        check(call(_p(w.packed), _p(hg), _p(ssq), C.c_float(eps), _p(out), None, M, N, K, GROUP, None))
        torch.cuda.synchronize()
        got = out[:-1].double().reshape(slices, M, N).sum(0)
    assert bool(((got - ref).abs() <= err).all())
    assert bool(out[-1].isnan().all())
