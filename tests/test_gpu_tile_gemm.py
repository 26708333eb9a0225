"""Prompt-sized products on the shared matrix-core tiles (csrc/tile_gemm.h) at the edges of their tiles, stages and shape choices,
and the decode-row linears at the edges of theirs."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    import torch
    import vllm_rust_amd as vmx
    assert torch.cuda.is_available()
    vmx.init(0)
    return vmx, torch


# rows and columns one below, at and one above the 64- and 128-wide tiles; one, two, three and many 64-deep stages; the last three take
# the 128 x 128 tiles (a workgroup for every compute unit), 40 x 20000 the 64 x 64 tiles in two stages
@pytest.mark.parametrize("M,N,K", [(17, 1, 64), (63, 64, 128), (64, 65, 192), (65, 63, 64), (127, 129, 256), (129, 200, 2048), (40, 20000, 128),
                                   (129, 16385, 64), (300, 12289, 192), (257, 16384, 320)])
@pytest.mark.parametrize("out", ["f32", "bf16"])
def test_bf16_linear_tiles(gpu, M, N, K, out):
    """Against float64 on the same bf16 operands: an f32 sum of K exact products is off by at most (K + 8) 2^-24 sum |x w| (the matrix
    core adds in f32, in blocks), a bf16 result by half an ulp more."""
    vmx, torch = gpu
    from vllm_rust_amd._lib import check, lib
    g = torch.Generator(device="cuda").manual_seed(M * 131 + N + K)
    x = torch.randn((M, K), device="cuda", generator=g).to(torch.bfloat16)
    w = torch.randn((N, K), device="cuda", generator=g).to(torch.bfloat16)
    guard = torch.full((M + 2, N), 7.0, device="cuda", dtype=torch.float32 if out == "f32" else torch.bfloat16)
    y = guard[1:M + 1]
    check(lib.vmx_linear_bf16w(y.data_ptr(), 0 if out == "f32" else 1, x.data_ptr(), 1, w.data_ptr(), M, N, K, 0, None))
    torch.cuda.synchronize()
    ref = x.double() @ w.double().T
    bound = (K + 8) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)
    if out == "bf16":
        bound = bound + 2.0 ** -8 * ref.abs()
    assert bool(((y.double() - ref).abs() <= bound).all())
    assert bool((guard[0] == 7.0).all()) and bool((guard[M + 1] == 7.0).all())


_LINEAR_SHAPES = {"64 x 64": (2, 2, 1, 1, 5), "64 x 128": (2, 2, 1, 2, 3), "128 x 128, two a unit": (2, 2, 2, 2, 2), "128 x 128, one a unit": (2, 4, 2, 1, 4), "192 x 128": (2, 2, 3, 2, 3),
                  "256 x 128": (4, 2, 2, 2, 3)}


# every tile shape of 256 compute units; rows and columns past the last whole tile, and whole tiles, whose bf16 results go out in pairs
@pytest.mark.parametrize("M,N,K,shape", [(100, 300, 64, "64 x 64"), (64, 64, 320, "64 x 64"), (129, 12801, 128, "64 x 128"), (128, 12800, 128, "64 x 128"),
                                         (513, 11001, 320, "128 x 128, two a unit"), (1023, 2049, 2048, "128 x 128, one a unit"), (383, 12281, 1024, "192 x 128"),
                                         (384, 12288, 1024, "192 x 128"), (511, 12281, 2048, "256 x 128"), (512, 12288, 2048, "256 x 128")])
@pytest.mark.parametrize("out", ["f32", "bf16"])
def test_bf16_linear_tile_shapes(gpu, M, N, K, shape, out):
    """As test_bf16_linear_tiles, the same bounds; and the shape that the call launches is the one named."""
    vmx, torch = gpu
    from tests.helpers import launched_kernels
    from vllm_rust_amd._lib import check, lib
    test_bf16_linear_tiles(gpu, M, N, K, out)
    x, w = (torch.zeros((n, K), dtype=torch.bfloat16, device="cuda") for n in (M, N))
    y = torch.empty((M, N), device="cuda", dtype=torch.float32 if out == "f32" else torch.bfloat16)
    (name,) = [k for k, *_ in launched_kernels(torch, lambda: check(lib.vmx_linear_bf16w(
        y.data_ptr(), 0 if out == "f32" else 1, x.data_ptr(), 1, w.data_ptr(), M, N, K, 0, torch.cuda.current_stream().cuda_stream)))]
    assert "linear_tile_kernel" in name and "TgShapeI%sLb0E" % "".join("Li%dE" % v for v in _LINEAR_SHAPES[shape]) in name, name


# f32 rows (64 x 128 tiles in two stages): rows and columns one below, at and one above a tile, one to many stages
@pytest.mark.parametrize("M,N,K", [(17, 1, 64), (63, 127, 128), (64, 128, 192), (65, 129, 64), (129, 130, 2048), (300, 1000, 320)])
@pytest.mark.parametrize("out", ["f32", "bf16"])
def test_f32_row_linear_tiles(gpu, M, N, K, out):
    """As test_bf16_linear_tiles, on the rows rounded to bf16 (which the kernel does): the same bounds."""
    vmx, torch = gpu
    from vllm_rust_amd._lib import check, lib
    g = torch.Generator(device="cuda").manual_seed(M * 131 + N + K)
    x = torch.randn((M, K), device="cuda", generator=g)
    w = torch.randn((N, K), device="cuda", generator=g).to(torch.bfloat16)
    guard = torch.full((M + 2, N), 7.0, device="cuda", dtype=torch.float32 if out == "f32" else torch.bfloat16)
    y = guard[1:M + 1]
    check(lib.vmx_linear_bf16w(y.data_ptr(), 0 if out == "f32" else 1, x.data_ptr(), 0, w.data_ptr(), M, N, K, 0, None))
    torch.cuda.synchronize()
    xr = x.to(torch.bfloat16).double()
    ref = xr @ w.double().T
    bound = (K + 8) * 2.0 ** -24 * (xr.abs() @ w.double().abs().T)
    if out == "bf16":
        bound = bound + 2.0 ** -8 * ref.abs()
    assert bool(((y.double() - ref).abs() <= bound).all())
    assert bool((guard[0] == 7.0).all()) and bool((guard[M + 1] == 7.0).all())


class _Linear(C.Structure):   # VmxLinear
    _fields_ = [("A", C.c_void_p), ("a_f32", C.c_int), ("lda", C.c_int64), ("W", C.c_void_p), ("w_sn", C.c_int64), ("w_sk", C.c_int64), ("C", C.c_void_p), ("c_f32", C.c_int),
                ("ldc", C.c_int64), ("M", C.c_int), ("N", C.c_int), ("K", C.c_int), ("batch", C.c_int), ("a_bs", C.c_int64), ("w_bs", C.c_int64), ("c_bs", C.c_int64),
                ("aux_bs", C.c_int64), ("row_ids", C.c_void_p), ("row_div", C.c_int), ("row_limit", C.c_int), ("block_expert", C.c_void_p), ("expert_stride", C.c_int64),
                ("block_rows", C.c_int), ("total_rows", C.c_void_p), ("bias", C.c_void_p), ("bias_bs", C.c_int64), ("epilogue", C.c_int), ("aux", C.c_void_p), ("ldaux", C.c_int64),
                ("aux_sn", C.c_int), ("silu_begin", C.c_int), ("silu_end", C.c_int), ("out_scale", C.c_float), ("exact", C.c_int)]


def _launch_linear(torch, shape, **kw):
    """One vmx_linear_launch, which must run as a linear_tile_kernel of that shape (None: of any)."""
    from tests.helpers import launched_kernels
    from vllm_rust_amd._lib import check, lib
    given = dict(w_sk=1, batch=1, row_div=1, aux_sn=1, out_scale=1.0) | kw
    p = _Linear(**{k: v.data_ptr() if hasattr(v, "data_ptr") else v for k, v in given.items()})
    run = lambda: check(lib.vmx_linear_launch(C.byref(p), C.c_void_p(torch.cuda.current_stream().cuda_stream)))   # noqa: E731
    (name,) = [k for k, *_ in launched_kernels(torch, run)]
    assert "linear_tile_kernel" in name and (shape is None or "TgShapeI%sE" % shape in name), name
    run()
    torch.cuda.synchronize()


_MUL_SIGMOID = 3   # VMX_EP_MUL_SIGMOID
_F32_ROWS = "Li2ELi2ELi1ELi2ELi2ELb1E"


# heads side by side in a wider row, as latent attention has them; whole 64 x 128 tiles and not; results in rows of an odd length (no pairs); the gate of a row and
# head, or of every output
@pytest.mark.parametrize("M,N,K,pad", [(70, 130, 128, 8), (128, 128, 64, 0), (128, 128, 64, 1), (17, 512, 192, 8)])
@pytest.mark.parametrize("gate", [None, "head", "element"])
@pytest.mark.parametrize("out", ["f32", "bf16"])
@pytest.mark.parametrize("rows", ["f32", "bf16"])
def test_batched_linear_tiles(gpu, M, N, K, pad, gate, out, rows):
    """Against float64 on the rows rounded to bf16.  An f32 sum of K exact products is off by at most (K + 8) 2^-24 sum |x w|; a sigmoid and the
    multiplication by it by a few units of 2^-24 of the result; a bf16 result by half an ulp more.  Nothing is written between the rows."""
    vmx, torch = gpu
    B = 3
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    lda, ldc = B * (K + 64) + 8, B * N + pad
    x = torch.randn((M, lda), device="cuda", generator=g)
    x = x if rows == "f32" else x.to(torch.bfloat16)
    w = torch.randn((B, N, K), device="cuda", generator=g).to(torch.bfloat16)
    aux = torch.randn((M, B * N), device="cuda", generator=g) * 2
    y = torch.full((M, ldc), 7.0, device="cuda", dtype=torch.float32 if out == "f32" else torch.bfloat16)
    gates = {} if gate is None else dict(epilogue=_MUL_SIGMOID, aux=aux, ldaux=B * N, aux_sn=0 if gate == "head" else 1, aux_bs=1 if gate == "head" else N)
    _launch_linear(torch, _F32_ROWS if rows == "f32" else None, A=x, a_f32=rows == "f32", lda=lda, a_bs=K + 64, W=w, w_sn=K, w_bs=N * K, C=y, c_f32=out == "f32", ldc=ldc, c_bs=N,
                   M=M, N=N, K=K, batch=B, **gates)
    for b in range(B):
        xr = x[:, b * (K + 64):b * (K + 64) + K].to(torch.bfloat16).double()
        ref, size = xr @ w[b].double().T, xr.abs() @ w[b].double().abs().T
        if gate:
            f = torch.sigmoid(aux[:, b:b + 1] if gate == "head" else aux[:, b * N:(b + 1) * N]).double()
            ref, size = ref * f, size * f
        bound = (K + 8 + 16) * 2.0 ** -24 * size + (2.0 ** -8 * ref.abs() if out == "bf16" else 0.0)
        assert bool(((y[:, b * N:(b + 1) * N].double() - ref).abs() <= bound).all()), b
    assert bool((y[:, B * N:] == 7.0).all())


# gathered rows, two outputs a source row, with ids that are padding (negative, past the limit); and the same in 64-row blocks of three experts, of which the last
# lies past the count of rows
@pytest.mark.parametrize("experts", [False, True])
@pytest.mark.parametrize("N,K", [(130, 128), (256, 64)])
@pytest.mark.parametrize("rows", ["f32", "bf16"])
def test_gathered_linear_tiles(gpu, experts, N, K, rows):
    """Against float64 as above; rows of padding and of blocks past the count stay as they were."""
    vmx, torch = gpu
    M, T = 256, 90
    g = torch.Generator(device="cuda").manual_seed(N + K)
    x = torch.randn((T, K + 8), device="cuda", generator=g)
    x = x if rows == "f32" else x.to(torch.bfloat16)
    w = torch.randn((3, N, K), device="cuda", generator=g).to(torch.bfloat16)
    ids = torch.randint(0, 2 * T, (M,), device="cuda", generator=g, dtype=torch.int32)
    ids[5::16] = -1
    ids[70] = 2 * T
    y = torch.full((M, N), 7.0, device="cuda")
    of = torch.tensor([2, 0, 0, 1], dtype=torch.int32, device="cuda")
    total = torch.tensor([192], dtype=torch.int32, device="cuda")
    more = dict(block_expert=of, expert_stride=N * K, block_rows=64, total_rows=total) if experts else {}
    _launch_linear(torch, _F32_ROWS if rows == "f32" else None, A=x, a_f32=rows == "f32", lda=K + 8, W=w, w_sn=K, C=y, c_f32=1, ldc=N, M=M, N=N, K=K, row_ids=ids, row_div=2, row_limit=2 * T,
                   **more)
    live = (ids >= 0) & (ids < 2 * T)
    if experts:
        live[192:] = False
    xr = x[(ids.long().clamp(0, 2 * T - 1) // 2), :K].to(torch.bfloat16).double()
    pick = (of.long() if experts else torch.zeros(4, dtype=torch.long, device="cuda")).repeat_interleave(64)
    ref = torch.stack([xr[m] @ w[pick[m]].double().T for m in range(M)])
    size = torch.stack([xr[m].abs() @ w[pick[m]].double().abs().T for m in range(M)])
    assert bool(((y.double() - ref).abs() <= (K + 8) * 2.0 ** -24 * size)[live].all())
    assert bool((y[~live] == 7.0).all())


# rows around the 64- and 128-row tiles; columns around the 128-wide ones; K of one super-block, an odd number of them, and enough with
# few tiles that the sums are cut into slices ((2048, 8192) gives the workspace room for them, (64, 256) does not)
@pytest.mark.parametrize("M", [17, 64, 65, 129, 300])
@pytest.mark.parametrize("ggml_type,N,K", [(18, 64, 256), (22, 129, 768), (21, 2048, 8192), (17, 2052, 7936)])
def test_iq_prompt_linear_tiles(gpu, M, ggml_type, N, K):
    """Against float64 on the dequantised weight: products of an fp16 activation and an integer are exact, 256 of them are added in
    f32 (error (256 + 8) 2^-24 of the sum of magnitudes), scaled and added up in f32 again."""
    vmx, torch = gpu
    from tests.helpers import random_iq_blocks
    ts = vmx.iq_type_size(ggml_type)
    raw = torch.from_numpy(np.ascontiguousarray(random_iq_blocks(np.random.default_rng(N + K), ts, N * K // 256))).reshape(-1).cuda()
    g = torch.Generator(device="cuda").manual_seed(M + N)
    x = torch.randn((M, K), device="cuda", generator=g).to(torch.bfloat16)
    y = vmx.iq_gemm(ggml_type, raw, x, N)
    torch.cuda.synchronize()
    w = vmx.iq_dequantize(ggml_type, raw, N * K // 256).reshape(N, K).double()
    ref = x.double() @ w.T
    bound = (264 + K // 256 + 8) * 2.0 ** -24 * (x.double().abs() @ w.abs().T)
    assert bool(((y.double() - ref).abs() <= bound).all())


# columns that are no multiple of four; a workspace that holds every slice, or the 4 N K bytes that the product must have and what slices fit them
@pytest.mark.parametrize("offset,M,N,room", [(0, 33, 512, 64 << 20), (1, 33, 512, 64 << 20), (2, 33, 512, 64 << 20), (3, 33, 512, 64 << 20), (0, 65, 131, 64 << 20),
                                             (1, 300, 130, 64 << 20), (0, 200, 512, 0), (0, 700, 131, 0), (3, 4000, 132, 0)])
def test_iq_prompt_linear_slices(gpu, offset, M, N, room):
    """The output of a product whose sums come in slices may start at any f32 of a larger tensor: the same values, nothing written beside it or
    behind the workspace."""
    vmx, torch = gpu
    from tests.helpers import random_iq_blocks
    from vllm_rust_amd._lib import check, lib
    K, t = 8192, 18
    raw = torch.from_numpy(np.ascontiguousarray(random_iq_blocks(np.random.default_rng(1), vmx.iq_type_size(t), N * K // 256))).reshape(-1).cuda()
    x = torch.randn((M, K), device="cuda", generator=torch.Generator(device="cuda").manual_seed(1)).to(torch.bfloat16)
    need = 4 * N * K + room
    assert lib.vmx_iq_gemm_workspace_bytes(N, K) >= 4 * N * K
    ws = torch.full((need + 64,), 7, dtype=torch.uint8, device="cuda")
    held = torch.full((M * N + 8,), 7.0, device="cuda")
    y = held[offset:offset + M * N]
    check(lib.vmx_iq_gemm_f32(t, raw.data_ptr(), x.data_ptr(), y.data_ptr(), M, N, K, ws.data_ptr(), need, None))
    torch.cuda.synchronize()
    w = vmx.iq_dequantize(t, raw, N * K // 256).reshape(N, K).double()
    bound = (264 + K // 256 + 8) * 2.0 ** -24 * (x.double().abs() @ w.abs().T)
    assert bool(((y.view(M, N).double() - x.double() @ w.T).abs() <= bound).all())
    assert bool((held[:offset] == 7.0).all()) and bool((held[offset + M * N:] == 7.0).all()) and bool((ws[need:] == 7).all())


# fewer than eight super-blocks: 64 x 64 tiles around whose edges rows and columns lie, in no slices, in as many as there are super-blocks, in slices of unequal
# length (seven super-blocks in four), and one super-block more and a tile row more than that form takes (1100 x 3900: 1116 tiles)
@pytest.mark.parametrize("M,N,K,sliced", [(17, 512, 1024, True), (65, 130, 512, False), (63, 65, 768, True), (129, 4100, 1024, False), (300, 1000, 1792, True),
                                          (64, 2048, 1024, True), (65, 4096, 1792, True), (1200, 512, 1024, False), (1100, 3900, 512, False), (65, 512, 2048, True)])
def test_iq_prompt_linear_short(gpu, M, N, K, sliced):
    """Against float64 as above.  A short product is a chain of stages, and where its output is small the chain is cut although it is short: the
    launch that adds the slices is one kernel more (weights, rows, product, sum), counted in a captured graph."""
    import ctypes as C
    vmx, torch = gpu
    from tests.helpers import random_iq_blocks
    from vllm_rust_amd._lib import check, lib
    t = 22
    raw = torch.from_numpy(np.ascontiguousarray(random_iq_blocks(np.random.default_rng(N + K), vmx.iq_type_size(t), N * K // 256))).reshape(-1).cuda()
    x = torch.randn((M, K), device="cuda", generator=torch.Generator(device="cuda").manual_seed(M + N)).to(torch.bfloat16)
    need = 4 * N * K + (32 << 20)
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    held = torch.full((M + 2, N), 7.0, device="cuda")
    y = held[1:M + 1]
    run = lambda: check(lib.vmx_iq_gemm_f32(t, raw.data_ptr(), x.data_ptr(), y.data_ptr(), M, N, K, ws.data_ptr(), need,   # noqa: E731
                                            torch.cuda.current_stream().cuda_stream))
    run()
    torch.cuda.synchronize()
    w = vmx.iq_dequantize(t, raw, N * K // 256).reshape(N, K).double()
    bound = (264 + K // 256 + 8) * 2.0 ** -24 * (x.double().abs() @ w.abs().T)
    assert bool(((y.double() - x.double() @ w.T).abs() <= bound).all())
    assert bool((held[0] == 7.0).all()) and bool((held[M + 1] == 7.0).all())
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph):
        run()
    n = C.c_size_t(0)
    assert C.CDLL("libamdhip64.so").hipGraphGetNodes(C.c_void_p(graph.raw_cuda_graph()), None, C.byref(n)) == 0
    assert n.value == (4 if sliced else 3)


# raw blocks decoded inside the product (tiles of 64, 128 and 192 rows; every height by name in test_iq_prompt_tile_heights): an odd number of super-blocks (block starts alternate between
# the halves of a dword along a row and from row to row) and an even one; columns past a tile; a weight that starts in the middle of a dword; room for
# slices of k and none
@pytest.mark.parametrize("M", [17, 64, 65, 129, 192, 256, 333])
@pytest.mark.parametrize("ggml_type,N,K,start,room", [(18, 2052, 4352, 2, 64 << 20), (21, 2177, 4096, 0, 64 << 20), (22, 1100, 7936, 2, 0), (17, 8193, 1024, 0, 64 << 20)])
def test_iq_prompt_decoded(gpu, M, ggml_type, N, K, start, room):
    """Against float64 on the dequantised weight, bounds as above; nothing written beside the result or behind the workspace."""
    vmx, torch = gpu
    from tests.helpers import random_iq_blocks
    from vllm_rust_amd._lib import check, lib
    ts = vmx.iq_type_size(ggml_type)
    raw = torch.from_numpy(np.ascontiguousarray(random_iq_blocks(np.random.default_rng(N + K), ts, N * K // 256))).reshape(-1)
    held = torch.zeros(start + raw.numel(), dtype=torch.uint8, device="cuda")
    held[start:] = raw.cuda()
    x = torch.randn((M, K), device="cuda", generator=torch.Generator(device="cuda").manual_seed(M + N)).to(torch.bfloat16)
    need = 4 * N * K + room
    ws = torch.full((need + 64,), 7, dtype=torch.uint8, device="cuda")
    guard = torch.full((M + 2, N), 7.0, device="cuda")
    y = guard[1:M + 1]
    check(lib.vmx_iq_gemm_f32(ggml_type, held.data_ptr() + start, x.data_ptr(), y.data_ptr(), M, N, K, ws.data_ptr(), need, None))
    torch.cuda.synchronize()
    w = vmx.iq_dequantize(ggml_type, raw.cuda(), N * K // 256).reshape(N, K).double()
    bound = (264 + K // 256 + 8) * 2.0 ** -24 * (x.double().abs() @ w.abs().T)
    assert bool(((y.double() - x.double() @ w.T).abs() <= bound).all())
    assert bool((guard[0] == 7.0).all()) and bool((guard[M + 1] == 7.0).all()) and bool((ws[need:] == 7).all())


# rows beyond what the least workspace holds in the integer form: the two-term bf16 split, whose activations stay bf16
@pytest.mark.parametrize("size", [1.0, 3e5, 2.0 ** -40])
def test_iq_gemm_rows_outside_fp16(gpu, size):
    """Activations above fp16's largest value and below its smallest.  A weight's two bf16 halves are off by at most 2^-17 of it (2^-9 of a remainder of
    2^-8); the f32 sums of two products a weight add (2 K + 8) 2^-24 of the sum of magnitudes."""
    vmx, torch = gpu
    from tests.helpers import random_iq_blocks
    from vllm_rust_amd._lib import check, lib
    M, N, K, t = 1500, 1024, 8192, 18
    raw = torch.from_numpy(np.ascontiguousarray(random_iq_blocks(np.random.default_rng(3), vmx.iq_type_size(t), N * K // 256))).reshape(-1).cuda()
    x = (torch.randn((M, K), device="cuda", generator=torch.Generator(device="cuda").manual_seed(3)) * size).to(torch.bfloat16)
    ws = torch.empty(4 * N * K, dtype=torch.uint8, device="cuda")
    y = torch.full((M, N), float("nan"), device="cuda")
    check(lib.vmx_iq_gemm_f32(t, raw.data_ptr(), x.data_ptr(), y.data_ptr(), M, N, K, ws.data_ptr(), ws.numel(), None))
    torch.cuda.synchronize()
    w = vmx.iq_dequantize(t, raw, N * K // 256).reshape(N, K).double()
    bound = (2.0 ** -17 + (2 * K + 8) * 2.0 ** -24) * (x.double().abs() @ w.abs().T)
    assert bool(((y.double() - x.double() @ w.T).abs() <= bound).all())


# decoded inside the product, or dequantised first where that leaves less of the last round of tiles empty
@pytest.mark.parametrize("M,N,K,inside", [(256, 30720, 3840, True), (2048, 30720, 3840, True), (1000, 13862, 3328, True), (2825, 13862, 3328, False),
                                          (2825, 8192, 3840, False), (8192, 8192, 3840, True), (1000, 4096, 4096, False), (2047, 12288, 1024, False), (333, 3840, 15360, True)])
def test_iq_prompt_or_dequantised(gpu, M, N, K, inside):
    """Which of the two products a call takes, on 256 compute units."""
    vmx, torch = gpu
    from tests.helpers import launched_kernels
    from vllm_rust_amd._lib import check, lib
    raw = torch.zeros(vmx.iq_type_size(18) * N * K // 256, dtype=torch.uint8, device="cuda")
    x, y = torch.zeros((M, K), dtype=torch.bfloat16, device="cuda"), torch.empty((M, N), device="cuda")
    ws = torch.empty(4 * N * K + 4 * M * K, dtype=torch.uint8, device="cuda")
    names = [name for name, *_ in launched_kernels(torch, lambda: check(lib.vmx_iq_gemm_f32(
        18, raw.data_ptr(), x.data_ptr(), y.data_ptr(), M, N, K, ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream)))]
    assert any("iq_prompt_kernel" in n for n in names) == inside


def test_iq_prompt_lds_of_all_types(gpu):
    """The types share a kernel and differ in the LDS they take.  What a launch sets the kernel's limit to is the same for all of them, or
    a thread with one type could lower it between another's setting and its launch."""
    vmx, torch = gpu
    from tests.helpers import launched_kernels
    from vllm_rust_amd._lib import check, lib
    M, N, K = 256, 8192, 1024
    x, y = torch.zeros((M, K), dtype=torch.bfloat16, device="cuda"), torch.empty((M, N), device="cuda")
    ws = torch.empty(8 * N * K, dtype=torch.uint8, device="cuda")
    seen = {}
    for t in (22, 18, 21, 17):
        raw = torch.zeros(vmx.iq_type_size(t) * N * K // 256, dtype=torch.uint8, device="cuda")
        run = lambda: check(lib.vmx_iq_gemm_f32(t, raw.data_ptr(), x.data_ptr(), y.data_ptr(), M, N, K, ws.data_ptr(), ws.numel(),   # noqa: E731, B023
                                                torch.cuda.current_stream().cuda_stream))
        run()
        torch.cuda.synchronize()
        for name, _, lds, most in launched_kernels(torch, run):
            if "iq_prompt_kernel" in name:
                seen.setdefault(name, []).append((lds, most))
    (of_types,) = seen.values()
    assert len(of_types) == 4 and len({lds for lds, _ in of_types}) > 1
    assert len({most for _, most in of_types}) == 1 and of_types[0][1] >= max(lds for lds, _ in of_types)


class _Seg(C.Structure):
    _fields_ = [("w", C.c_void_p), ("ggml_type", C.c_int), ("n_out", C.c_int), ("y_off", C.c_int)]


# three projections of three types as one product, none of whose widths is whole tiles; in slices and in none
@pytest.mark.parametrize("M", [33, 130, 300])
@pytest.mark.parametrize("K,room", [(1280, 0), (4096, 64 << 20)])
def test_iq_prompt_projections(gpu, M, K, room):
    """Against float64 as above; the columns beside the projections' stay as they were."""
    vmx, torch = gpu
    from tests.helpers import random_iq_blocks
    from vllm_rust_amd._lib import check, lib
    types, widths = (18, 22, 21), (300, 129, 64)
    raws = [torch.from_numpy(np.ascontiguousarray(random_iq_blocks(np.random.default_rng(t + K), vmx.iq_type_size(t), n * K // 256))).reshape(-1).cuda()
            for t, n in zip(types, widths)]
    x = torch.randn((M, K), device="cuda", generator=torch.Generator(device="cuda").manual_seed(M + K)).to(torch.float16)
    N, off = sum(widths), [0, widths[0], widths[0] + widths[1]]
    segs = (_Seg * 3)(*[_Seg(r.data_ptr(), t, n, o) for r, t, n, o in zip(raws, types, widths, off)])
    y = torch.full((M, N + 3), 7.0, device="cuda")
    part = torch.empty(max(room, 1), dtype=torch.uint8, device="cuda")
    check(lib.vmx_iq_prompt_f32(segs, 3, C.c_void_p(x.data_ptr()), C.c_void_p(y.data_ptr()), M, K, C.c_int64(N + 3), C.c_void_p(part.data_ptr()), C.c_size_t(room), None))
    torch.cuda.synchronize()
    w = torch.cat([vmx.iq_dequantize(t, r, n * K // 256).reshape(n, K).double() for r, t, n in zip(raws, types, widths)])
    bound = (264 + K // 256 + 8) * 2.0 ** -24 * (x.double().abs() @ w.abs().T)
    assert bool(((y[:, :N].double() - x.double() @ w.T).abs() <= bound).all())
    assert bool((y[:, N:] == 7.0).all())


# gate columns below, at and past the 64 that a tile takes (tiles of 64 rows: too few columns for others)
@pytest.mark.parametrize("M", [17, 65, 129, 192, 256])
@pytest.mark.parametrize("ggml_type,inter,K", [(18, 40, 256), (21, 64, 512), (22, 200, 1280), (17, 130, 768)])
def test_iq_prompt_geglu(gpu, M, ggml_type, inter, K):
    """act = bf16(bf16(gelu(gate)) * up), gate and up rounded to bf16, against float64 on the dequantised weights.  The f32 sums may fall on the
    other side of a bf16 rounding: one step (2^-8 relative) of gate and of up, and one of each product behind."""
    err, by_gate, ref = _geglu(gpu, M, ggml_type, inter, K, 64)
    assert bool((err <= 2.0 ** -8 * (by_gate + 3 * ref) + 2.0 ** -20).all())


def _geglu(gpu, M, ggml_type, inter, K, height):
    """|act - exact| of a product that must take tiles of that height, |d exact / d gate * gate| and |exact|."""
    vmx, torch = gpu
    from tests.helpers import random_iq_blocks
    from vllm_rust_amd._lib import check, lib
    raw = [torch.from_numpy(np.ascontiguousarray(random_iq_blocks(np.random.default_rng(s + K), vmx.iq_type_size(ggml_type), inter * K // 256))).reshape(-1).cuda()
           for s in (1, 2)]
    w = [vmx.iq_dequantize(ggml_type, r, inter * K // 256).reshape(inter, K).double() for r in raw]
    scale = 1.0 / float((w[0] ** 2).mean().sqrt() * K ** 0.5)           # sums of order 1
    x = (torch.randn((M, K), device="cuda", generator=torch.Generator(device="cuda").manual_seed(M + K)) * scale).to(torch.float16)
    guard = torch.full((M + 2, inter), 7.0, dtype=torch.float16, device="cuda")
    act = guard[1:M + 1]
    gate, up = [_Seg(r.data_ptr(), ggml_type, inter, 0) for r in raw]
    run = lambda: check(lib.vmx_iq_prompt_geglu(C.byref(gate), C.byref(up), C.c_void_p(x.data_ptr()), C.c_void_p(act.data_ptr()), M, K,   # noqa: E731
                                                C.c_void_p(torch.cuda.current_stream().cuda_stream)))
    assert _iq_tile(torch, run) == (height, True)
    run()
    torch.cuda.synchronize()
    gate, up = [(x.double() @ m.T).to(torch.bfloat16).double() for m in w]
    cdf = 0.5 * (1 + torch.erf(gate / 2 ** 0.5))
    slope = cdf + gate * torch.exp(-gate * gate / 2) / (2 * np.pi) ** 0.5
    ref = gate * cdf * up
    assert bool((guard[0] == 7.0).all()) and bool((guard[M + 1] == 7.0).all())
    return (act.double() - ref).abs(), (slope * gate * up).abs(), ref.abs()


_IQ_SHAPES = {64: (2, 4, 1, 1), 128: (4, 2, 1, 2), 192: (2, 4, 3, 1), 256: (4, 2, 2, 2)}


def _iq_tile(torch, run):
    """Rows of the tile of the one iq_prompt_kernel that run() launches, and whether its epilogue is GeGLU."""
    from tests.helpers import launched_kernels
    (name,) = [k for k, *_ in launched_kernels(torch, run) if "iq_prompt_kernel" in k]
    (rows,) = [r for r, s in _IQ_SHAPES.items() if "IqpShapeI%sEE" % "".join("Li%dE" % v for v in s) in name]
    return rows, "EELb1EE" in name


# every height with columns for more than half of 256 units (129 .. 131 tiles), its last rows missing or not, and with its results in slices
@pytest.mark.parametrize("ggml_type", [17, 18, 21, 22])
@pytest.mark.parametrize("M,N,K,room,height", [(50, 16700, 512, 0, 64), (64, 16640, 512, 0, 64), (127, 16700, 512, 0, 128), (128, 16640, 768, 0, 128), (190, 16700, 512, 0, 192), (192, 16640, 768, 0, 192),
                                               (250, 16700, 512, 0, 256), (256, 16640, 768, 0, 256), (1000, 1060, 8192, 64 << 20, 256), (290, 1060, 8192, 64 << 20, 192)])
def test_iq_prompt_tile_heights(gpu, ggml_type, M, N, K, room, height):
    """Against float64 on the dequantised weight, bounds as in test_iq_prompt_linear_tiles; and the tile is of the height named."""
    vmx, torch = gpu
    from tests.helpers import random_iq_blocks
    from vllm_rust_amd._lib import check, lib
    raw = torch.from_numpy(np.ascontiguousarray(random_iq_blocks(np.random.default_rng(N + K), vmx.iq_type_size(ggml_type), N * K // 256))).reshape(-1).cuda()
    x = torch.randn((M, K), device="cuda", generator=torch.Generator(device="cuda").manual_seed(M + N)).to(torch.float16)
    seg = (_Seg * 1)(_Seg(raw.data_ptr(), ggml_type, N, 0))
    guard = torch.full((M + 2, N), 7.0, device="cuda")
    y = guard[1:M + 1]
    part = torch.empty(max(room, 1), dtype=torch.uint8, device="cuda")
    run = lambda: check(lib.vmx_iq_prompt_f32(seg, 1, C.c_void_p(x.data_ptr()), C.c_void_p(y.data_ptr()), M, K, C.c_int64(N), C.c_void_p(part.data_ptr()),   # noqa: E731
                                              C.c_size_t(room), C.c_void_p(torch.cuda.current_stream().cuda_stream)))
    assert _iq_tile(torch, run) == (height, False)
    run()
    torch.cuda.synchronize()
    w = vmx.iq_dequantize(ggml_type, raw, N * K // 256).reshape(N, K).double()
    bound = (264 + K // 256 + 8) * 2.0 ** -24 * (x.double().abs() @ w.abs().T)
    assert bool(((y.double() - x.double() @ w.T).abs() <= bound).all())
    assert bool((guard[0] == 7.0).all()) and bool((guard[M + 1] == 7.0).all())


# the same with the GeGLU epilogue: 130 tiles of 64 gate and 64 up columns
@pytest.mark.parametrize("ggml_type", [17, 18, 21, 22])
@pytest.mark.parametrize("M,inter,K,height", [(64, 8300, 512, 64), (127, 8300, 512, 128), (128, 8320, 768, 128), (190, 8300, 512, 192), (192, 8320, 768, 192), (250, 8300, 512, 256), (256, 8320, 768, 256)])
def test_iq_prompt_geglu_tile_heights(gpu, ggml_type, M, inter, K, height):
    """As test_iq_prompt_geglu.  Among millions of results some have a gate or an up whose f32 sum falls on the other side of a rounding where the step is
    widest, 2^-7 of the value (8 bits from 1.0 on); gelu and the product behind are rounded to the nearest, 2^-8 each; 2^-6 of all that for their products."""
    err, by_gate, ref = _geglu(gpu, M, ggml_type, inter, K, height)
    assert bool((err <= (1 + 2.0 ** -6) * 2.0 ** -7 * (by_gate + 2 * ref) + 2.0 ** -20).all())


# 256-column blocks; one k-block, odd numbers of them (17; 33 in slices) and groups wider than a
# k-block; rows around the 64-row tiles and past a strip of eight of them
@pytest.mark.parametrize("M", [49, 64, 65, 200, 577])
@pytest.mark.parametrize("N,K,group", [(256, 128, 128), (512, 2176, 128), (2304, 4224, 128), (256, 1536, 512), (256, 16384, 128)])
def test_int4_prompt_tiles(gpu, M, N, K, group):
    """Against float64 on (nibble - zero point) * scale.  The kernel adds x * (16 + nibble) and x * (16 + zero point) apart, in f32: a path through
    the sums has at most four roundings in each of a k-block's eight instructions and two more a k-block, and no term is larger than
    |x| s (31 + 31); half a bf16 ulp for the result on top."""
    vmx, torch = gpu
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x = torch.randn((M, K), device="cuda", generator=g).to(torch.bfloat16)
    words = lambda *s: torch.randint(-2 ** 31, 2 ** 31 - 1, s, dtype=torch.int32, device="cuda", generator=g)   # noqa: E731
    qw, qz = words(K // 8, N), words(K // group, N // 8)
    sc = ((torch.rand((K // group, N), device="cuda", generator=g) + 0.5) * 0.01).to(torch.bfloat16)
    bias = torch.randn(N, device="cuda", generator=g).to(torch.bfloat16)
    y = vmx.int4_gemm(x, vmx.int4_pack(qw, sc, qz, K, N, group), bias, N, K, group)
    torch.cuda.synchronize()
    sh = torch.arange(0, 32, 4, dtype=torch.int32, device="cuda")
    nib = ((qw.unsqueeze(-1) >> sh) & 15).permute(0, 2, 1).reshape(K, N)
    zp = ((qz.unsqueeze(-1) >> sh) & 15).reshape(K // group, N).repeat_interleave(group, 0)
    s = sc.double().repeat_interleave(group, 0)
    ref = x.double() @ ((nib - zp).double() * s) + bias.double()
    bound = 2.0 ** -8 * ref.abs() + (32 + 2 * K // 128 + 8) * 2.0 ** -24 * 62 * (x.double().abs() @ s)
    assert bool(((y.double() - ref).abs() <= bound).all())


# weights equal to their zero points: the product is exactly zero and the output is the rounding of the f32 sums itself
@pytest.mark.parametrize("M,N,K", [(2048, 4096, 12288), (333, 1024, 16512)])
@pytest.mark.parametrize("mean", [0, 1, 5])
def test_int4_prompt_f32_sums(gpu, M, N, K, mean):
    """The zero-point term comes off with every k-block, so no partial sum outgrows a k-block's offset (16 + zero point) s sum x.  A k-block
    rounds eight chained products (sizes 1/8 .. 1: 3.2 in squares), four of its row sum (1.9), its scaling and its zero-point term; eight
    roundings of at most 2^-24 of the largest prefix, of independent sign, bound the rms.  (Taken off once at the end, the sums grow with
    the number of k-blocks: up to fifty times this bound.)"""
    vmx, torch = gpu
    g = torch.Generator(device="cuda").manual_seed(M + N + K + mean)
    x = (torch.randn((M, K), device="cuda", generator=g) + mean).to(torch.bfloat16)
    qz = torch.randint(-2 ** 31, 2 ** 31 - 1, (K // 128, N // 8), dtype=torch.int32, device="cuda", generator=g)
    sc = ((torch.rand((K // 128, N), device="cuda", generator=g) + 0.5) * 0.01).to(torch.bfloat16)
    zp = ((qz.unsqueeze(-1) >> torch.arange(0, 32, 4, dtype=torch.int32, device="cuda")) & 15).reshape(K // 128, N)
    eight = torch.zeros_like(zp)
    for i in range(8):
        eight |= zp << (4 * i)
    qw = eight.repeat_interleave(16, 0).contiguous()   # [K / 8, N]: eight nibbles of one column in a word
    y = vmx.int4_gemm(x, vmx.int4_pack(qw, sc, qz, K, N, 128), None, N, K, 128).double()
    torch.cuda.synchronize()
    prefix = x.double().reshape(M, K // 128, 128).cumsum(2).abs().amax(2)
    size = (prefix ** 2).mean().sqrt() * ((sc.double() * (16 + zp)) ** 2).mean().sqrt()
    assert float((y ** 2).mean().sqrt()) <= float(2.0 ** -24 * (8 * K // 128) ** 0.5 * size)


# decode rows: column groups below one per compute unit (up to 512 deep, beyond with halved k; 4 and 8 waves, a second round), between one and two, and above
@pytest.mark.parametrize("M,N,K", [(1, 40, 72), (16, 30, 384), (9, 2100, 512), (4, 200, 520), (16, 2048, 2040), (5, 1000, 2312), (3, 4100, 520), (16, 4096, 1032), (7, 6000, 2056), (16, 9000, 136)])
@pytest.mark.parametrize("x_f32", [False, True])
def test_bf16_linear_decode_rows(gpu, M, N, K, x_f32):
    """f32 sums of bf16 products in at most K terms: |error| <= K 2^-24 sum |x w|, doubled for the order of the partial sums."""
    vmx, torch = gpu
    from vllm_rust_amd._lib import check, lib
    g = torch.Generator(device="cuda").manual_seed(M * 7 + N + K)
    x = torch.randn((M, K), device="cuda", generator=g).to(torch.bfloat16)
    w = torch.randn((N, K), device="cuda", generator=g).to(torch.bfloat16)
    xin = x.float() if x_f32 else x
    y = torch.full((M, N), float("nan"), device="cuda")
    check(lib.vmx_linear_bf16w(y.data_ptr(), 0, xin.data_ptr(), 0 if x_f32 else 1, w.data_ptr(), M, N, K, 0, None))
    torch.cuda.synchronize()
    exact = x.double() @ w.double().T
    bound = K * 2.0 ** -23 * (x.double().abs() @ w.double().abs().T)
    assert bool(((y.double() - exact).abs() <= bound).all())


def test_int4_prompt_slices(gpu):
    """A prompt of 2048 tokens at once (its tiles fill the chip: one slice of k for o and down) against the same prompt in pieces whose last one,
    which leaves the row compared, is multiplied in slices: 300 rows (three for o and down) and 65 (four and three).  The last hidden row
    agrees to what the order of f32 sums and bf16 rounding behind it allow."""
    from vllm_rust_amd._lib import lib
    from vllm_rust_amd.qwen3 import QuantizedQwen3ForCausalLM, Qwen3Spec
    vmx, torch = gpu
    slices = lambda rows: (lib._Z20vmx_int4_splits_rowsiii(rows, 4096, 4096), lib._Z20vmx_int4_splits_rowsiii(rows, 4096, 12288))   # noqa: E731
    assert slices(2048) == (1, 1) and slices(300) == (3, 3) and slices(65) == (4, 3)
    spec = Qwen3Spec(4096, 2, 32, 8, 128, 12288, 512, tie_word_embeddings=True, max_position=2048, num_blocks=128, max_batch=1, max_seq_len=2048,
                     max_prefill_tokens=2048)
    model = QuantizedQwen3ForCausalLM(spec)
    try:
        model.load_synthetic(seed=3)
        ids = torch.from_numpy(np.random.default_rng(1).integers(0, 512, 2048).astype(np.int32)).cuda()
        bt = torch.randperm(128, device="cuda", generator=torch.Generator(device="cuda").manual_seed(2)).to(torch.int32)
        last = []
        for cuts in ([0, 2048], [0, 1748, 2048], [0, 1700, 1983, 2048]):
            for a, b in zip(cuts, cuts[1:]):
                model.prefill(ids[a:b].contiguous(), a, bt)
            last.append(model.debug_read(0, (b - a, 4096))[-1].double())
        for other in last[1:]:
            assert float((last[0] - other).norm() / last[0].norm()) <= 2e-2
    finally:
        model.close()


# every count of slices (K = 33 k-blocks: slices of unequal length), a chip that is less than, just and more than filled, a remainder of rows
@pytest.mark.parametrize("M,N,K", [(49, 1024, 4224), (65, 4096, 4224), (200, 4096, 4096), (300, 4096, 4096), (333, 4096, 4224), (640, 2048, 4096), (1024, 4096, 4096)])
def test_int4_partial_slices(gpu, M, N, K):
    """The f32 slices that the executor's consumers add, against float64.  A path through the sums has at most four roundings in each of a k-block's
    eight instructions and two more a k-block, and no term is larger than |x| s (16 + nibble + 16 + zero point) <= 62 |x| s.  Nothing is
    written behind the last slice."""
    import ctypes as C
    vmx, torch = gpu
    from vllm_rust_amd._lib import check, lib
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x = torch.randn((M, K), device="cuda", generator=g).to(torch.bfloat16)
    words = lambda *s: torch.randint(-2 ** 31, 2 ** 31 - 1, s, dtype=torch.int32, device="cuda", generator=g)   # noqa: E731
    qw, qz = words(K // 8, N), words(K // 128, N // 8)
    sc = ((torch.rand((K // 128, N), device="cuda", generator=g) + 0.5) * 0.01).to(torch.bfloat16)
    packed = vmx.int4_pack(qw, sc, qz, K, N, 128)
    n = lib._Z20vmx_int4_splits_rowsiii(M, N, K)
    part = torch.full((n * M * N + 64,), float("nan"), device="cuda")
    check(lib._Z21vmx_int4_gemm_partialPKvPKtPfiiiiP12ihipStream_t(C.c_void_p(packed.data_ptr()), C.c_void_p(x.data_ptr()), C.c_void_p(part.data_ptr()), M, N, K,
                                                                128, None))
    torch.cuda.synchronize()
    sh = torch.arange(0, 32, 4, dtype=torch.int32, device="cuda")
    nib = ((qw.unsqueeze(-1) >> sh) & 15).permute(0, 2, 1).reshape(K, N)
    zp = ((qz.unsqueeze(-1) >> sh) & 15).reshape(K // 128, N).repeat_interleave(128, 0)
    s = sc.double().repeat_interleave(128, 0)
    y = part[:n * M * N].view(n, M, N).double().sum(0)
    bound = (32 + 2 * K // 128 + 8) * 2.0 ** -24 * 62 * (x.double().abs() @ s)
    assert bool(((y - x.double() @ ((nib - zp).double() * s)).abs() <= bound).all())
    assert bool(part[n * M * N:].isnan().all())
