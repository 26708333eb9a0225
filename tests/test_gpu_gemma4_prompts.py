"""Gemma-4 prompts past 16 rows: the integer products of merged projections at the edges of their tiles, slices and scale groups, and
groups whose projections do not all have the integer form."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    import torch
    import vllm_rust_amd as vmx
    vmx.init(0)
    return vmx, torch


# rows below, at and past a tile of 64 and past one of 128 (64 x 128 and 128 x 128 tiles); one, two and five scale groups; gate columns below, at and past the
# 64 that a tile takes
@pytest.mark.parametrize("M", [17, 64, 65, 129])
@pytest.mark.parametrize("inter,K", [(40, 256), (64, 512), (200, 1280)])
def test_geglu_tiles(gpu, M, inter, K):
    """act = bf16(bf16(gelu(gate)) * up) with gate and up rounded to bf16, against float64 on the same integers, scales and fp16 rows.  The
    f32 sums may fall on the other side of a bf16 rounding: one step (2^-8 relative) of gate and of up, and one of each product behind."""
    vmx, torch = gpu
    from vllm_rust_amd._lib import check, lib
    g = torch.Generator(device="cuda").manual_seed(M + inter + K)
    N = 2 * inter
    q = torch.randint(-1922, 1923, (N, K), device="cuda", generator=g).to(torch.float16)
    dt = (torch.rand((K // 256, N), device="cuda", generator=g) + 0.5) * (1.0 / (1100 * K ** 0.5))
    x = torch.randn((M, K), device="cuda", generator=g).to(torch.float16)
    ws = torch.cat([q.reshape(-1).view(torch.uint8), dt.reshape(-1).view(torch.uint8)])
    guard = torch.full((M + 2, inter), 7.0, dtype=torch.float16, device="cuda")
    act = guard[1:M + 1]
    check(lib._Z18vmx_int_gemm_gegluPKtPKvPtiiiP12ihipStream_t(C.c_void_p(x.data_ptr()), C.c_void_p(ws.data_ptr()), C.c_void_p(act.data_ptr()), M, inter,
                                                              K, None))
    torch.cuda.synchronize()
    w = q.double() * dt.double().T.repeat_interleave(256, 1)
    s = x.double() @ w.T
    gate, up = s[:, :inter].to(torch.bfloat16).double(), s[:, inter:].to(torch.bfloat16).double()
    cdf = 0.5 * (1 + torch.erf(gate / 2 ** 0.5))
    slope = cdf + gate * torch.exp(-gate * gate / 2) / (2 * np.pi) ** 0.5
    ref = gate * cdf * up
    bound = 2.0 ** -8 * ((slope * gate * up).abs() + 3 * ref.abs()) + 2.0 ** -20
    assert bool(((act.double() - ref).abs() <= bound).all())
    assert bool((guard[0] == 7.0).all()) and bool((guard[M + 1] == 7.0).all())


def _model(spec, types, seed=5):
    import torch
    from vllm_rust_amd.gemma4 import QuantizedGemma4ForCausalLM, T_K_NORM, T_Q_NORM
    model = QuantizedGemma4ForCausalLM(spec)
    ck = model.load_synthetic(slot_types=types, seed=seed, keep_host_copy=True)
    gq = torch.Generator(device="cuda").manual_seed(9)      # q/k norm weights of head_dim^-1/4: logits of order 1, as trained weights give
    for li in range(spec.num_layers):
        hd = spec.layer_geom(li)[0]
        for which, name in ((T_Q_NORM, "q_norm"), (T_K_NORM, "k_norm")):
            w = ((1.0 + 0.1 * torch.randn(hd, device="cuda", generator=gq)) * (1.0 / (hd ** 0.25))).to(torch.bfloat16)
            model.load_tensor(which, li, w)
            ck[f"{li}.{name}"] = w.cpu()
    return model, ck


# hidden 768: three scale groups, whose sums q|k|v, o and down take in slices; 128-row tiles from 65 rows on.  IQ4_XS (23) has no integer form: v, then
# gate (no GEGLU epilogue), then down (the epilogue's fp16 rows would have no reader)
@pytest.mark.parametrize("rows,types", [(65, {}), (130, {}), (300, {}), (130, {2: 23}), (65, {4: 23}), (65, {6: 23}), (33, {0: 17, 1: 21, 2: 22, 3: 17, 6: 22})])
def test_prompt_rows(gpu, rows, types):
    """Every row of the residual stream after one pass against the CPU oracle, which takes the same rows as one batch: 2e-2 relative L2 a row,
    as for the whole model."""
    vmx, torch = gpu
    from oracle import oracle as orc
    from tests.model_oracle import OracleGemma4
    from vllm_rust_amd.gemma4 import GEMMA4_12B_IQ3_MIX, Gemma4Spec
    spec = Gemma4Spec(768, 2, 4, 1280, 512, head_dim_sliding=64, head_dim_full=128, kv_heads_sliding=2, kv_heads_full=1, sliding_window=24,
                      full_every=2, max_position=512, kv_cache_dtype=0, num_blocks=24, max_batch=1, max_seq_len=320, max_prefill_tokens=300)
    model, ck = _model(spec, {**GEMMA4_12B_IQ3_MIX, **types})
    try:
        ref = OracleGemma4(spec, ck, model.cos_sin_sliding, model.cos_sin_full)
        bs = spec.block_size
        bt = np.random.default_rng(2).permutation(spec.num_blocks)[:20].astype(np.int32)[None]
        prompt = np.random.default_rng(1).integers(0, spec.vocab_size, rows).astype(np.int32)
        model.prefill(torch.from_numpy(prompt).cuda(), 0, torch.from_numpy(bt).cuda()[0])
        torch.cuda.synchronize()
        got = model.debug_read(0, (rows, spec.hidden_size)).double().cpu().numpy()
        pos = np.arange(rows, dtype=np.int32)
        _, h, _ = ref.decode(prompt, pos, (bt[0, pos // bs] * bs + pos % bs).astype(np.int32), np.repeat(bt, rows, axis=0), pos + 1)
        exp = orc.bf16_to_f32(h).astype(np.float64)
        assert (np.linalg.norm(got - exp, axis=1) <= 2e-2 * np.linalg.norm(exp, axis=1)).all()
    finally:
        model.close()


# 256- and 512-wide heads (attention results as fp16 rows) and projections of more than 8 M weights, whose slices of q|k|v, o and down the launches behind them
# add; IQ4_XS o (fp16 rows would have no reader) and k (no merged q|k|v) among them
@pytest.mark.parametrize("rows,types", [(65, {}), (200, {}), (65, {3: 23}), (65, {1: 23})])
def test_prompt_rows_wide_heads(gpu, rows, types):
    """As test_prompt_rows, the same bound."""
    vmx, torch = gpu
    from oracle import oracle as orc
    from tests.model_oracle import OracleGemma4
    from vllm_rust_amd.gemma4 import GEMMA4_12B_IQ3_MIX, Gemma4Spec
    spec = Gemma4Spec(2048, 2, 16, 4096, 512, head_dim_sliding=256, head_dim_full=512, kv_heads_sliding=2, kv_heads_full=1, sliding_window=24,
                      full_every=2, max_position=512, kv_cache_dtype=0, num_blocks=24, max_batch=1, max_seq_len=320, max_prefill_tokens=300)
    model, ck = _model(spec, {**GEMMA4_12B_IQ3_MIX, **types})
    try:
        ref = OracleGemma4(spec, ck, model.cos_sin_sliding, model.cos_sin_full)
        bs = spec.block_size
        bt = np.random.default_rng(2).permutation(spec.num_blocks)[:20].astype(np.int32)[None]
        prompt = np.random.default_rng(1).integers(0, spec.vocab_size, rows).astype(np.int32)
        model.prefill(torch.from_numpy(prompt).cuda(), 0, torch.from_numpy(bt).cuda()[0])
        torch.cuda.synchronize()
        got = model.debug_read(0, (rows, spec.hidden_size)).double().cpu().numpy()
        pos = np.arange(rows, dtype=np.int32)
        _, h, _ = ref.decode(prompt, pos, (bt[0, pos // bs] * bs + pos % bs).astype(np.int32), np.repeat(bt, rows, axis=0), pos + 1)
        exp = orc.bf16_to_f32(h).astype(np.float64)
        assert (np.linalg.norm(got - exp, axis=1) <= 2e-2 * np.linalg.norm(exp, axis=1)).all()
    finally:
        model.close()


def _launches(torch, types):
    """Kernels of one prompt pass, counted in a captured graph."""
    from vllm_rust_amd._lib import check, lib
    from vllm_rust_amd.gemma4 import GEMMA4_12B_IQ3_MIX, Gemma4Spec
    spec = Gemma4Spec(256, 3, 4, 256, 512, head_dim_sliding=64, head_dim_full=64, kv_heads_sliding=4, kv_heads_full=4, sliding_window=64, full_every=4,
                      max_position=128, kv_cache_dtype=0, num_blocks=8, max_batch=1, max_seq_len=96, max_prefill_tokens=64)
    model, _ = _model(spec, {**GEMMA4_12B_IQ3_MIX, **types})
    try:
        ids, slots, bt = (torch.arange(n, dtype=torch.int32, device="cuda") for n in (40, 40, 4))
        out = torch.zeros(1, dtype=torch.int32, device="cuda")
        run = lambda: check(lib.vmx_gemma4_prefill(model._h, ids.data_ptr(), 0, slots.data_ptr(), bt.data_ptr(), 40, out.data_ptr(), None,   # noqa: E731
                                                   torch.cuda.current_stream().cuda_stream))
        run()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph(keep_graph=True)
        with torch.cuda.graph(graph):
            run()
        n = C.c_size_t(0)
        assert C.CDLL("libamdhip64.so").hipGraphGetNodes(C.c_void_p(graph.raw_cuda_graph()), None, C.byref(n)) == 0
        return n.value
    finally:
        model.close()


def test_mixed_group_converts_its_rows_once(gpu):
    """One scale group, so no slices: an integer projection and an IQ4_XS one are an expansion and a product each, and the fp16 copy of the rows
    that the integer ones read is made once for the group.  q and k integer is then as many launches as q alone."""
    vmx, torch = gpu
    assert _launches(torch, {0: 18, 1: 22, 2: 23}) == _launches(torch, {0: 18, 1: 23, 2: 23})
