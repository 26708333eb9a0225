"""Gemma-4 prompts past 16 rows: the integer products of merged projections at the edges of their tiles, slices and scale groups, and
groups whose projections do not all have the integer form."""
import ctypes as C

import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    import torch
    import vllm_rust_amd as vmx
    vmx.init(0)
    return vmx, torch


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
