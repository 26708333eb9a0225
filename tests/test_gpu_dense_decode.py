"""Unquantised (bf16) layers: decode rows run as norm-prologue / residual-epilogue products, prompts on the tiled linears.  Checked
against the CPU oracle model at every workgroup width and a K that ends in half a block."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    import torch
    import vllm_rust_amd as vmx
    vmx.init(0)
    return vmx, torch


# (hidden, query heads, KV heads, head_dim, intermediate), contexts: K of 1.5 ... 25 blocks (4, 8, 16 waves; 192 = one block and a half); one to
# four rows merge the attention partitions, five and sixteen read attention rows; past 512 tokens the merge is a launch of its own
@pytest.mark.parametrize("geometry,contexts", [
    ((640, 3, 1, 64, 1152), [0]),
    ((640, 3, 1, 64, 1152), [3, 64, 17, 254]),
    ((1664, 18, 6, 128, 3200), [40, 7, 300]),
    ((2176, 16, 8, 128, 640), [600]),
    ((640, 5, 5, 64, 2176), [9, 2, 33, 70, 0]),
    ((1664, 18, 6, 128, 640), list(range(1, 17))),
    ((640, 3, 1, 64, 8960), [40, 7]),
])
def test_dense_decode_rows(gpu, geometry, contexts):
    """bf16 rounding points are the oracle's and only the order of the f32 sums differs: 2e-2 relative L2, as for the whole models."""
    from tests.test_gpu_true_geometry import _decode_and_compare, _fill_kv
    from tests.model_oracle import OracleQwen3
    from vllm_rust_amd.qwen3 import QuantizedQwen3ForCausalLM, Qwen3Spec, rope_cos_sin_cache
    vmx, torch = gpu
    H, hq, hkv, hd, inter = geometry
    B = len(contexts)
    spec = Qwen3Spec(H, 3, hq, hkv, hd, inter, 512, tie_word_embeddings=True, max_position=1024, num_blocks=96, max_batch=B,
                     max_seq_len=1024, max_prefill_tokens=48)
    model = QuantizedQwen3ForCausalLM(spec)
    try:
        ck = model.load_synthetic_bf16(seed=21, keep_host_copy=True)
        ref = OracleQwen3(spec, ck, rope_cos_sin_cache(spec.head_dim, spec.max_position, spec.rope_theta))
        shape = (spec.num_blocks, spec.block_size, spec.num_kv_heads, spec.head_dim)
        _fill_kv(torch, model, ref, spec.num_layers, [shape] * spec.num_layers, spec.kv_cache_dtype, seed=3)
        _decode_and_compare(torch, model, ref, spec, contexts, 2, [17 + 5 * b for b in range(B)])
    finally:
        model.close()


# every head width (heads, KV heads, head_dim, FP8 cache): the q/k/v kernel's lanes a head, the attention's tiles before, at and past 16 tokens
@pytest.mark.parametrize("heads,kv_heads,head_dim,fp8", [(3, 1, 64, 0), (2, 1, 128, 1), (2, 1, 256, 0), (3, 1, 256, 1), (2, 2, 512, 0), (4, 1, 512, 1)])
@pytest.mark.parametrize("tokens", [2, 17, 40])
def test_dense_prompt_rows(gpu, tokens, heads, kv_heads, head_dim, fp8):
    """The last hidden row of a prompt pass against the oracle fed the same tokens one at a time."""
    from tests.model_oracle import OracleQwen3
    from vllm_rust_amd.qwen3 import QuantizedQwen3ForCausalLM, Qwen3Spec, rope_cos_sin_cache
    from oracle import oracle as orc
    vmx, torch = gpu
    spec = Qwen3Spec(640, 3, heads, kv_heads, head_dim, 1152, 512, tie_word_embeddings=True, max_position=256, num_blocks=8, max_batch=1,
                     max_seq_len=64, max_prefill_tokens=48, kv_cache_dtype=fp8)
    model = QuantizedQwen3ForCausalLM(spec)
    try:
        ck = model.load_synthetic_bf16(seed=5, keep_host_copy=True)
        ref = OracleQwen3(spec, ck, rope_cos_sin_cache(spec.head_dim, spec.max_position, spec.rope_theta))
        ids = np.random.default_rng(tokens).integers(0, 512, tokens).astype(np.int32)
        bt = np.asarray([[5, 2, 7, 1]], np.int32)
        model.prefill(torch.from_numpy(ids).cuda(), 0, torch.from_numpy(bt[0]).cuda())
        torch.cuda.synchronize()
        got = model.debug_read(0, (tokens, 640))[-1].float().cpu().numpy()
        for p in range(tokens):
            slot = np.asarray([bt[0, p // spec.block_size] * spec.block_size + p % spec.block_size], np.int32)
            _, h, _ = ref.decode(ids[p:p + 1], np.asarray([p], np.int32), slot, bt, np.asarray([p + 1], np.int32))
        exp = orc.bf16_to_f32(h)[0]
        assert np.linalg.norm(got - exp) <= 2e-2 * np.linalg.norm(exp)
    finally:
        model.close()


# KV heads times rows of 6, 128, 256 and 512 on 256 compute units: 42 and 4 partitions a KV head up to 2048 tokens, block tables of more than 64
# entries; of 128, 256 and 512 up to 1024 tokens: 4, 2 and 1; beyond 2048 tokens never fewer than 8
@pytest.mark.parametrize("heads,kv_heads,head_dim,rows,longest", [
    (4, 2, 64, 3, 1100), (8, 8, 128, 16, 1100), (16, 16, 64, 16, 1100), (32, 32, 64, 16, 1100), (8, 8, 128, 16, 900), (16, 16, 64, 16, 900),
    (32, 32, 64, 16, 900), (32, 32, 64, 9, 2100)])
def test_long_contexts_partitions(gpu, heads, kv_heads, head_dim, rows, longest):
    from tests.test_gpu_true_geometry import _decode_and_compare, _fill_kv
    from tests.model_oracle import OracleQwen3
    from vllm_rust_amd.qwen3 import QuantizedQwen3ForCausalLM, Qwen3Spec, rope_cos_sin_cache
    vmx, torch = gpu
    contexts = [min(c, longest) for c in [longest, 3, 1030, 0, 15, 16, 17, 511, 512, 700, 1023, 1024, 255, 64, 900, 1][:rows]]
    spec = Qwen3Spec(256, 2, heads, kv_heads, head_dim, 256, 512, tie_word_embeddings=True, max_position=4096, num_blocks=(longest // 16 + 4) * rows,
                     max_batch=rows, max_seq_len=longest + 100, max_prefill_tokens=16)
    model = QuantizedQwen3ForCausalLM(spec)
    try:
        ck = model.load_synthetic_bf16(seed=21, keep_host_copy=True)
        ref = OracleQwen3(spec, ck, rope_cos_sin_cache(spec.head_dim, spec.max_position, spec.rope_theta))
        shape = (spec.num_blocks, spec.block_size, spec.num_kv_heads, spec.head_dim)
        _fill_kv(torch, model, ref, spec.num_layers, [shape] * spec.num_layers, spec.kv_cache_dtype, seed=3)
        _decode_and_compare(torch, model, ref, spec, contexts, 1, [17 + 5 * b for b in range(rows)])
    finally:
        model.close()
