"""Gemma-4 prompts: norm, rotation and cache write of 256- and 512-wide heads, in both cache types, with K as V, shared layers and heads rotated in part."""
import numpy as np
import pytest

from tests.test_gpu_gemma4_prompts import _model, gpu  # noqa: F401

pytestmark = pytest.mark.gpu


# 24 rotated dimensions do not end with a lane's eight elements: the form of any size
@pytest.mark.parametrize("rows,kv,k_eq_v,shared,rotated", [(67, 1, False, 0, 0.25), (33, 0, True, 0, 1.0), (65, 0, False, 1, 0.0625), (65, 1, True, 0, 0.047)])
def test_wide_heads(gpu, rows, kv, k_eq_v, shared, rotated):  # noqa: F811
    """Every row of the residual stream against the CPU oracle: 2e-2 relative L2 a row with a bf16 cache, as for the whole model; an FP8 cache on both
    sides may round an element to the other neighbour (2^-4 of it): 5e-2."""
    vmx, torch = gpu
    from oracle import oracle as orc
    from tests.model_oracle import OracleGemma4
    from vllm_rust_amd.gemma4 import GEMMA4_12B_IQ3_MIX, Gemma4Spec
    spec = Gemma4Spec(1024, 2 + shared, 4, 1024, 512, head_dim_sliding=256, head_dim_full=512, kv_heads_sliding=2, kv_heads_full=1, sliding_window=24,
                      full_every=2, k_eq_v_on_full=k_eq_v, num_kv_shared_layers=shared, partial_rotary_factor_full=rotated, max_position=512,
                      kv_cache_dtype=kv, num_blocks=24, max_batch=1, max_seq_len=320, max_prefill_tokens=300)
    assert spec.rot_dim_full() % 16 == (8 if rotated == 0.047 else 0)
    model, ck = _model(spec, GEMMA4_12B_IQ3_MIX)
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
        assert (np.linalg.norm(got - exp, axis=1) <= (5e-2 if kv else 2e-2) * np.linalg.norm(exp, axis=1)).all()
    finally:
        model.close()
