"""int4 layers at 5 .. 16 rows whose residual adds and norm gains sit in the epilogues of o_proj, down and the expert combine and whose norms'
row factors multiply the sums of the next linear, against the composed CPU oracle: the fewest and the most rows, an odd count, and the row
below, which takes another form.  Every row of the dense model is compared by itself, since each has a factor of its own; single rows of the experts' model
move by up to 0.04 whichever form computes them (the router's probabilities are rounded to bf16), so its batch is compared as a whole."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", params=[False, True], ids=["dense", "experts"])
def models(request):
    import torch
    import vllm_rust_amd as vmx
    from tests.model_oracle import OracleQwen3
    from vllm_rust_amd.qwen3 import QuantizedQwen3ForCausalLM, Qwen3Spec, rope_cos_sin_cache
    vmx.init(0)
    moe = request.param
    # q|k|v 2048 -> 6144 in two slices, o 4096 deep (four passes), gate|up 2048 -> 12288, down 6144 deep (six): the smallest widths the form takes
    spec = Qwen3Spec(hidden_size=2048, num_layers=2, num_heads=32, num_kv_heads=8, head_dim=128, intermediate_size=512 if moe else 6144, vocab_size=500,
                     max_position=128, num_blocks=32, max_batch=16, max_seq_len=64, max_prefill_tokens=16, qk_norm=not moe, num_experts=4 if moe else 0, experts_per_tok=4 if moe else 0)   # all experts: no row can land on another choice
    model = QuantizedQwen3ForCausalLM(spec)
    ck = (model.load_synthetic_moe if moe else model.load_synthetic)(seed=5, keep_host_copy=True)
    yield torch, spec, model, lambda: OracleQwen3(spec, ck, rope_cos_sin_cache(spec.head_dim, spec.max_position, spec.rope_theta))
    model.close()


@pytest.mark.parametrize("rows", [4, 5, 11, 16])
def test_layers_match_oracle(models, rows):
    from oracle import oracle as orc
    torch, spec, model, oracle = models
    ref = oracle()
    bt = np.arange(rows * 2, dtype=np.int32).reshape(rows, 2)
    ids = np.random.default_rng(rows).integers(0, spec.vocab_size, rows).astype(np.int32)
    for p in range(2):
        pos = np.full(rows, p, np.int32)
        slots = (bt[:, 0] * spec.block_size + p).astype(np.int32)
        logits = torch.empty((rows, spec.vocab_size), dtype=torch.bfloat16, device="cuda")
        out = model.forward_decode_batch(*(torch.from_numpy(a).cuda() for a in (ids, pos, slots, bt, pos + 1)), logits=logits)
        torch.cuda.synchronize()
        exp, exp_h, _ = ref.decode(ids, pos, slots, bt, pos + 1)
        got = orc.bf16_to_f32(logits.cpu().view(torch.int16).numpy().view(np.uint16)); exp = orc.bf16_to_f32(exp)
        got_h = orc.bf16_to_f32(model.debug_read(0, (rows, spec.hidden_size)).cpu().view(torch.int16).numpy().view(np.uint16)); exp_h = orc.bf16_to_f32(exp_h)
        for g, e in ((got, exp), (got_h, exp_h)):   # the decoder tests' bar
            err, norm = ((g - e) ** 2).sum(1), (e ** 2).sum(1)
            rel = np.sqrt(err.sum() / norm.sum() if spec.num_experts else (err / norm).max())
            assert rel <= 3e-2, (p, rel)
        ids = out.cpu().numpy().astype(np.int32)


@pytest.mark.parametrize("rows", [5, 16])
def test_short_prompts_match_oracle(models, rows):
    """Prompts of as many rows take the same layers: a first part and one with history, every row of the residual stream and the last row's logits."""
    from oracle import oracle as orc
    torch, spec, model, oracle = models
    ref = oracle()
    bt = np.random.default_rng(rows).permutation(spec.num_blocks)[:2 * rows // spec.block_size + 1].astype(np.int32)
    for part in range(2):
        ids = np.random.default_rng(10 * rows + part).integers(0, spec.vocab_size, rows).astype(np.int32)
        pos = np.arange(part * rows, (part + 1) * rows, dtype=np.int32)
        last = torch.empty(spec.vocab_size, dtype=torch.bfloat16, device="cuda")
        model.prefill(torch.from_numpy(ids).cuda(), part * rows, torch.from_numpy(bt).cuda(), logits_last=last)
        got_h = model.debug_read(0, (rows, spec.hidden_size)).double().cpu().numpy()
        slots = (bt[pos // spec.block_size] * spec.block_size + pos % spec.block_size).astype(np.int32)
        exp, exp_h, _ = ref.decode(ids, pos, slots, np.repeat(bt[None], rows, axis=0), pos + 1)
        for g, e in ((last.double().cpu().numpy()[None], orc.bf16_to_f32(exp[-1:])), (got_h, orc.bf16_to_f32(exp_h))):   # the decoder tests' bar
            err, norm = ((g - e) ** 2).sum(1), (e.astype(np.float64) ** 2).sum(1)
            assert np.sqrt(err.sum() / norm.sum() if spec.num_experts else (err / norm).max()) <= 3e-2, part


_SMALL = dict(hidden_size=256, num_heads=4, num_kv_heads=2, head_dim=64, intermediate_size=512)
_WIDE = dict(hidden_size=2048, num_heads=32, num_kv_heads=8, head_dim=128, intermediate_size=12288)


@pytest.mark.parametrize("sizes,rows", [(_SMALL, 49), (_SMALL, 64), (_SMALL, 65), (_SMALL, 130), (_WIDE, 320), (_WIDE, 321), (_WIDE, 333), (_WIDE, 336), (_WIDE, 337)])
def test_prompts_match_the_decode_path(sizes, rows):
    """Prompts whose linears take all of k in one slice pass bf16 sums on (256 and 512 wide, so that every projection does); 1 to 16 rows behind the last
    whole tile take a pass of their own (gate|up, q|k|v), none and 17 do not."""
    import torch
    import vllm_rust_amd as vmx
    from vllm_rust_amd.qwen3 import QuantizedQwen3ForCausalLM, Qwen3Spec
    vmx.init(0)
    spec = Qwen3Spec(**sizes, num_layers=2, vocab_size=1000, max_position=512, num_blocks=24, max_batch=16, max_seq_len=384, max_prefill_tokens=rows)
    model = QuantizedQwen3ForCausalLM(spec)
    model.load_synthetic(seed=9)
    prompt = torch.randint(0, spec.vocab_size, (rows,), dtype=torch.int32, device="cuda", generator=torch.Generator(device="cuda").manual_seed(rows))
    bt = torch.randperm(24, dtype=torch.int32, device="cuda")
    got = torch.empty(spec.vocab_size, dtype=torch.bfloat16, device="cuda")
    _, want = model.forward(prompt, 0, bt)
    model.prefill(prompt, 0, bt, logits_last=got)
    torch.cuda.synchronize()
    want = want[-1].float()
    assert float((got.float() - want).norm() / want.norm()) <= 2e-2   # the decoder tests' bar
    model.close()
