"""What this framework is used for, as cases that can be timed and compared.

A user of the framework loads a checkpoint into one of its executors and then serves it: a prompt goes through the executor's
native prompt pass, and from then on every step is one decode pass over the running sequences, captured once into a graph and
replayed.  The cases are those two passes for the models that the benchmark and the tests run: Qwen3-8B with AWQ int4 linears (the
headline model), Qwen3-8B with EXL3 trellis linears in fp16, Gemma-4-12B with GGUF I-quant linears and an FP8 cache, Mixtral-8x7B with
GPTQ experts, the small unquantised Qwen3-0.6B, and one of the configuration-described families (Larolorn, the benchmark's larger size).

Every model has its true layer sizes.  The deep ones are slices: Qwen3-8B 9 of 36 layers, Gemma 12 of 48 (ten windowed and two full
ones, as in the whole), Mixtral 4 of 32, each with the same share of the vocabulary, so that layers and logits stand to each other
as in the whole model while a state is made in a fraction of a second.  Weights are random in the checkpoint's own format.

A decode case starts from caches that already hold the sequences' rows and repeats one step (the row it writes is the same each
time); the lengths of several sequences are spread from `context` down to half of it.  A prompt case repeats a whole prompt from
position 0.  Larolorn's decode step carries its matrix memories on from pass to pass, as in use.
Every cached row of a prompt reaches the logits of its last token through the attention of the layers, so the logits stand for them.
"""
import math
import os
import struct

import torch

BLOCK = 16            # tokens per cache page (the benchmark's)
GROUP = 128           # int4 quantisation group

# model -> sizes.  kind: how the linears are stored.
QWEN = {
    "qwen3_0_6b_bf16": dict(kind="bf16", width=1024, layers=28, heads=16, kv=8, ff=3072, vocab=151936, tied=True),
    "qwen3_8b_awq": dict(kind="awq", width=4096, layers=9, heads=32, kv=8, ff=12288, vocab=37984, tied=False),
    "qwen3_8b_exl3": dict(kind="exl3", width=4096, layers=9, heads=32, kv=8, ff=12288, vocab=37984, tied=False),
    "mixtral_8x7b_gptq": dict(kind="moe", width=4096, layers=4, heads=32, kv=8, ff=14336, vocab=4000, tied=False, experts=8, top=2),
}
HEAD = 128
GEMMA = dict(width=3840, layers=12, heads=16, ff=15360, vocab=65536, softcap=30.0, eps=1e-6)
IQ_SIZE = {18: 98, 22: 82, 21: 110}                      # GGUF super-block bytes: IQ3_XXS, IQ2_S, IQ3_S
GEMMA_TYPES = {0: 18, 1: 22, 2: 18, 3: 21, 4: 18, 5: 18, 6: 21}   # q k v o gate up down of the UD-IQ3_XXS mix
LARO = dict(width=2048, lat=(16, 128, 64, 128, 512, 4096), att=(16, 4, 128, 4096), mem=(16, 128), ff=6144, vocab=32000, limit=7.0, eps=1e-6, mult=0.5)


def listed():
    return [
        # one user talking to the smallest model: the shortest step there is, nearly all of it launches and first loads
        {"name": "qwen3-0.6b decode 1", "model": "qwen3_0_6b_bf16", "phase": "decode", "rows": 1, "context": 128},
        # the headline: one sequence on the AWQ model, a few hundred tokens in
        {"name": "qwen3-8b awq decode 1", "model": "qwen3_8b_awq", "phase": "decode", "rows": 1, "context": 300},
        # a serving batch of 16 sequences of unequal length
        {"name": "qwen3-8b awq decode 16", "model": "qwen3_8b_awq", "phase": "decode", "rows": 16, "context": 1500},
        # a chat turn of an odd length
        {"name": "qwen3-8b awq prompt 333", "model": "qwen3_8b_awq", "phase": "prompt", "rows": 333, "context": 0},
        # a document
        {"name": "qwen3-8b awq prompt 2048", "model": "qwen3_8b_awq", "phase": "prompt", "rows": 2048, "context": 0},
        # the trellis-quantised checkpoint, fp16 end to end
        {"name": "qwen3-8b exl3 decode 1", "model": "qwen3_8b_exl3", "phase": "decode", "rows": 1, "context": 300},
        # GGUF I-quants over an FP8 cache: one sequence, and the benchmark's prompt
        {"name": "gemma4-12b iq3 decode 1", "model": "gemma4_12b_iq3", "phase": "decode", "rows": 1, "context": 300},
        {"name": "gemma4-12b iq3 prompt 256", "model": "gemma4_12b_iq3", "phase": "prompt", "rows": 256, "context": 0},
        # mixture of experts: a small serving batch, and the benchmark's prompt
        {"name": "mixtral gptq decode 8", "model": "mixtral_8x7b_gptq", "phase": "decode", "rows": 8, "context": 500},
        {"name": "mixtral gptq prompt 256", "model": "mixtral_8x7b_gptq", "phase": "prompt", "rows": 256, "context": 0},
        # a configuration-described family: three prompts of unequal length packed into one step, and a serving batch
        {"name": "larolorn prompt 1500", "model": "larolorn_2k", "phase": "prompt", "rows": 1500, "context": 0},
        {"name": "larolorn decode 16", "model": "larolorn_2k", "phase": "decode", "rows": 16, "context": 1000},
    ]


# longest drawn prompt of a model (the shortest has 33 tokens); decode: 1 to 16 sequences of 32 to 2047 cached tokens
_MOST = {"qwen3_8b_awq": 2000, "gemma4_12b_iq3": 512, "mixtral_8x7b_gptq": 512, "larolorn_2k": 2000}


def draw(rng):
    which = rng.choice([(c["model"], c["phase"]) for c in listed()])
    log = lambda lo, hi: int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))   # noqa: E731
    if which[1] == "prompt":
        return {"model": which[0], "phase": "prompt", "rows": log(33, _MOST[which[0]]), "context": 0}
    return {"model": which[0], "phase": "decode", "rows": log(1, 16), "context": log(32, 2047)}


# ------------------------------------------------------------------------------------------------ inputs, from the seed alone
def _gen(seed, salt):
    return torch.Generator(device="cuda").manual_seed(1_000_003 * (seed + 1) + salt)


def _rand(g, *shape):
    return torch.rand(shape, device="cuda", generator=g)


def _randn(g, *shape):
    return torch.randn(shape, device="cuda", generator=g)


def _words(g, *shape):
    return torch.randint(-2 ** 31, 2 ** 31 - 1, shape, dtype=torch.int32, device="cuda", generator=g)


def _gains(g, n, dtype):
    return (1.0 + 0.1 * _randn(g, n)).to(dtype)


def _lengths(case):
    """Rows that each sequence has in its cache before the step."""
    n, c = case["rows"], case["context"]
    return [c - (c // 2) * b // n for b in range(n)]


def _prompt_lengths(case):
    """Larolorn packs a step's prompts: two fifths, a third and the rest."""
    n = case["rows"]
    a, b = 2 * n // 5, n // 3
    return [a, b, n - a - b]


def _steps_of(case, seed):
    """Token ids and the scattered block table of the sequences (host-side choices on the GPU's generator)."""
    g = _gen(seed, 7)
    lens = _lengths(case) if case["phase"] == "decode" else [case["rows"]]
    width = max(lens) // BLOCK + 1
    n = len(lens)
    table = torch.randperm(n * width, device="cuda", generator=g).to(torch.int32).reshape(n, width).contiguous()
    ids = torch.randint(0, _vocab(case), (case["rows"],), dtype=torch.int32, device="cuda", generator=g)
    return ids, table, lens


def _vocab(case):
    m = case["model"]
    return QWEN[m]["vocab"] if m in QWEN else GEMMA["vocab"] if m == "gemma4_12b_iq3" else LARO["vocab"]


def _qwen_shapes(m):
    W, Q, K, F = m["width"], m["heads"] * HEAD, m["kv"] * HEAD, m["ff"]
    sh = [(W, Q), (W, K), (W, K), (Q, W)]
    return sh if m["kind"] == "moe" else sh + [(W, F), (W, F), (F, W)]


def _qwen_linear(m, g, K, N, gain=1.0):
    """One projection K -> N in the checkpoint's format, of gain `gain`."""
    if m["kind"] == "bf16":
        return (_randn(g, N, K) * (gain / math.sqrt(K))).to(torch.bfloat16)
    if m["kind"] == "exl3":
        tr = torch.randint(-32768, 32767, (K // 16, N // 16, 64), dtype=torch.int16, device="cuda", generator=g)
        suh = (torch.randint(0, 2, (K,), device="cuda", generator=g) * 2 - 1).to(torch.float16)
        svh = ((torch.randint(0, 2, (N,), device="cuda", generator=g) * 2 - 1) * (_rand(g, N) * 0.5 + 0.75) * (gain / math.sqrt(K))).to(torch.float16)
        return tr, suh, svh
    sc = ((_rand(g, K // GROUP, N) * 0.5 + 0.75) * (gain / (6.5 * math.sqrt(K)))).to(torch.float16)
    return _words(g, K, N // 8), _words(g, K // GROUP, N // 8), sc


def _qwen_expert(m, g):
    def one(K, N, gain=1.0):
        w = _words(g, K // 8, N)                             # symmetric weights: a nibble of 0 (-8) becomes 8 (0), so that the mean is 0
        return w | ((~(w | w >> 1 | w >> 2 | w >> 3) & 0x11111111) << 3), ((_rand(g, K // GROUP, N) * 0.5 + 0.75) * (gain / (4.6 * math.sqrt(K)))).to(torch.float16)
    return one(m["width"], m["ff"]), one(m["width"], m["ff"]), one(m["ff"], m["width"], _branch(m))


def _branch(m):
    """Gain of the projections that write to the residual stream, as depth-scaled initialisation has it."""
    return 1.0 / math.sqrt(2 * m["layers"])


def _qwen_dtype(m):
    return torch.float16 if m["kind"] == "exl3" else torch.bfloat16


def _expert_directions(m, seed):
    return _randn(_gen(seed, 3), m["experts"], m["width"])


def _favoured(m):
    """Two experts for every token of the vocabulary: embeddings lean towards them, so that routing has the margins of a trained router
    (with none, a rounding error swaps whole experts)."""
    t, n = torch.arange(m["vocab"], device="cuda"), m["experts"]
    return torch.stack([t % n, (t + 1 + t // n % (n - 1)) % n], 1)


def _qwen_ends(m, seed):
    """Embedding, head (None where tied) and final gain.  The head is the embedding moved by one token, so that a step has a clear
    answer, as a trained model's has."""
    g, dt = _gen(seed, 1), _qwen_dtype(m)
    emb = _randn(g, m["vocab"], m["width"]) * 0.5
    if m["kind"] == "moe":
        emb += _expert_directions(m, seed)[_favoured(m)].mul_(torch.tensor([0.4, 0.25], device="cuda")[:, None]).sum(1)
    emb = emb.to(dt)
    head = None if m["tied"] else (emb.float().roll(1, 0) * 0.1).to(dt)
    return emb, head, _gains(g, m["width"], dt)


def _qwen_layer(m, seed, li):
    g, dt = _gen(seed, 100 + li), _qwen_dtype(m)
    gains = [_gains(g, n, dt) for n in (m["width"], m["width"], HEAD, HEAD)]
    lin = [_qwen_linear(m, g, K, N, _branch(m) if slot in (3, 6) else 1.0) for slot, (K, N) in enumerate(_qwen_shapes(m))]
    if m["kind"] != "moe":
        return gains, lin, None, None
    return gains, lin, (_expert_directions(m, seed).roll(li, 0) * (8.0 / m["width"])).to(dt), [_qwen_expert(m, g) for _ in range(m["experts"])]


def _qwen_cache(m, seed, li, blocks):
    g, dt = _gen(seed, 5000 + li), _qwen_dtype(m)
    return [_randn(g, blocks, BLOCK, m["kv"], HEAD).to(dt) for _ in range(2)]


def _gemma_geom(li):
    """(head width, KV heads, rotated numbers, window) of layer li; every sixth layer is a full one."""
    return (512, 1, 128, 0) if (li + 1) % 6 == 0 else (256, 8, 256, 1024)


def _gemma_shapes(li):
    hd, kv = _gemma_geom(li)[:2]
    W, Q, K, F = GEMMA["width"], GEMMA["heads"] * hd, kv * hd, GEMMA["ff"]
    return {0: (W, Q), 1: (W, K), 2: (W, K), 3: (Q, W), 4: (W, F), 5: (W, F), 6: (F, W)}


def _super_scales(raw, at, d):
    bits = d.to(torch.float16).view(torch.int16)
    raw[:, at] = (bits & 0xFF).to(torch.uint8)
    raw[:, at + 1] = ((bits >> 8) & 0xFF).to(torch.uint8)


def _gemma_ends(seed):
    g = _gen(seed, 1)
    blocks = GEMMA["vocab"] * GEMMA["width"] // 256
    tab = torch.randint(0, 256, (blocks, 110), dtype=torch.uint8, device="cuda", generator=g)
    _super_scales(tab, 108, (_rand(g, blocks) * 0.5 + 0.75) * 0.0008)
    return tab, _gains(g, GEMMA["width"], torch.bfloat16)


def _gemma_layer(seed, li):
    """Gains (input, post-attention, pre-feed-forward, post-feed-forward, q, k, layer scalar) and raw I-quant blocks per projection.
    Attention runs with scale 1, so q's gains carry 1 / sqrt(head width); the gains behind a sublayer are small, as trained ones are."""
    g, W, hd = _gen(seed, 100 + li), GEMMA["width"], _gemma_geom(li)[0]
    gains = [(_gains(g, W, torch.float32) * s).to(torch.bfloat16) for s in (1.0, 0.2, 1.0, 0.2)]
    gains.append(((1.0 + 0.1 * _randn(g, hd)) / math.sqrt(hd)).to(torch.bfloat16))
    gains.append(_gains(g, hd, torch.bfloat16))
    gains.append((0.75 + 0.5 * _rand(g, 1)).to(torch.bfloat16))
    lin = {}
    for slot, (K, N) in _gemma_shapes(li).items():
        nb = N * K // 256
        raw = torch.randint(0, 256, (nb, IQ_SIZE[GEMMA_TYPES[slot]]), dtype=torch.uint8, device="cuda", generator=g)
        _super_scales(raw, 0, (_rand(g, nb) * 0.5 + 0.75) / (120.0 * math.sqrt(K)))
        lin[slot] = raw
    return gains, lin


def _gemma_cache(seed, li, blocks):
    hd, kv = _gemma_geom(li)[:2]
    g = _gen(seed, 5000 + li)
    return [_randn(g, blocks, BLOCK, kv, hd).to(torch.float8_e4m3fn) for _ in range(2)]


def _laro_weights(seed):
    """Name -> bf16 tensor of a checkpoint: latent attention, attention beside a memory, and both again."""
    g, W, F = _gen(seed, 1), LARO["width"], LARO["ff"]
    H, D, RD, V, R, _ = LARO["lat"]
    AH, AG, AD, _ = LARO["att"]
    MH, MD = LARO["mem"]
    shapes = {"embed": (LARO["vocab"], W)}
    for i in range(4):
        p = f"l{i}."
        shapes[p + "norm1"], shapes[p + "norm2"] = (W,), (W,)
        if i % 2 == 0:
            for n, s in (("q", (H * (D + RD), W)), ("dkv", (R + RD, W)), ("dkv.norm", (R,)), ("uk", (H * D, R)), ("uv", (H * V, R)), ("g", (H, W)), ("o", (W, H * V))):
                shapes[p + "mix." + n] = s
        else:
            for n, rows in (("q", AH * AD), ("k", AG * AD), ("v", AG * AD)):
                shapes[p + f"mix.left.{n}"], shapes[p + f"mix.left.{n}.b"] = (rows, W), (rows,)
            for n, s in (("left.q.norm", (AH * AD,)), ("left.k.norm", (AG * AD,)), ("left.sink", (AH,)), ("left.o", (W, AH * AD)), ("left.o.b", (W,)),
                         ("right.q", (MH * MD, W)), ("right.k", (MH * MD, W)), ("right.v", (MH * MD, W)), ("right.g", (MH * MD, W)),
                         ("right.o", (W, MH * MD)), ("right.norm", (MH * MD,)), ("left.out", (W,)), ("right.out", (W,))):
                shapes[p + "mix." + n] = s
        shapes[p + "mlp.gate"], shapes[p + "mlp.up"], shapes[p + "mlp.down"] = (F, W), (F, W), (W, F)
    shapes["final.norm"], shapes["head"] = (W,), (LARO["vocab"], W)
    out = {}
    for name, s in shapes.items():
        if name.endswith((".out", "norm", "norm1", "norm2")):
            t = 1.0 + 0.1 * _randn(g, *s)
        elif name.endswith(".b"):
            t = 0.5 * _randn(g, *s)
        elif name == "head":
            t = out["embed"].float().roll(1, 0) / math.sqrt(s[-1])
        elif name == "embed" or name.endswith(".sink"):
            t = _randn(g, *s)
        else:
            t = _randn(g, *s) / math.sqrt(s[-1])
        out[name] = t.to(torch.bfloat16)
    return out


def _laro_decay():
    n = LARO["mem"][0]
    return [1.0 - 2.0 ** (-5 - 5 * i / (n - 1)) for i in range(n)]


def _laro_tokens(case, seed):
    """Token ids of every sequence's prompt, and (decode) of the step's tokens."""
    g = _gen(seed, 7)
    lens = _lengths(case) if case["phase"] == "decode" else _prompt_lengths(case)
    ids = [torch.randint(0, LARO["vocab"], (n,), dtype=torch.int32, device="cuda", generator=g) for n in lens]
    step = torch.randint(0, LARO["vocab"], (len(lens),), dtype=torch.int32, device="cuda", generator=g)
    width = max(lens) // BLOCK + 1
    table = torch.randperm(len(lens) * width, device="cuda", generator=g).to(torch.int32).reshape(len(lens), width).contiguous()
    return ids, step, table, lens


# ------------------------------------------------------------------------------------------------ what a program has in hand
def _i32(a):
    return torch.as_tensor(a, dtype=torch.int32, device="cuda").contiguous()


def _captured(step, before_replay=None):
    """The step as a graph, the way a server runs it: once eagerly (first-call set-up), then recorded."""
    step()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step()
    if before_replay is not None:
        before_replay()
    torch.cuda.synchronize()
    return graph


def _decode_inputs(ids, table, lens):
    pos = _i32(lens)
    slots = (table[torch.arange(len(lens), device="cuda"), (pos // BLOCK).long()] * BLOCK + pos % BLOCK).to(torch.int32).contiguous()
    return ids, pos, slots, table, (pos + 1).contiguous()


def _ready(case, model, ids, table, lens, act):
    """The state of a Qwen3-shaped or Gemma executor whose weights and caches are in place."""
    if case["phase"] == "prompt":
        return {"case": case, "model": model, "ids": ids, "table": table[0].contiguous(), "out": torch.empty(1, dtype=torch.int32, device="cuda"),
                "logits": torch.empty(_vocab(case), dtype=act, device="cuda")}
    args = _decode_inputs(ids, table, lens)
    out = torch.empty(case["rows"], dtype=torch.int32, device="cuda")
    logits = torch.empty((case["rows"], _vocab(case)), dtype=act, device="cuda")
    step = lambda: model.forward_decode_batch(*args, max_seq_len=_bound(case), out_ids=out, logits=logits)   # noqa: E731
    return {"case": case, "graph": _captured(step), "keep": args, "model": model, "out": out, "logits": logits}


def _bound(case):
    """The sequence length a captured step is good for: some generation beyond the context."""
    return case["context"] + 128


def prepare(case, seed):
    import vllm_rust_amd as vmx
    vmx.init(0)
    if case["model"] in QWEN:
        return _prepare_qwen(case, seed)
    return _prepare_gemma(case, seed) if case["model"] == "gemma4_12b_iq3" else _prepare_laro(case, seed)


def _prepare_qwen(case, seed):
    from vllm_rust_amd import qwen3 as q
    m = QWEN[case["model"]]
    ids, table, lens = _steps_of(case, seed)
    decode = case["phase"] == "decode"
    moe = m["kind"] == "moe"
    spec = q.Qwen3Spec(m["width"], m["layers"], m["heads"], m["kv"], HEAD, m["ff"], m["vocab"], rms_norm_eps=1e-5 if moe else 1e-6, qk_norm=not moe,
                       tie_word_embeddings=m["tied"], block_size=BLOCK, num_blocks=table.numel(), max_batch=case["rows"] if decode else 1,
                       max_seq_len=_bound(case) if decode else case["rows"] + 128, max_prefill_tokens=0 if decode else case["rows"],
                       num_experts=m.get("experts", 0), experts_per_tok=m.get("top", 0), act_dtype="f16" if m["kind"] == "exl3" else "bf16")
    model = q.QuantizedQwen3ForCausalLM(spec)
    emb, head, final = _qwen_ends(m, seed)
    model.load_tensor(q.T_EMBED, 0, emb)
    if head is not None:
        model.load_tensor(q.T_LM_HEAD, 0, head)
    model.load_tensor(q.T_FINAL_NORM, 0, final)
    for li in range(m["layers"]):
        gains, lin, router, experts = _qwen_layer(m, seed, li)
        for which, t in zip((q.T_INPUT_LN, q.T_POST_LN, q.T_Q_NORM, q.T_K_NORM), gains):
            model.load_tensor(which, li, t)
        for slot, w in enumerate(lin):
            if m["kind"] == "bf16":
                model.load_dense_linear(li, slot, w)
            elif m["kind"] == "exl3":
                model.load_exl3_linear(li, slot, *w)
            else:
                model.load_awq_linear(li, slot, *w)
        if moe:
            model.load_tensor(q.T_ROUTER, li, router)
            for e, ws in enumerate(experts):
                model.load_gptq_expert(li, e, *ws)
        if decode:
            for which, t in enumerate(_qwen_cache(m, seed, li, table.numel())):
                model.debug_kv(li, which, t, True)
    return _ready(case, model, ids, table, lens, _qwen_dtype(m))


def _prepare_gemma(case, seed):
    from vllm_rust_amd import gemma4 as q
    ids, table, lens = _steps_of(case, seed)
    decode = case["phase"] == "decode"
    spec = q.Gemma4Spec(GEMMA["width"], GEMMA["layers"], GEMMA["heads"], GEMMA["ff"], GEMMA["vocab"], sliding_window=1024, max_position=4096,
                        kv_cache_dtype=1, block_size=BLOCK, num_blocks=table.numel(), max_batch=case["rows"] if decode else 1,
                        max_seq_len=_bound(case) if decode else case["rows"] + 128, embed_ggml_type=11, final_logit_softcap=GEMMA["softcap"],
                        max_prefill_tokens=0 if decode else case["rows"])
    model = q.QuantizedGemma4ForCausalLM(spec)
    tab, final = _gemma_ends(seed)
    model.load_tensor(q.T_EMBED, 0, tab.reshape(-1))
    model.load_tensor(q.T_FINAL_NORM, 0, final)
    for li in range(GEMMA["layers"]):
        gains, lin = _gemma_layer(seed, li)
        for which, t in zip((q.T_INPUT_LN, q.T_POST_ATTN_LN, q.T_PRE_FFN_LN, q.T_POST_FFN_LN, q.T_Q_NORM, q.T_K_NORM, q.T_LAYER_SCALAR), gains):
            model.load_tensor(which, li, t)
        for slot, raw in lin.items():
            model.load_iq_linear(li, slot, GEMMA_TYPES[slot], raw.reshape(-1))
        if decode:
            for which, t in enumerate(_gemma_cache(seed, li, table.numel())):
                model.debug_kv(li, which, t.view(torch.uint8), True)
    return _ready(case, model, ids, table, lens, torch.bfloat16)


def _laro_spec():
    from vllm_rust_amd.larolorn import LarolornLayerSpec, LarolornSpec
    from vllm_rust_amd.rotation import RotationSpec
    H, D, RD, V, R, win = LARO["lat"]
    AH, AG, AD, chunk = LARO["att"]
    MH, MD = LARO["mem"]
    lat = LarolornLayerSpec(mixer="latent_attention", heads=H, dim=D, rot_dim=RD, vdim=V, kv_rank=R, scale=1.0 / math.sqrt(D + RD), mask=win,
                            rot=RotationSpec(RD, 1e5), mlp="dense", ff=LARO["ff"], limit=LARO["limit"])
    two = LarolornLayerSpec(mixer="parallel", heads=AH, kv_heads=AG, dim=AD, vdim=AD, scale=1.0 / math.sqrt(AD), mask=chunk, rot=RotationSpec(AD, 1e5),
                            r_heads=MH, r_dim=MD, r_vdim=MD, decay=tuple(_laro_decay()), mlp="dense", ff=LARO["ff"], limit=LARO["limit"])
    return LarolornSpec(vocab=LARO["vocab"], width=LARO["width"], layers=[lat, two, lat, two], norm_eps=LARO["eps"], residual_mult=LARO["mult"])


def _packed(table, parts):
    """Arguments of one packed step: parts = [(sequence, token ids, first position)]."""
    tok = torch.cat([t for _, t, _ in parts])
    pos = torch.cat([torch.arange(p, p + t.numel(), dtype=torch.int32, device="cuda") for _, t, p in parts])
    sid = torch.cat([torch.full((t.numel(),), i, dtype=torch.int32, device="cuda") for i, (_, t, _) in enumerate(parts)])
    rows = table[torch.as_tensor([s for s, _, _ in parts], device="cuda")].contiguous()
    slots = (rows[sid.long(), (pos // BLOCK).long()] * BLOCK + pos % BLOCK).to(torch.int32).contiguous()
    starts = [0]
    for _, t, _ in parts:
        starts.append(starts[-1] + t.numel())
    return (tok, torch.zeros_like(tok), pos, slots, sid, rows, _i32([s - 1 for s in starts[1:]])), {"seq_starts": _i32(starts), "state_slots": _i32([s for s, _, _ in parts])}


def _prepare_laro(case, seed):
    from vllm_rust_amd.larolorn import LarolornForCausalLM
    ids, step_ids, table, lens = _laro_tokens(case, seed)
    model = LarolornForCausalLM(_laro_spec(), "bfloat16", block_size=BLOCK, num_blocks=table.numel(), max_tokens=max(case["rows"], max(lens)), max_seqs=len(lens))
    model.load_state(_laro_weights(seed))
    torch.cuda.synchronize()
    if case["phase"] == "prompt":
        args, kw = _packed(table, [(i, t, 0) for i, t in enumerate(ids)])
        return {"case": case, "model": model, "args": args, "kw": kw}
    args, kw = _packed(table, [(i, step_ids[i:i + 1], n) for i, n in enumerate(lens)])
    got = {}

    def step():
        got["logits"], got["out"], _ = model.forward(*args, want_greedy=True, **kw)

    def prompts():
        for i, t in enumerate(ids):
            a, k = _packed(table, [(i, t, 0)])
            model.forward(*a, want_logits=False, want_greedy=True, **k)
    return {"case": case, "graph": _captured(step, prompts), "keep": (args, kw), "model": model, **got}


def run(state):
    case = state["case"]
    if case["phase"] == "decode":
        state["graph"].replay()
        return {"ids": state["out"], "logits": state["logits"]}
    if case["model"] == "larolorn_2k":
        logits, ids, _ = state["model"].forward(*state["args"], want_greedy=True, **state["kw"])
        return {"ids": ids, "logits": logits}
    state["model"].prefill(state["ids"], 0, state["table"], out_id=state["out"], logits_last=state["logits"])
    return {"ids": state["out"], "logits": state["logits"]}


# ------------------------------------------------------------------------------------------------ what a pass cannot do without
def _linear_bytes(kind, K, N):
    return {"bf16": 2.0 * K * N, "exl3": K * N / 2 + 2 * (K + N), "awq": K * N / 2 + K / GROUP * N * 2.5, "moe": K * N / 2 + K / GROUP * N * 2.5}[kind]


def work(case):
    decode = case["phase"] == "decode"
    n = case["rows"]
    if case["model"] == "larolorn_2k":
        lens = _lengths(case) if decode else _prompt_lengths(case)
    else:
        lens = _lengths(case) if decode else [n]
    keys = sum(c + 1 for c in lens) if decode else sum(c * (c + 1) / 2 for c in lens)        # (query, key) pairs
    rows_kept = sum(c + 1 for c in lens) if decode else sum(lens)                            # cache rows read or written
    outs = n if decode else (3 if case["model"] == "larolorn_2k" else 1)                     # logits rows
    if case["model"] in QWEN:
        m = QWEN[case["model"]]
        L, W = m["layers"], m["width"]
        params = sum(K * N for K, N in _qwen_shapes(m))
        by = L * sum(_linear_bytes(m["kind"], K, N) for K, N in _qwen_shapes(m))
        if m["kind"] == "moe":
            hit = m["experts"] * (1 - (1 - m["top"] / m["experts"]) ** n)                    # expected number of experts in use
            by += L * hit * 3 * _linear_bytes("moe", W, m["ff"])
            params += m["top"] * 3 * W * m["ff"]
        by += m["vocab"] * W * 2 + outs * m["vocab"] * 2 + L * rows_kept * 2 * m["kv"] * HEAD * 2
        fl = 2.0 * n * L * params + 2.0 * outs * m["vocab"] * W + L * 4.0 * keys * m["heads"] * HEAD
    elif case["model"] == "gemma4_12b_iq3":
        by = GEMMA["vocab"] * GEMMA["width"] / 256 * 110 + outs * GEMMA["vocab"] * 2
        fl = 2.0 * outs * GEMMA["vocab"] * GEMMA["width"]
        for li in range(GEMMA["layers"]):
            hd, kv = _gemma_geom(li)[:2]
            for slot, (K, N) in _gemma_shapes(li).items():
                by += N * K / 256 * IQ_SIZE[GEMMA_TYPES[slot]]
                fl += 2.0 * n * K * N
            by += rows_kept * 2 * kv * hd
            fl += 4.0 * keys * GEMMA["heads"] * hd
    else:
        W, F = LARO["width"], LARO["ff"]
        H, D, RD, V, R, _ = LARO["lat"]
        AH, AG, AD, _ = LARO["att"]
        MH, MD = LARO["mem"]
        lat = W * (H * (D + RD) + R + RD + H) + H * D * R + H * V * R + H * V * W
        two = W * (AH * AD + 2 * AG * AD + 4 * MH * MD) + AH * AD * W + MH * MD * W
        params = 2 * (lat + two) + 4 * 3 * W * F
        by = 2.0 * (params + LARO["vocab"] * W) + outs * LARO["vocab"] * 4 + 2 * 2 * rows_kept * (R + RD + 2 * AG * AD) + 2 * 2 * len(lens) * MH * MD * MD * 4
        # latent attention by whichever form needs fewer operations: expanded keys and values (prompts), latent space (a decode step)
        per_pair = min(2.0 * H * (D + RD + V), 2.0 * H * (2 * R + RD))
        fl = 2.0 * n * params + 2.0 * outs * LARO["vocab"] * W + 2 * keys * (per_pair + 4.0 * AH * AD) + 2 * n * 4.0 * MH * MD * MD
    return {"bytes": by, "flops": fl}


# Relative error (2-norm) of the logits: two to four times what the path shows against 64-bit arithmetic, which is what rounding every
# operator's result to the model's 16-bit type leaves behind so many layers (bf16: 0.9 % for the 8B slice, 1.5 % for the 28 layers of
# the 0.6B, up to 2 % for Gemma, whose cached rows are FP8 as well, 0.16 % for Mixtral's four layers; fp16: 0.17 %; Larolorn, whose
# stream is f32: 0.35 %).
_REL = {"qwen3_0_6b_bf16": 3e-2, "qwen3_8b_awq": 3e-2, "qwen3_8b_exl3": 7e-3, "mixtral_8x7b_gptq": 7e-3, "gemma4_12b_iq3": 3e-2, "larolorn_2k": 1.4e-2}


def tolerance(case):
    return {"rel": _REL[case["model"]], "max": 10 * _REL[case["model"]], "differ": 0.0}


# ------------------------------------------------------------------------------------------------ the same in 64 bits
F64 = torch.float64


def _rms(x, w, eps):
    x = x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)
    return x if w is None else x * w.to(F64)


def _turned(x, pos, dims, of, base, dtype):
    """x [T, heads, d]: coordinate i < dims / 2 turns with i + dims / 2 (in the first `dims`), cosines and sines in the model's type."""
    step = 1.0 / torch.pow(torch.tensor(base, dtype=F64, device="cuda"), torch.arange(0, dims, 2, dtype=F64, device="cuda") / of)
    a = pos.to(F64)[:, None] * step[None, :]
    c, s = torch.cos(a).to(dtype).to(F64)[:, None], torch.sin(a).to(dtype).to(F64)[:, None]
    u, v = x[..., :dims // 2], x[..., dims // 2:dims]
    return torch.cat([u * c - v * s, v * c + u * s, x[..., dims:]], -1)


def _attend(q, k, v, scale, window=0, sink=None):
    """q [n, H, D] are the last n rows of a sequence whose keys k [T, G, D] and values v [T, G, V] are whole -> [n, H * V]."""
    n, H, T, G = q.shape[0], q.shape[1], k.shape[0], k.shape[1]
    at = torch.arange(T - n, T, device="cuda")[:, None]
    seen = torch.arange(T, device="cuda")[None, :] <= at
    if window:
        seen &= torch.arange(T, device="cuda")[None, :] > at - window
    out = []
    for h in range(H):
        s = (q[:, h] @ k[:, h // (H // G)].T) * scale
        s = s.masked_fill(~seen, -math.inf)
        if sink is not None:
            s = torch.cat([s, sink[h].to(F64).expand(n, 1)], 1)
        out.append(torch.softmax(s, -1)[:, :T] @ v[:, h // (H // G)])
    return torch.stack(out, 1).reshape(n, -1)


def _nibbles(words, order):
    sh = torch.tensor(order, dtype=torch.int32, device="cuda")
    return (words.unsqueeze(-1) >> sh) & 15


_AWQ = [0, 16, 4, 20, 8, 24, 12, 28]      # shift of the i-th of the eight columns that share a word
_SEQ = [0, 4, 8, 12, 16, 20, 24, 28]


def _bf16_scales(sc):
    return sc.to(torch.bfloat16).to(F64)     # int4 linears of a bf16 model hold their scales in bf16


def _awq_dense(qw, qz, sc):
    K, N = qw.shape[0], qw.shape[1] * 8
    q = _nibbles(qw, _AWQ).reshape(K // GROUP, GROUP, N) - _nibbles(qz, _AWQ).reshape(K // GROUP, 1, N)
    return (q.to(F64) * _bf16_scales(sc)[:, None]).reshape(K, N)


def _gptq_dense(qw, sc):
    K, N = qw.shape[0] * 8, qw.shape[1]
    q = _nibbles(qw, _SEQ).permute(0, 2, 1).reshape(K // GROUP, GROUP, N) - 8
    return (q.to(F64) * _bf16_scales(sc)[:, None]).reshape(K, N)


def _exl3_dense(tr):
    """Trellis words [K/16, N/16, 64] -> [K, N]: weight t of a tile is a 16-bit window of the tile's cyclic bit stream, hashed."""
    tk, tn, _ = tr.shape
    half = tr.to(torch.int64) & 0xFFFF
    w = half[..., 0::2] | (half[..., 1::2] << 16)                                    # 32 words, stream bit i is bit 31 - i % 32 of word i / 32
    t = torch.arange(256, device="cuda")
    b0 = ((t + 257) * 4 - 16) % 1024
    lo, hi = b0 // 32, (b0 // 32 + 1) % 32
    s = b0 % 32                                                                      # windows past bit 16 run into the next word
    x = torch.where(s <= 16, w[..., lo] >> (16 - s).clamp(min=0), (w[..., lo] << (s - 16).clamp(min=0)) | (w[..., hi] >> (48 - s))) & 0xFFFF
    x = (x * 89226354 + 64248484) & 0xFFFFFFFF
    x = (x & 0x8FFF8FFF) ^ 0x3B603B60
    val = (x & 0xFFFF).to(torch.int32).to(torch.int16).view(torch.float16) + (x >> 16).to(torch.int32).to(torch.int16).view(torch.float16)
    lane, i = t >> 3, t & 7
    row = 2 * (lane & 3) + (i & 1) + 8 * ((i >> 1) & 1)
    col = 2 * (lane >> 3) + ((lane >> 2) & 1) + 8 * (i >> 2)
    out = torch.empty(tk, tn, 256, dtype=F64, device="cuda")
    out[..., row * 16 + col] = val.to(F64)
    return out.reshape(tk, tn, 16, 16).permute(0, 2, 1, 3).reshape(tk * 16, tn * 16)


def _hadamard(x):
    y = x.reshape(*x.shape[:-1], -1, 128)
    h = torch.ones(1, 1, dtype=F64, device="cuda")
    for _ in range(7):
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return (y @ h / math.sqrt(128.0)).reshape(x.shape)


def _times(kind, x, w):
    if kind == "bf16":
        return x @ w.to(F64).T
    if kind == "exl3":
        return _hadamard(_hadamard(x * w[1].to(F64)) @ _exl3_dense(w[0])) * w[2].to(F64)
    return x @ _awq_dense(*w)


def _exact_qwen(case, seed):
    m = QWEN[case["model"]]
    ids, table, lens = _steps_of(case, seed)
    decode, dt = case["phase"] == "decode", _qwen_dtype(m)
    eps = 1e-5 if m["kind"] == "moe" else 1e-6
    pos = _i32(lens) if decode else torch.arange(case["rows"], device="cuda")
    emb, head, final = _qwen_ends(m, seed)
    x = emb[ids.long()].to(F64)
    n = x.shape[0]
    for li in range(m["layers"]):
        (g1, g2, gq, gk), lin, router, experts = _qwen_layer(m, seed, li)
        h = _rms(x, g1, eps)
        q, k, v = (_times(m["kind"], h, lin[s]).reshape(n, -1, HEAD) for s in range(3))
        if m["kind"] != "moe":
            q, k = _rms(q, gq, eps), _rms(k, gk, eps)
        q, k = (_turned(t, pos, HEAD, HEAD, 1e6, dt) for t in (q, k))
        if decode:
            kc, vc = _qwen_cache(m, seed, li, table.numel())
            att = []
            for b, c in enumerate(lens):
                rows = (table[b].long()[:, None] * BLOCK + torch.arange(BLOCK, device="cuda")).reshape(-1)[:c]
                past = [t.reshape(-1, m["kv"], HEAD)[rows].to(F64) for t in (kc, vc)]
                att.append(_attend(q[b:b + 1], torch.cat([past[0], k[b:b + 1]]), torch.cat([past[1], v[b:b + 1]]), HEAD ** -0.5))
            a = torch.cat(att)
        else:
            a = _attend(q, k, v, HEAD ** -0.5)
        x = x + _times(m["kind"], a, lin[3])
        h = _rms(x, g2, eps)
        if m["kind"] != "moe":
            x = x + _times(m["kind"], torch.nn.functional.silu(_times(m["kind"], h, lin[4])) * _times(m["kind"], h, lin[5]), lin[6])
            continue
        p, who = torch.softmax(h @ router.to(F64).T, -1).topk(m["top"], -1)
        p = p / p.sum(-1, keepdim=True)
        y = torch.zeros_like(x)
        for e, (w1, w3, w2) in enumerate(experts):
            r, j = (who == e).nonzero(as_tuple=True)
            if r.numel():
                hid = torch.nn.functional.silu(h[r] @ _gptq_dense(*w1)) * (h[r] @ _gptq_dense(*w3))
                y[r] += p[r, j][:, None] * (hid @ _gptq_dense(*w2))
        x = x + y
    x = x if decode else x[-1:]
    logits = _rms(x, final, eps) @ (emb if head is None else head).to(F64).T
    return {"ids": None, "logits": logits if decode else logits[0]}


def _iq_tables():
    """Codebooks of the GGUF I-quant formats, from the data file the repository keeps beside its sources."""
    here = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "vllm-rust_amd", "csrc", "data", "iq_tables.bin")
    with open(here, "rb") as f:
        data = f.read()
    at, out = 0, {}
    for name, fmt, count in (("mask", "B", 8), ("signs", "B", 128), ("iq2xs", "8B", 512), ("iq2s", "8B", 1024), ("iq3xxs", "4B", 256), ("iq3s", "4B", 512)):
        size = struct.calcsize(fmt) * count
        out[name] = torch.frombuffer(bytearray(data[at:at + size]), dtype=torch.uint8).reshape(count, -1).to("cuda").to(torch.int64)
        at += size
    return out


def _iq_dense(kind, raw, N, K, tab):
    """Raw super-blocks [N * K / 256, bytes] -> [N, K] in 64 bits."""
    nb = raw.shape[0]
    b = raw.to(torch.int64)
    d = raw[:, :2].contiguous().view(torch.float16).to(F64)[:, 0]
    eight = torch.arange(8, device="cuda")
    if kind == 18:                                                     # IQ3_XXS: 64 index bytes, 8 words of 4 x 7 sign bits and a scale
        mag = tab["iq3xxs"][b[:, 2:66]].reshape(nb, 8, 32)
        aux = b[:, 66:98].reshape(nb, 8, 4)
        aux = aux[..., 0] | (aux[..., 1] << 8) | (aux[..., 2] << 16) | (aux[..., 3] << 24)
        sg = tab["signs"][:, 0][(aux.unsqueeze(-1) >> torch.tensor([0, 7, 14, 21], device="cuda")) & 127]      # [nb, 8, 4]
        scale = (0.5 + (aux >> 28).to(F64)).unsqueeze(-1) * 0.5
    elif kind == 22:                                                   # IQ2_S: 32 index bytes, 32 sign bytes, 8 high-bit bytes, 8 scale bytes
        qh = b[:, 66:74]
        idx = b[:, 2:34].reshape(nb, 8, 4) | (((qh.unsqueeze(-1) >> torch.tensor([0, 2, 4, 6], device="cuda")) & 3) << 8)
        mag = tab["iq2s"][idx].reshape(nb, 8, 32)
        sg = b[:, 34:66].reshape(nb, 8, 4)
        sc = torch.stack([b[:, 74:82] & 15, b[:, 74:82] >> 4], -1).to(F64)                                     # two halves
        scale = ((0.5 + sc) * 0.25).repeat_interleave(16, -1)
    else:                                                              # IQ3_S: 64 index bytes, 8 high-bit bytes, 32 sign bytes, 4 scale bytes
        qh = b[:, 66:74]
        idx = b[:, 2:66].reshape(nb, 8, 8) | (((qh.unsqueeze(-1) >> eight) & 1) << 8)
        mag = tab["iq3s"][idx].reshape(nb, 8, 32)
        sg = b[:, 74:106].reshape(nb, 8, 4)
        sc = torch.stack([b[:, 106:110] & 15, b[:, 106:110] >> 4], -1).reshape(nb, 8)
        scale = (1 + 2 * sc).to(F64).unsqueeze(-1)
    neg = ((sg.unsqueeze(-1) >> eight) & 1).reshape(nb, 8, 32)
    w = torch.where(neg == 1, -mag, mag).to(F64) * scale * d[:, None, None]
    return w.reshape(N, K)


def _q3k_dense(raw):
    """Q3_K super-blocks [n, 110] -> [n, 256]."""
    n = raw.shape[0]
    b = raw.to(torch.int64)
    d = raw[:, 108:110].contiguous().view(torch.float16).to(F64)
    lo = torch.cat([b[:, 96:104] & 15, b[:, 96:104] >> 4], 1)
    hi = torch.stack([(b[:, 104:108] >> s) & 3 for s in (0, 2, 4, 6)], 1).reshape(n, 16)
    scale = (lo | (hi << 4)) - 32
    q = torch.stack([(b[:, 32:96].reshape(n, 2, 32) >> s) & 3 for s in (0, 2, 4, 6)], 2)                        # [n, 2, 4, 32]
    h = torch.stack([(b[:, :32] >> s) & 1 for s in range(8)], 1).reshape(n, 2, 4, 32)
    return (d * scale.repeat_interleave(16, 1)) * (q - 4 * (1 - h)).reshape(n, 256).to(F64)


def _exact_gemma(case, seed):
    ids, table, lens = _steps_of(case, seed)
    decode, eps, W = case["phase"] == "decode", GEMMA["eps"], GEMMA["width"]
    pos = _i32(lens) if decode else torch.arange(case["rows"], device="cuda")
    tab, final = _gemma_ends(seed)
    per = W // 256
    books = _iq_tables()
    x = _q3k_dense(tab.reshape(-1, per, 110)[ids.long()].reshape(-1, 110)).reshape(-1, W) * float(torch.tensor(math.sqrt(W)).to(torch.bfloat16))
    n = x.shape[0]
    stored = lambda t: t.to(torch.float32).to(torch.float8_e4m3fn).to(F64)   # noqa: E731  (rows of the FP8 cache)
    for li in range(GEMMA["layers"]):
        (g1, g2, g3, g4, gq, gk, scalar), lin = _gemma_layer(seed, li)
        hd, kv, rot, window = _gemma_geom(li)
        w = {s: _iq_dense(GEMMA_TYPES[s], lin[s], N, K, books) for s, (K, N) in _gemma_shapes(li).items()}
        h = _rms(x, g1, eps)
        q = _rms((h @ w[0].T).reshape(n, -1, hd), gq, eps)
        kp = (h @ w[1].T).reshape(n, kv, hd)
        v = _rms((h @ w[2].T).reshape(n, kv, hd), None, eps)
        base = 1e4 if window else 1e6
        q, k = (_turned(t, pos, rot, hd, base, torch.bfloat16) for t in (q, _rms(kp, gk, eps)))
        k, v = stored(k), stored(v)
        if decode:
            kc, vc = _gemma_cache(seed, li, table.numel())
            att = []
            for b, c in enumerate(lens):
                rows = (table[b].long()[:, None] * BLOCK + torch.arange(BLOCK, device="cuda")).reshape(-1)[:c]
                past = [t.view(torch.uint8).reshape(-1, kv, hd)[rows].view(torch.float8_e4m3fn).to(F64) for t in (kc, vc)]
                att.append(_attend(q[b:b + 1], torch.cat([past[0], k[b:b + 1]]), torch.cat([past[1], v[b:b + 1]]), 1.0, window))
            a = torch.cat(att)
        else:
            a = _attend(q, k, v, 1.0, window)
        x = x + _rms(a @ w[3].T, g2, eps)
        h = _rms(x, g3, eps)
        x = x + _rms((torch.nn.functional.gelu(h @ w[4].T) * (h @ w[5].T)) @ w[6].T, g4, eps)
        x = x * scalar.to(F64)
        del w
    x = _rms(x if decode else x[-1:], final, eps)
    logits = torch.cat([x @ _q3k_dense(part.reshape(-1, 110)).reshape(-1, W).T for part in tab.reshape(-1, per, 110).split(8192)], 1)
    logits = GEMMA["softcap"] * torch.tanh(logits / GEMMA["softcap"])
    return {"ids": None, "logits": logits if decode else logits[0]}


def _neighbours(x, pos, base):
    """x [T, heads, d]: coordinate 2i turns with 2i + 1."""
    d = x.shape[-1]
    a = pos.to(F64)[:, None] * (float(base) ** (-torch.arange(0, d, 2, dtype=F64, device="cuda") / d))[None, :]
    c, s = torch.cos(a)[:, None], torch.sin(a)[:, None]
    u, v = x[..., 0::2], x[..., 1::2]
    return torch.stack([u * c - v * s, v * c + u * s], -1).reshape(x.shape)


def _laro_sequence(w, ids):
    """Logits of the last token of one sequence from its first token."""
    eps, T = LARO["eps"], ids.numel()
    H, D, RD, V, R, win = LARO["lat"]
    AH, AG, AD, chunk = LARO["att"]
    MH, MD = LARO["mem"]
    assert T <= chunk
    pos = torch.arange(T, device="cuda")
    x = w["embed"][ids.long()]
    gap = (pos[:, None] - pos[None, :]).to(F64)
    for i in range(4):
        p = f"l{i}.mix."
        if i % 2 == 0:
            q = (x @ w[p + "q"].T).reshape(T, H, D + RD)
            q = torch.cat([q[..., :D], _neighbours(q[..., D:], pos, 1e5)], -1)
            y = x @ w[p + "dkv"].T
            c = _rms(y[:, :R], w[p + "dkv.norm"], eps)
            kr = _neighbours(y[:, None, R:], pos, 1e5).expand(T, H, RD)
            k = torch.cat([(c @ w[p + "uk"].T).reshape(T, H, D), kr], -1)
            o = _attend(q, k, (c @ w[p + "uv"].T).reshape(T, H, V), 1.0 / math.sqrt(D + RD), win).reshape(T, H, V)
            mix = (o * torch.sigmoid(x @ w[p + "g"].T)[..., None]).reshape(T, -1) @ w[p + "o"].T
        else:
            l, r = p + "left.", p + "right."
            q, k, v = (x @ w[l + n].T + w[l + n + ".b"] for n in "qkv")
            q, k = _rms(q, w[l + "q.norm"], eps).reshape(T, AH, AD), _rms(k, w[l + "k.norm"], eps).reshape(T, AG, AD)
            q, k = (_turned(t, pos, AD, AD, 1e5, F64) for t in (q, k))
            left = _attend(q, k, v.reshape(T, AG, AD), 1.0 / math.sqrt(AD), 0, w[l + "sink"]) @ w[l + "o"].T + w[l + "o.b"]
            mq, mk, mv = (torch.nn.functional.silu(x @ w[r + n].T).reshape(T, MH, MD) for n in "qkv")
            out = []
            for hd, decay in enumerate(_laro_decay()):
                f = torch.tensor(decay, dtype=torch.float32).to(F64).item()
                keep = torch.where(gap >= 0, f ** gap.clamp(min=0), torch.zeros((), dtype=F64, device="cuda"))
                out.append(((mq[:, hd] @ mk[:, hd].T) * keep) @ mv[:, hd])
            o = _rms(torch.stack(out, 1).reshape(T, -1), w[r + "norm"], eps) * torch.sigmoid(x @ w[r + "g"].T)
            mix = 0.5 * (_rms(left, w[l + "out"], eps) + _rms(o @ w[r + "o"].T, w[r + "out"], eps))
        x = x + LARO["mult"] * _rms(mix, w[f"l{i}.norm1"], eps)
        g, u = (x @ w[f"l{i}.mlp.gate"].T).clamp(max=LARO["limit"]), (x @ w[f"l{i}.mlp.up"].T).clamp(-LARO["limit"], LARO["limit"])
        x = x + LARO["mult"] * _rms((g * torch.sigmoid(1.702 * g) * (u + 1.0)) @ w[f"l{i}.mlp.down"].T, w[f"l{i}.norm2"], eps)
    return _rms(x[-1:], w["final.norm"], eps) @ w["head"].T


def _exact_laro(case, seed):
    ids, step, _, lens = _laro_tokens(case, seed)
    w = {k: v.to(F64) for k, v in _laro_weights(seed).items()}
    if case["phase"] == "decode":
        ids = [torch.cat([t, step[i:i + 1]]) for i, t in enumerate(ids)]
    return {"ids": None, "logits": torch.cat([_laro_sequence(w, t) for t in ids])}


def exact(case, seed):
    if case["model"] in QWEN:
        return _exact_qwen(case, seed)
    return _exact_gemma(case, seed) if case["model"] == "gemma4_12b_iq3" else _exact_laro(case, seed)
