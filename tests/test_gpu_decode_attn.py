"""Decode attention with both products on the matrix cores, seen through a one-layer executor whose o projection, MLP and head are
the identity, nothing and the identity: the logits are the final norm of token embedding + attention output.  Reference: float64 torch on
the same caches.  Pages that hold no token of the sequence, and rows behind a sequence's end, are NaN."""
import math

import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    import torch
    import vllm_rust_amd as vmx
    vmx.init(0)
    return vmx, torch


def _setup(torch, heads, kv, hd, fp8, block, lens, seed, bound):
    from vllm_rust_amd import qwen3 as q
    W = heads * hd
    n, width = len(lens), (bound + block - 1) // block
    spec = q.Qwen3Spec(W, 1, heads, kv, hd, 128, W, qk_norm=True, block_size=block, num_blocks=n * width, max_batch=n, max_seq_len=bound,
                       max_position=bound + 1, kv_cache_dtype=1 if fp8 else 0)
    m = q.QuantizedQwen3ForCausalLM(spec)
    g = torch.Generator(device="cuda").manual_seed(seed)
    r = lambda *s: torch.randn(s, device="cuda", generator=g)   # noqa: E731
    emb = (r(W, W) * 0.02).to(torch.bfloat16)
    ones = torch.ones(W, device="cuda", dtype=torch.bfloat16)
    w = {s: (r(o, W) / math.sqrt(W)).to(torch.bfloat16) for s, o in ((q.L_Q, W), (q.L_K, kv * hd), (q.L_V, kv * hd))}
    w[q.L_O] = torch.eye(W, device="cuda", dtype=torch.bfloat16)
    w[q.L_GATE] = w[q.L_UP] = torch.zeros(128, W, device="cuda", dtype=torch.bfloat16)
    w[q.L_DOWN] = torch.zeros(W, 128, device="cuda", dtype=torch.bfloat16)
    gq, gk = ((1 + 0.1 * r(hd)).to(torch.bfloat16) for _ in range(2))
    for which, t in ((q.T_EMBED, emb), (q.T_LM_HEAD, torch.eye(W, device="cuda", dtype=torch.bfloat16)), (q.T_FINAL_NORM, ones), (q.T_INPUT_LN, ones),
                     (q.T_POST_LN, ones), (q.T_Q_NORM, gq), (q.T_K_NORM, gk)):
        m.load_tensor(which, 0, t)
    for s, t in w.items():
        m.load_dense_linear(0, s, t)
    table = torch.randperm(n * width, device="cuda", generator=g).to(torch.int32).reshape(n, width).contiguous()
    store = torch.float8_e4m3fn if fp8 else torch.bfloat16
    past = []
    caches = [torch.full((n * width * block, kv, hd), float("nan"), device="cuda").to(store) for _ in range(2)]
    for b, c in enumerate(lens):
        rows = (table[b].long()[:, None] * block + torch.arange(block, device="cuda")).reshape(-1)[:c]
        kvs = [r(c, kv, hd).to(store) for _ in range(2)]
        for cache, t in zip(caches, kvs):
            cache.view(torch.uint8 if fp8 else torch.int16)[rows] = t.view(torch.uint8 if fp8 else torch.int16)
        past.append(kvs)
    return q, m, emb, w, (gq, gk), table, caches, past, g


def _run(torch, heads, kv, hd, fp8, block, lens, bound, seed=1):
    q, m, emb, w, gains, table, caches, past, g = _setup(torch, heads, kv, hd, fp8, block, lens, seed, bound)
    W, n = heads * hd, len(lens)
    for which, t in enumerate(caches):
        m.debug_kv(0, which, t.view(torch.uint8) if fp8 else t, True)
    ids = torch.randint(0, W, (n,), dtype=torch.int32, device="cuda", generator=g)
    pos = torch.tensor(lens, dtype=torch.int32, device="cuda")
    slots = (table[torch.arange(n, device="cuda"), (pos // block).long()] * block + pos % block).to(torch.int32).contiguous()
    logits = torch.empty(n, W, dtype=torch.bfloat16, device="cuda")
    m.forward_decode_batch(ids, pos, slots, table, (pos + 1).contiguous(), max_seq_len=bound, logits=logits)
    torch.cuda.synchronize()
    f = torch.float64
    rms = lambda t: t / torch.sqrt((t * t).mean(-1, keepdim=True) + 1e-6)   # noqa: E731
    x = emb[ids.long()].to(f)
    h = rms(x)
    a = torch.arange(0, hd, 2, device="cuda", dtype=f) / hd
    ang = pos.to(f)[:, None] / (1e6 ** a)[None]
    c, s = (t.to(torch.bfloat16).to(f)[:, None] for t in (torch.cos(ang), torch.sin(ang)))

    def head(t, gain):
        t = rms(t) * gain.to(f)
        u, v = t[..., :hd // 2], t[..., hd // 2:]
        return torch.cat([u * c - v * s, v * c + u * s], -1)
    qh = head((h @ w[q.L_Q].to(f).T).reshape(n, heads, hd), gains[0])
    kh = head((h @ w[q.L_K].to(f).T).reshape(n, kv, hd), gains[1])
    vh = (h @ w[q.L_V].to(f).T).reshape(n, kv, hd)
    if fp8:
        kh, vh = (t.float().to(torch.float8_e4m3fn).to(f) for t in (kh, vh))
    out = []
    for b in range(n):
        K, V = (torch.cat([p.to(f), t[b:b + 1]]) for p, t in zip(past[b], (kh, vh)))
        K, V = K.repeat_interleave(heads // kv, 1), V.repeat_interleave(heads // kv, 1)
        p = torch.softmax(torch.einsum("hd,thd->ht", qh[b], K) / math.sqrt(hd), -1)
        out.append(torch.einsum("ht,thd->hd", p, V).reshape(-1))
    return m, logits.to(f), x + torch.stack(out), rms


CASES = [  # heads, kv heads, head width, fp8, block, lengths before the step, bound
    (8, 4, 128, False, 16, [128], 160), (4, 4, 128, False, 16, [1], 160), (8, 2, 128, False, 16, [0], 64), (8, 2, 128, False, 16, [15, 16, 17], 160),
    (8, 1, 128, False, 16, [300], 400), (16, 4, 64, False, 16, [33, 200], 300), (8, 2, 128, False, 24, [95, 96, 250], 300), (8, 2, 128, True, 16, [47, 130], 200),
    (8, 2, 128, False, 16, [600, 31, 511, 512, 900], 1100), (8, 2, 128, False, 5, [701] + [37 * i for i in range(15)], 1024), (8, 2, 128, True, 16, [2000, 40], 2100),
    (4, 2, 128, False, 16, [2500], 3000),
]


@pytest.mark.parametrize("heads,kv,hd,fp8,block,lens,bound", CASES)
def test_decode_attention_matches_float64(gpu, heads, kv, hd, fp8, block, lens, bound):
    """q, k, v, the cached row and the output are rounded to bf16 (k and v of an FP8 cache to 4 bits): a score moves by at most 2^-8 sqrt(hd)
    / sqrt(3) of a standard deviation ~ 2.5 %, its share of the output by as much of 1 / sqrt(keys); 1.5 % in all (FP8 6 %: the new row
    alone can carry a rounding of 2^-4)."""
    vmx, torch = gpu
    m, got, h, rms = _run(torch, heads, kv, hd, fp8, block, lens, bound)
    want = rms(h)
    assert torch.isfinite(got).all()
    for b in range(len(lens)):
        rel = ((got[b] - want[b]).norm() / want[b].norm()).item()
        assert rel <= (6e-2 if fp8 else 1.5e-2), (b, lens[b], rel)
    m.close()


# Eight query heads a KV head
EIGHT = [(8, 1, 128, False, 16, [600, 31, 1000], 1100), (8, 1, 128, True, 16, [600, 31, 1000], 1100), (16, 2, 64, False, 5, [701, 15, 511], 1024),
         (16, 2, 64, True, 16, [701, 15, 511], 1024), (16, 2, 128, False, 1, [150, 950], 1000)]
# 16 rows over two KV heads have 64 waves each: 4900 tokens on pages of one are 76 pages a wave, more than its lanes hold, so that its lookups go to memory
LONG = [4900, 4300] + [100 + 311 * i for i in range(14)]
PAGES = [(4, 2, 64, False, 1, LONG, 5000), (4, 2, 64, True, 1, LONG, 5000), (4, 2, 128, False, 1, LONG, 5000), (16, 2, 64, False, 1, LONG, 5000), (16, 2, 128, True, 1, LONG, 5000)]


@pytest.mark.parametrize("heads,kv,hd,fp8,block,lens,bound", EIGHT + PAGES)
def test_eight_heads_and_long_walks_match_float64(gpu, heads, kv, hd, fp8, block, lens, bound):
    """As above, with its bounds."""
    test_decode_attention_matches_float64(gpu, heads, kv, hd, fp8, block, lens, bound)
