"""Latent attention over rows of 512 + 64 values (the form with constant sizes and rows requested a tile ahead) at the edges of its
64-key tiles: prompts with more row tiles than compute units (not partitioned) and decode steps (partitioned)."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    import torch
    import vllm_rust_amd as vmx
    vmx.init(0)
    return vmx, torch


# (contexts per sequence, new tokens per sequence, heads, window)
@pytest.mark.parametrize("contexts,new,heads,window", [
    ([300], 300, 16, 0), ([321], 257, 16, 70), ([64, 63, 65, 1], 1, 16, 0), ([128, 129, 700], 1, 20, 0), ([200, 513], 3, 3, 64),
    ([530, 90], 600, 8, 0),
])
def test_whole_rows(gpu, contexts, new, heads, window):
    """Against float64 on the operands the kernel multiplies (bf16 rows, queries rounded to bf16).  A score is an f32 sum of 576 products
    (off by at most d = 576 2^-24 scale sum |q k|), a weight is then off by a factor exp(2 d), its two bf16 halves by 2^-16, and the sums
    of up to 1024 weighted rows by 1024 2^-24 of sum p |c| <= max |c|."""
    vmx, torch = gpu
    from vllm_rust_amd._lib import check, lib
    R, RD, bs, scale = 512, 64, 16, 0.06
    g = torch.Generator(device="cuda").manual_seed(sum(contexts) + heads)
    n = len(contexts)
    mb = (max(contexts) + bs - 1) // bs
    bt = torch.randperm(n * mb, device="cuda", generator=g).to(torch.int32).view(n, mb)
    cache = torch.randn((n * mb * bs, R + RD), device="cuda", generator=g).to(torch.bfloat16)
    sid, pos = [], []
    for b, c in enumerate(contexts):
        k = min(new, c)
        sid += [b] * k
        pos += list(range(c - k, c))
    T = len(pos)
    qa = torch.randn((T, heads, R), device="cuda", generator=g).to(torch.bfloat16).float()
    qr = torch.randn((T, heads, RD), device="cuda", generator=g).to(torch.bfloat16).float()
    ts, tp = (torch.tensor(v, device="cuda", dtype=torch.int32) for v in (sid, pos))
    out = torch.full((T, heads, R), float("nan"), device="cuda")
    need = lib.vmx_latent_attention_workspace_bytes(T, heads, R, window, mb, bs)
    ws = torch.empty(max(need, 16), dtype=torch.uint8, device="cuda")
    check(lib.vmx_latent_attention(out.data_ptr(), qa.data_ptr(), qr.data_ptr(), cache.data_ptr(), 1, bt.data_ptr(), mb, ts.data_ptr(), tp.data_ptr(),
                                   None, scale, window, T, heads, R, RD, bs, ws.data_ptr(), ws.numel(), None))
    torch.cuda.synchronize()
    for t in range(T):
        lo = max(0, pos[t] - window + 1) if window else 0
        j = torch.arange(lo, pos[t] + 1, device="cuda")
        rows = cache[bt[sid[t]].long()[j // bs] * bs + j % bs].double()
        q = torch.cat([qa[t], qr[t]], 1).double()
        d = 576 * 2.0 ** -24 * scale * (q.abs() @ rows.abs().T).max()
        exact = torch.softmax(q @ rows.T * scale, 1) @ rows[:, :R]
        bound = (torch.expm1(4 * d) + 2.0 ** -15 + 1024 * 2.0 ** -24) * rows[:, :R].abs().max()
        assert bool(((out[t].double() - exact).abs() <= bound).all()), (t, float((out[t].double() - exact).abs().max()), float(bound))


# rows of 512 + 64 values, 256 + 32 and 96 + 32: the three forms; 16 heads (a tile is one token) and 3 (five tokens of several sequences)
@pytest.mark.parametrize("R,RD", [(512, 64), (256, 32), (96, 32)])
@pytest.mark.parametrize("heads", [16, 3])
@pytest.mark.parametrize("parts", [True, False])
def test_position_without_keys(gpu, R, RD, heads, parts):
    """A token at position -1 has no keys: its output is zero whatever the cache and the memory before it hold (NaN here), and its neighbours
    are what they are without it."""
    vmx, torch = gpu
    from vllm_rust_amd._lib import check, lib
    bs, mb = 16, 10
    g = torch.Generator(device="cuda").manual_seed(R + heads)
    held = torch.full(((4 * mb + 1) * bs, R + RD), float("nan"), device="cuda", dtype=torch.bfloat16)
    cache = held[bs:]
    cache.copy_(torch.randn((4 * mb * bs, R + RD), device="cuda", generator=g))
    bt = torch.arange(4 * mb, dtype=torch.int32, device="cuda").view(4, mb)
    pos = torch.tensor([-1, 130, -1, 3], dtype=torch.int32, device="cuda")
    sid = torch.arange(4, dtype=torch.int32, device="cuda")
    qa = torch.randn((4, heads, R), device="cuda", generator=g)
    qr = torch.randn((4, heads, RD), device="cuda", generator=g)
    ws = torch.empty(lib.vmx_latent_attention_workspace_bytes(4, heads, R, 0, mb, bs) if parts else 16, dtype=torch.uint8, device="cuda")

    def run(pick):
        o = torch.full((len(pick), heads, R), float("nan"), device="cuda")
        a, r, t, p = (v[pick].contiguous() for v in (qa, qr, sid, pos))
        check(lib.vmx_latent_attention(o.data_ptr(), a.data_ptr(), r.data_ptr(), cache.data_ptr(), 1, bt.data_ptr(), mb, t.data_ptr(), p.data_ptr(), None,
                                       0.05, 0, len(pick), heads, R, RD, bs, ws.data_ptr(), ws.numel(), None))
        torch.cuda.synchronize()
        return o

    out, alone = run([0, 1, 2, 3]), run([1, 3])
    assert bool((out[[0, 2]] == 0).all())
    # the keys may be cut into other partitions: a weight's two bf16 halves are off by 2^-16, on either side
    assert float((out[[1, 3]] - alone).abs().max()) <= 2.0 ** -15 * float(cache.abs().max())


# row tiles of a workgroup that share their keys (one sequence), that do not (decode steps, ends of prompts), with two head groups, few heads, a
# window's lower edge inside a tile, tokens out of order, a padding token among them
@pytest.mark.parametrize("contexts,new,heads,window,shuffled", [
    ([270], 270, 20, 0, False), ([97, 66, 110], 110, 16, 33, True), ([33] * 259, 1, 16, 0, False), ([700], 600, 5, 100, True), ([257], 257, 16, 0, True),
])
def test_shared_keys(gpu, contexts, new, heads, window, shuffled):
    """Launches of more row tiles than compute units, with a sink, against float64; the bound is the one above."""
    vmx, torch = gpu
    from vllm_rust_amd._lib import check, lib
    R, RD, bs, scale = 512, 64, 16, 0.06
    g = torch.Generator(device="cuda").manual_seed(sum(contexts) + heads)
    n = len(contexts)
    mb = (max(contexts) + bs - 1) // bs
    bt = torch.randperm(n * mb, device="cuda", generator=g).to(torch.int32).view(n, mb)
    cache = torch.randn((n * mb * bs, R + RD), device="cuda", generator=g).to(torch.bfloat16)
    sid, pos = [], []
    for b, c in enumerate(contexts):
        k = min(new, c)
        p = list(range(c - k, c))
        if shuffled:
            p = p[::-1]
            p[1] = -1
        sid += [b] * k
        pos += p
    T = len(pos)
    qa = torch.randn((T, heads, R), device="cuda", generator=g).to(torch.bfloat16).float()
    qr = torch.randn((T, heads, RD), device="cuda", generator=g).to(torch.bfloat16).float()
    sink = torch.randn(heads, device="cuda", generator=g).to(torch.bfloat16)
    ts, tp = (torch.tensor(v, device="cuda", dtype=torch.int32) for v in (sid, pos))
    out = torch.full((T, heads, R), float("nan"), device="cuda")
    assert lib.vmx_latent_attention_workspace_bytes(T, heads, R, window, mb, bs) == 0
    check(lib.vmx_latent_attention(out.data_ptr(), qa.data_ptr(), qr.data_ptr(), cache.data_ptr(), 1, bt.data_ptr(), mb, ts.data_ptr(), tp.data_ptr(),
                                   sink.data_ptr(), scale, window, T, heads, R, RD, bs, None, 0, None))
    torch.cuda.synchronize()
    for t in range(T):
        lo = max(0, pos[t] - window + 1) if window else 0
        j = torch.arange(lo, pos[t] + 1, device="cuda")
        if not len(j):
            assert bool((out[t] == 0).all())
            continue
        rows = cache[bt[sid[t]].long()[j // bs] * bs + j % bs].double()
        q = torch.cat([qa[t], qr[t]], 1).double()
        d = 576 * 2.0 ** -24 * scale * (q.abs() @ rows.abs().T).max()
        logits = torch.cat([q @ rows.T * scale, sink.double()[:, None]], 1)
        exact = torch.softmax(logits, 1)[:, :-1] @ rows[:, :R]
        bound = (torch.expm1(4 * d) + 2.0 ** -15 + 1024 * 2.0 ** -24) * rows[:, :R].abs().max()
        assert bool(((out[t].double() - exact).abs() <= bound).all()), (t, float((out[t].double() - exact).abs().max()), float(bound))


# one token a row tile, with one and two head groups, and two tokens a row tile; a whole prompt and a window
@pytest.mark.parametrize("heads,window", [(16, 0), (16, 40), (20, 0), (8, 0), (8, 40)])
def test_rows_that_are_not_finite(gpu, heads, window):
    """An infinity or a NaN in a token's cache row reaches the tokens that have it among their keys (at least one result of each is not finite) and
    of the others at most those of its own row tile, before it: row tiles that share their keys with that token keep every bit."""
    vmx, torch = gpu
    from vllm_rust_amd._lib import check, lib
    R, RD, bs, scale, T = 512, 64, 16, 0.06, 532
    g = torch.Generator(device="cuda").manual_seed(heads + window)
    mb = (T + bs - 1) // bs
    bt = torch.randperm(mb, device="cuda", generator=g).to(torch.int32).view(1, mb)
    cache = torch.randn((mb * bs, R + RD), device="cuda", generator=g).to(torch.bfloat16)
    qa = torch.randn((T, heads, R), device="cuda", generator=g).to(torch.bfloat16).float()
    qr = torch.randn((T, heads, RD), device="cuda", generator=g).to(torch.bfloat16).float()
    pos = torch.arange(T, dtype=torch.int32, device="cuda")
    sid = torch.zeros(T, dtype=torch.int32, device="cuda")
    assert lib.vmx_latent_attention_workspace_bytes(T, heads, R, window, mb, bs) == 0

    def run():
        out = torch.full((T, heads, R), 7.0, device="cuda")
        check(lib.vmx_latent_attention(out.data_ptr(), qa.data_ptr(), qr.data_ptr(), cache.data_ptr(), 1, bt.data_ptr(), mb, sid.data_ptr(), pos.data_ptr(),
                                       None, scale, window, T, heads, R, RD, bs, None, 0, None))
        torch.cuda.synchronize()
        return out

    clean = run()
    tile = 16 // min(heads, 16)   # tokens a row tile
    for at, value in ((3, float("inf")), (98, float("nan")), (255, float("-inf")), (T - 1, float("nan"))):   # last of four tiles, in the middle, of a 32-key tile, of all
        row = int(bt[0, at // bs]) * bs + at % bs
        held = cache[row].clone()
        cache[row, 5:R:64] = value
        out = run()
        cache[row] = held
        last = min(T, at + window) if window else T      # tokens at .. last - 1 have the key
        assert bool((~torch.isfinite(out[at:last])).flatten(1).any(1).all())
        assert torch.equal(out[:at // tile * tile], clean[:at // tile * tile])
        first = (last + tile - 1) // tile * tile
        assert torch.equal(out[first:], clean[first:])


# the prompt alone, behind a whole group of row tiles of another one, and behind parts of a group; a window whose edges lie anywhere in a key tile
@pytest.mark.parametrize("heads", [16, 8])
@pytest.mark.parametrize("window", [0, 70])
def test_neighbours_in_a_step(gpu, heads, window):
    """Row tiles that share their keys give a token the same bits whichever tokens of its sequence are beside it.  Those whose group has another prompt's tokens in it
    sum in another order: their weights' two bf16 halves are off by 2^-16 on either side, as in test_position_without_keys, and the f32 sums of
    280 products by as many roundings."""
    vmx, torch = gpu
    from vllm_rust_amd._lib import check, lib
    R, RD, bs, scale, n = 512, 64, 16, 0.06, 280
    g = torch.Generator(device="cuda").manual_seed(heads + window)
    mb = (n + 15) // bs + 1
    bt = torch.randperm(2 * mb, device="cuda", generator=g).to(torch.int32).view(2, mb)
    cache = torch.randn((2 * mb * bs, R + RD), device="cuda", generator=g).to(torch.bfloat16)
    qa = torch.randn((2 * n, heads, R), device="cuda", generator=g)
    qr = torch.randn((2 * n, heads, RD), device="cuda", generator=g)

    def run(before):   # `before` tokens of sequence 1, then the n of sequence 0
        T = before + n
        pos = torch.cat([torch.arange(before), torch.arange(n)]).to(torch.int32).cuda()
        sid = torch.tensor([1] * before + [0] * n, dtype=torch.int32, device="cuda")
        a, r = (torch.cat([q[n:n + before], q[:n]]).contiguous() for q in (qa, qr))
        out = torch.full((T, heads, R), float("nan"), device="cuda")
        check(lib.vmx_latent_attention(out.data_ptr(), a.data_ptr(), r.data_ptr(), cache.data_ptr(), 1, bt.data_ptr(), mb, sid.data_ptr(), pos.data_ptr(),
                                       None, scale, window, T, heads, R, RD, bs, None, 0, None))
        torch.cuda.synchronize()
        return out[before:]

    group = 4 * (16 // heads)   # tokens of four row tiles
    alone = run(0)
    for before in (group, group + 1, 2 * group - 1, 33):
        got = run(before)
        mixed = -before % group   # tokens in the group with the other prompt's last ones
        assert torch.equal(got[mixed:], alone[mixed:])
        assert float((got[:mixed] - alone[:mixed]).abs().max() if mixed else 0.0) <= (2.0 ** -15 + 280 * 2.0 ** -23) * float(cache.abs().max())


# (R, RD, contexts, new tokens, heads, window): row tiles that share their keys, that lie in several sequences (prompts' ends, decode steps), partitions and their
# merge, and rows of other sizes
@pytest.mark.parametrize("R,RD,contexts,new,heads,window,parts", [
    (512, 64, [270], 270, 20, 0, False), (512, 64, [97, 66, 111], 111, 16, 33, False), (512, 64, [33] * 259, 1, 16, 0, False), (512, 64, [300, 301], 300, 5, 0, False),
    (512, 64, [128, 129, 700], 1, 16, 0, True), (256, 32, [70, 41], 60, 16, 0, True), (96, 32, [90, 41], 90, 3, 0, True),
])
def test_bf16_queries_and_results(gpu, R, RD, contexts, new, heads, window, parts):
    """Queries that are bf16 already, handed over as bf16 and as f32: the bf16 results are the f32 ones (which the tests above hold against float64)
    rounded, bit by bit.  Nothing is written beside them."""
    import ctypes as C
    vmx, torch = gpu
    from vllm_rust_amd._lib import check, lib
    bs, scale = 16, 0.06
    g = torch.Generator(device="cuda").manual_seed(sum(contexts) + heads + R)
    n = len(contexts)
    mb = (max(contexts) + bs - 1) // bs
    bt = torch.randperm(n * mb, device="cuda", generator=g).to(torch.int32).view(n, mb)
    cache = torch.randn((n * mb * bs, R + RD), device="cuda", generator=g).to(torch.bfloat16)
    sid, pos = [], []
    for b, c in enumerate(contexts):
        k = min(new, c)
        sid += [b] * k
        pos += list(range(c - k, c))
    pos[1] = -1                     # a row without keys
    T = len(pos)
    qa = torch.randn((T, heads, R), device="cuda", generator=g).to(torch.bfloat16)
    qr = torch.randn((T, heads, RD), device="cuda", generator=g)
    sink = torch.randn(heads, device="cuda", generator=g).to(torch.bfloat16)
    ts, tp = (torch.tensor(v, device="cuda", dtype=torch.int32) for v in (sid, pos))
    need = lib.vmx_latent_attention_workspace_bytes(T, heads, R, window, mb, bs)
    assert (need > 0) == parts
    ws = torch.empty(max(need, 16), dtype=torch.uint8, device="cuda")
    got = {}
    for io16, dt in ((0, torch.float32), (1, torch.bfloat16)):
        q, held = qa.to(dt), torch.full((T + 2, heads, R), 7.0, dtype=dt, device="cuda")
        p = lambda t: C.c_void_p(t.data_ptr())   # noqa: E731
        check(lib.vmx_latent_attention_launch(p(held[1:]), p(q), io16, p(qr), p(cache), 1, p(bt), mb, p(ts), p(tp), p(sink), C.c_float(scale), window, T, heads, R, RD, bs,
                                              p(ws), C.c_size_t(ws.numel()), None))
        torch.cuda.synchronize()
        assert bool((held[0] == 7.0).all()) and bool((held[T + 1] == 7.0).all())
        got[io16] = held[1:T + 1]
    assert bool((got[0][1] == 0).all()) and bool(got[0].isfinite().all())
    assert torch.equal(got[1], got[0].to(torch.bfloat16))
