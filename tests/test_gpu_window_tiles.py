"""Window attention of prompts on the matrix cores: tiles that every row sees and tiles in which keys are hidden, block sizes of any kind."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    import torch
    import vllm_rust_amd as vmx
    vmx.init(0)
    return vmx, torch


# tiles hold 64 keys and a wave 16 rows; heads that fill their 16-byte chunks' rounded width and heads that do not
@pytest.mark.parametrize("block", [1, 7, 16, 48])
@pytest.mark.parametrize("heads,groups,dim,vdim", [(4, 1, 64, 64), (6, 2, 72, 24), (2, 2, 128, 128), (5, 1, 200, 40)])
@pytest.mark.parametrize("window,keep,chunk,softcap,dist", [(0, 0, 0, 0.0, False), (100, 3, 0, 0.0, True), (90, 0, 0, 5.0, False), (0, 0, 96, 5.0, True)])
def test_prompt_tiles(gpu, block, heads, groups, dim, vdim, window, keep, chunk, softcap, dist):
    """Against float64 on the operands the kernel multiplies.  A score is off by at most d = (dim + 8) 2^-24 scale sum |q k| (capped: plus
    softcap 2^-20 of tanh through one exponential; with the penalty: plus 2^-20 of its size), a weight by a factor exp(2 d) and its bf16 pair by
    2^-16, the sums of up to 512 weighted rows by 512 2^-24 of the largest value.  Cache rows of no sequence hold NaN and may not be read."""
    vmx, torch = gpu
    import ctypes as C
    from vllm_rust_amd._lib import WindowAttnExtras, check, lib
    lens, before, scale = [1, 64, 65, 130, 200], [0, 3, 128, 0, 250], 0.09
    total = [a + b for a, b in zip(lens, before)]
    n, T = len(lens), sum(lens)
    g = torch.Generator(device="cuda").manual_seed(block * 1000 + dim + window)
    used = [(c + block - 1) // block for c in total]
    mb = max(used) + 1
    order = torch.randperm(sum(used) + 2, device="cuda", generator=g).to(torch.int32)
    bt = torch.full((n, mb), int(order[-1]), dtype=torch.int32, device="cuda")
    slots = []
    for b, u in enumerate(used):
        bt[b, :u] = order[sum(used[:b]):sum(used[:b]) + u]
        j = torch.arange(total[b], device="cuda")
        slots.append(bt[b].long()[j // block] * block + j % block)
    kc = torch.full(((sum(used) + 2) * block, groups, dim), float("nan"), device="cuda", dtype=torch.bfloat16)
    vc = torch.full(((sum(used) + 2) * block, groups, vdim), float("nan"), device="cuda", dtype=torch.bfloat16)
    for s in slots:
        kc[s] = torch.randn((len(s), groups, dim), device="cuda", generator=g).to(torch.bfloat16)
        vc[s] = torch.randn((len(s), groups, vdim), device="cuda", generator=g).to(torch.bfloat16)
    q = torch.randn((T, heads, dim), device="cuda", generator=g).to(torch.bfloat16).float()
    starts = torch.tensor([sum(lens[:i]) for i in range(n + 1)], dtype=torch.int32, device="cuda")
    sid = torch.tensor([b for b in range(n) for _ in range(lens[b])], dtype=torch.int32, device="cuda")
    pos = torch.tensor([before[b] + i for b in range(n) for i in range(lens[b])], dtype=torch.int32, device="cuda")
    r1, r2 = (torch.rand(heads, device="cuda", generator=g).to(torch.bfloat16) for _ in range(2))
    ex = WindowAttnExtras()
    ex.chunk = chunk
    if dist:
        ex.dist_r1_bf16, ex.dist_r2_bf16 = r1.data_ptr(), r2.data_ptr()
    out = torch.empty((T, heads, vdim), device="cuda")
    check(lib.vmx_window_attention_ex(out.data_ptr(), 0, q.data_ptr(), heads * dim, kc.data_ptr(), vc.data_ptr(), 1, bt.data_ptr(), mb, sid.data_ptr(),
                                      pos.data_ptr(), None, None, 0, scale, softcap, window, keep, T, heads, groups, dim, vdim, block, starts.data_ptr(), n,
                                      None, 0, C.byref(ex), None))
    torch.cuda.synchronize()
    for b in range(n):
        i = torch.arange(before[b], total[b], device="cuda")[:, None]
        j = torch.arange(total[b], device="cuda")[None, :]
        lo = torch.zeros_like(i)
        if window:
            lo = torch.maximum(lo, i - window + 1)
        if chunk:
            lo = torch.maximum(lo, i // chunk * chunk)
        seen = (j <= i) & ((j >= lo) | (j < keep))
        for h in range(heads):
            k, v = (t[slots[b], h // (heads // groups)].double() for t in (kc, vc))
            x = q[int(starts[b]):int(starts[b + 1]), h].double()
            s = x @ k.T.contiguous() * scale
            d = (dim + 8) * 2.0 ** -24 * scale * float((x.abs() @ k.abs().T.contiguous()).max())
            if softcap:
                s, d = softcap * torch.tanh(s / softcap), d + softcap * 2.0 ** -20
            if dist:
                pen = r1[h].double() * torch.log(1 + r2[h].double() * (i - j).clamp(min=0))
                s, d = s - pen, d + 2.0 ** -20 * float(pen.max())
            exact = torch.softmax(s.masked_fill(~seen, float("-inf")), 1) @ v
            bound = (2 * d + 2.0 ** -15 + 512 * 2.0 ** -24) * float(v.abs().max())
            got = out[int(starts[b]):int(starts[b + 1]), h].double()
            assert float((got - exact).abs().max()) <= bound, (b, h)


@pytest.mark.parametrize("talk,sink", [(False, False), (False, True), (True, False)])
@pytest.mark.parametrize("shares", [False, True])
@pytest.mark.parametrize("block", [16, 7])
def test_rows_without_keys(gpu, block, shares, talk, sink):
    """A row at position -1 sees no key: it is what a softmax over nothing gives (zeros with a sink, else not a number), with and without shares of keys and their merge, and
    the other rows are what they are without it.  (Whether its block table is read shows in no result: all it could bring is hidden.)"""
    vmx, torch = gpu
    import ctypes as C
    from vllm_rust_amd._lib import WindowAttnExtras, check, lib
    heads, dim, T = 4, 64, 70
    g = torch.Generator(device="cuda").manual_seed(block)
    mb = (T + block - 1) // block
    bt = torch.zeros((2, mb), dtype=torch.int32, device="cuda")
    bt[0] = torch.randperm(mb, device="cuda", generator=g).to(torch.int32)
    bt[1] = -1
    kc, vc = (torch.randn((mb * block, 1, dim), device="cuda", generator=g).to(torch.bfloat16) for _ in range(2))
    q = torch.randn((T + 1, heads, dim), device="cuda", generator=g)
    mix, sinks = torch.randn((heads, heads), device="cuda", generator=g).to(torch.bfloat16), torch.randn(heads, device="cuda", generator=g).to(torch.bfloat16)
    ex = WindowAttnExtras()
    if talk:
        ex.talk_bf16 = mix.data_ptr()
    if sink:
        ex.sink_bf16 = sinks.data_ptr()
    sid = torch.tensor([0] * T + [1], dtype=torch.int32, device="cuda")
    pos = torch.tensor(list(range(T)) + [-1], dtype=torch.int32, device="cuda")
    starts = torch.tensor([0, T, T + 1], dtype=torch.int32, device="cuda")
    size = lib.vmx_window_attention_workspace_bytes(T + 1, heads, dim) if shares else 0
    ws = torch.full((size // 4,), float("nan"), device="cuda")

    def run(rows, seqs):
        out = torch.full((T + 2, heads, dim), 3.0, device="cuda")
        check(lib.vmx_window_attention_ex(out.data_ptr(), 0, q.data_ptr(), heads * dim, kc.data_ptr(), vc.data_ptr(), 1, bt.data_ptr(), mb, sid.data_ptr(),
                                          pos.data_ptr(), None, None, 0, 0.1, 0.0, 0, 0, rows, heads, 1, dim, dim, block, starts.data_ptr(), seqs,
                                          ws.data_ptr() if shares else None, size, C.byref(ex), None))
        torch.cuda.synchronize()
        assert bool((out[rows:] == 3.0).all())
        return out
    both, alone = run(T + 1, 2), run(T, 1)
    assert torch.equal(both[:T], alone[:T]) and bool(both[:T].isfinite().all())
    assert bool((both[T] == 0).all()) if sink else bool(both[T].isnan().all())
