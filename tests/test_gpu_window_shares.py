"""Window attention of decode rows whose key tiles are dealt to several workgroups: sequences with fewer tiles than there are shares."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    import torch
    import vllm_rust_amd as vmx
    vmx.init(0)
    return vmx, torch


# tiles hold 64 keys; a table of 1000 tokens allows 16 of them, one of 112 tokens two; a kept first token and a window; six heads a key/value head
# take two workgroups of four
@pytest.mark.parametrize("contexts,table,window,keep,heads", [
    ([1, 64, 65, 1000, 130], 1000, 0, 0, 8), ([100, 3], 112, 0, 0, 8), ([100, 3, 700], 4096, 0, 0, 12), ([900, 40, 129], 1000, 70, 2, 8), ([64], 64, 0, 0, 2),
])
@pytest.mark.parametrize("sink", [False, True])
def test_shares_without_keys(gpu, contexts, table, window, keep, heads, sink):
    """Against float64 on the operands the kernel multiplies; the workspace holds NaN beforehand, so a sum that no share wrote may not be read.
    A score is off by at most d = 64 2^-24 scale sum |q k|, a weight by a factor exp(2 d) and its bf16 pair by 2^-16, the sums of up to
    1024 weighted rows by 1024 2^-24 of the largest value."""
    vmx, torch = gpu
    import ctypes as C
    from vllm_rust_amd._lib import WindowAttnExtras, check, lib
    G, D, bs, scale = 2, 64, 16, 0.11
    n, mb = len(contexts), (table + bs - 1) // bs
    g = torch.Generator(device="cuda").manual_seed(sum(contexts) + heads)
    bt = torch.zeros((n, mb), dtype=torch.int32, device="cuda")
    used = [(c + bs - 1) // bs for c in contexts]
    free = torch.randperm(sum(used), device="cuda", generator=g).to(torch.int32)
    for b, u in enumerate(used):
        bt[b, :u] = free[sum(used[:b]):sum(used[:b]) + u]
    kc = torch.randn((sum(used) * bs, G, D), device="cuda", generator=g).to(torch.bfloat16)
    vc = torch.randn((sum(used) * bs, G, D), device="cuda", generator=g).to(torch.bfloat16)
    q = torch.randn((n, heads, D), device="cuda", generator=g).to(torch.bfloat16).float()
    sid, starts = torch.arange(n, dtype=torch.int32, device="cuda"), torch.arange(n + 1, dtype=torch.int32, device="cuda")
    pos = torch.tensor([c - 1 for c in contexts], dtype=torch.int32, device="cuda")
    sinks = torch.randn(heads, device="cuda", generator=g).to(torch.bfloat16)
    ex = WindowAttnExtras()
    if sink:
        ex.sink_bf16 = sinks.data_ptr()
    size = lib.vmx_window_attention_workspace_bytes(n, heads, D)
    ws = torch.full((size // 4,), float("nan"), device="cuda")
    out = torch.empty((n, heads, D), device="cuda")
    check(lib.vmx_window_attention_ex(out.data_ptr(), 0, q.data_ptr(), heads * D, kc.data_ptr(), vc.data_ptr(), 1, bt.data_ptr(), mb, sid.data_ptr(),
                                      pos.data_ptr(), None, None, 0, scale, 0.0, window, keep, n, heads, G, D, D, bs, starts.data_ptr(), n, ws.data_ptr(),
                                      size, C.byref(ex), None))
    torch.cuda.synchronize()
    for b, c in enumerate(contexts):
        lo = max(0, c - window) if window else 0
        j = torch.tensor(list(range(min(keep, lo))) + list(range(lo, c)), device="cuda")
        rows = bt[b].long()[j // bs] * bs + j % bs
        for h in range(heads):
            k, v = (t[rows, h // (heads // G)].double() for t in (kc, vc))
            s = (k @ q[b, h].double()) * scale
            d = 64 * 2.0 ** -24 * scale * float((k.abs() @ q[b, h].double().abs()).max())
            e = torch.cat([s, sinks[h].double().view(1)]) if sink else s
            exact = torch.softmax(e, 0)[:len(s)] @ v
            bound = (2 * d + 2.0 ** -15 + 1024 * 2.0 ** -24) * float(v.abs().max())
            assert float((out[b, h].double() - exact).abs().max()) <= bound, (b, h)
