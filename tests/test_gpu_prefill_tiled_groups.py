"""Prompts of 64- and 128-wide heads whose key tiles two groups of a workgroup share: the first key count that takes the form (321: six tiles) and the last that does not,
an odd and an even number of tiles, windows, history, every number of heads a workgroup has and every cache; and cache blocks of sizes that are no power of two, whose
places are found by a reciprocal."""
import pytest

import tests.test_gpu_prefill_attn as one_group

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hd,H,KVH,q_len,offset,window,kv_dtype", [
    (128, 8, 2, 320, 0, 0, 0), (128, 8, 2, 321, 0, 0, 0), (128, 8, 2, 385, 0, 0, 1), (128, 8, 2, 448, 0, 0, 3), (64, 4, 2, 450, 0, 0, 0), (64, 2, 2, 333, 0, 0, 1),
    (128, 2, 2, 1, 320, 0, 0), (128, 6, 2, 33, 400, 0, 0), (128, 8, 1, 31, 1000, 0, 3), (64, 8, 2, 5, 500, 0, 1),                        # history
    (128, 8, 2, 400, 0, 288, 0), (128, 8, 2, 400, 0, 289, 0), (128, 4, 2, 500, 77, 300, 1), (64, 4, 4, 350, 50, 310, 0),                 # windows that start inside a tile
])
def test_key_groups(hd, H, KVH, q_len, offset, window, kv_dtype):
    one_group.test_prefill_attention_matches_float64(hd, H, KVH, q_len, offset, window, kv_dtype)


@pytest.mark.parametrize("block_size", [1, 3, 7, 24, 48, 100])
@pytest.mark.parametrize("q_len,offset", [(70, 9), (400, 0)])
def test_block_sizes(block_size, q_len, offset):
    """The same rows in blocks of another size: the same results to the bit."""
    import torch
    import vllm_rust_amd as vmx
    from vllm_rust_amd._lib import check, lib
    vmx.init(0)
    H, KVH, hd, total = 8, 2, 128, q_len + offset
    g = torch.Generator().manual_seed(block_size + q_len)
    k, v, q = (torch.randn(n, h, hd, generator=g).bfloat16().cuda() for n, h in ((total, KVH), (total, KVH), (q_len, H)))
    outs = []
    for bs in (16, block_size):
        n = (total + bs - 1) // bs
        table = torch.randperm(n + 2, generator=g)[:n].int().cuda()
        pos = torch.arange(total).cuda()
        slots = table.long()[pos // bs] * bs + pos % bs
        caches = []
        for rows in (k, v):
            c = torch.zeros((n + 2) * bs, KVH, hd, dtype=torch.bfloat16, device="cuda")
            c[slots] = rows
            caches.append(c)
        out = torch.empty_like(q)
        check(lib.vmx_prefill_attention_bf16(out.data_ptr(), q.data_ptr(), caches[0].data_ptr(), caches[1].data_ptr(), table.data_ptr(), q_len, offset, hd ** -0.5, H,
                                             KVH, hd, bs, 0, 0, None, None, torch.cuda.current_stream().cuda_stream))
        torch.cuda.synchronize()
        outs.append(out)
    assert torch.equal(outs[0], outs[1])


@pytest.mark.parametrize("hd,H,KVH,q_len,offset,window,kv_dtype", [(64, 128, 16, 352, 0, 296, 0), (64, 128, 16, 340, 169, 0, 1)])
def test_more_workgroups_than_units(hd, H, KVH, q_len, offset, window, kv_dtype):
    """352 workgroups and even chains: one group."""
    one_group.test_prefill_attention_matches_float64(hd, H, KVH, q_len, offset, window, kv_dtype)


# 256 compute units: up to that many workgroups whatever the chains, up to twice as many where the average chain is at most 0.7 of the longest and that is nine tiles or more
@pytest.mark.parametrize("H,KVH,q_len,offset,window,groups", [
    (8, 2, 321, 0, 0, 2), (16, 2, 2562, 0, 494, 1), (32, 8, 1627, 0, 406, 1), (32, 8, 1024, 0, 400, 2), (32, 8, 1025, 0, 400, 1), (32, 8, 1025, 0, 0, 2), (64, 16, 539, 0, 0, 1),
    (64, 16, 576, 0, 0, 2), (64, 16, 600, 900, 0, 1), (32, 8, 1102, 423, 0, 2), (32, 8, 1500, 3000, 0, 1), (16, 8, 2100, 0, 1100, 1), (16, 8, 2100, 0, 2080, 2), (8, 2, 64, 1000, 0, 2)])
def test_groups_chosen(H, KVH, q_len, offset, window, groups):
    import torch
    import vllm_rust_amd as vmx
    from tests.helpers import launched_kernels
    from vllm_rust_amd._lib import check, lib
    vmx.init(0)
    total = q_len + offset
    q, k = torch.zeros(q_len, H, 128, dtype=torch.bfloat16, device="cuda"), torch.zeros((total + 15) // 16 * 16, KVH, 128, dtype=torch.bfloat16, device="cuda")
    table, out = torch.arange((total + 15) // 16, dtype=torch.int32, device="cuda"), torch.empty_like(q)
    (name,) = [n for n, *_ in launched_kernels(torch, lambda: check(lib.vmx_prefill_attention_bf16(
        out.data_ptr(), q.data_ptr(), k.data_ptr(), k.data_ptr(), table.data_ptr(), q_len, offset, 128 ** -0.5, H, KVH, 128, 16, window, 0, None, None,
        torch.cuda.current_stream().cuda_stream)))]
    assert f"Li4ELi{groups}EE" in name, name
