"""How many workgroups share a KV head of a decode row (host arithmetic, no GPU): vmx_split_decode_attention_long_parts."""
import pytest


def _parts(bound, kv_heads, rows):
    from vllm_rust_amd._lib import lib
    return lib._Z37vmx_split_decode_attention_long_partsiiiiiii(128, 1, 128, bound, 0, kv_heads, rows)


@pytest.mark.parametrize("kv_heads", [1, 4, 8, 16, 32])
@pytest.mark.parametrize("rows", [1, 3, 8, 12, 16])
def test_a_long_row_keeps_its_workgroups(kv_heads, rows):
    """A row of the bound's length may sit among short ones, whose workgroups finish early: beyond 2048 tokens eight are the least, beyond
    1024 four, whatever the batch; the count never falls as the bound grows and never exceeds what the workspace holds."""
    counts = [_parts(b, kv_heads, rows) for b in (513, 1024, 1025, 2048, 2049, 8192, 32768)]
    assert counts == sorted(counts) and 1 <= counts[0] and counts[-1] <= 64
    assert min(counts[2:]) >= 4 and min(counts[4:]) >= 8


def test_short_contexts_are_not_covered():
    assert _parts(512, 8, 16) == 0
