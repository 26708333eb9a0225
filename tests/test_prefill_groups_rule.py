"""How many groups of waves share the keys of a wide-head prompt's workgroup (host arithmetic, no GPU): vmx_prefill_attention_groups."""
import pytest


def _groups(head_dim, heads, kv_heads, cache, q_len, offset=0, window=0):
    from vllm_rust_amd._lib import lib
    return lib._Z28vmx_prefill_attention_groupsiiiiiii(head_dim, heads // kv_heads, kv_heads, cache, q_len, offset, window)


# the time of one group over that of several: where a few tiles take no longer than the merge there is one group
@pytest.mark.parametrize("head_dim,heads,kv_heads,cache,keys,ratio", [
    (256, 16, 8, 0, 65, 0.93), (256, 16, 8, 0, 80, 0.88), (256, 16, 8, 0, 81, 1.01), (256, 16, 8, 1, 80, 0.94), (256, 16, 8, 1, 97, 1.09), (256, 8, 8, 0, 80, 0.92),
    (256, 8, 8, 1, 97, 1.15), (256, 32, 8, 0, 65, 1.06), (256, 32, 8, 1, 80, 1.09), (256, 8, 1, 0, 80, 1.04), (512, 16, 1, 0, 80, 0.93), (512, 16, 1, 0, 112, 0.99),
    (512, 16, 1, 0, 129, 1.03), (512, 16, 1, 1, 80, 0.98), (512, 16, 1, 1, 97, 1.07), (512, 8, 4, 0, 97, 0.98), (512, 8, 4, 0, 113, 1.13), (512, 8, 4, 1, 80, 0.95),
])
def test_the_faster_side(head_dim, heads, kv_heads, cache, keys, ratio):
    assert (_groups(head_dim, heads, kv_heads, cache, keys) > 1) == (ratio > 1)


def test_keys_are_those_that_a_workgroup_walks():
    assert _groups(256, 16, 8, 1, 1, offset=80) > 1 and _groups(256, 16, 8, 1, 1, offset=79) == 1      # history counts
    assert _groups(256, 16, 8, 1, 200, window=40) == 1 and _groups(256, 16, 8, 1, 200, window=100) > 1   # what a window hides does not
    assert _groups(128, 16, 8, 1, 4096) == 1                                                             # heads of up to 128: a form of their own


def test_groups_leave_room_for_the_workgroups():
    assert [_groups(256, 16, 8, 1, n) for n in (256, 512, 1024, 2048, 4096)] == [4, 4, 2, 2, 1]
    assert [_groups(512, 16, 1, 1, n) for n in (256, 4096)] == [2, 2]
