"""Wide-head prompts whose key tiles several groups of a workgroup share: the first key count that takes the form and the last that does not, tile counts that leave
groups without a last tile, windows that start inside a group's run, history, every head ratio that has a form of its own; against float64 as the prompts of one group."""
import pytest

import tests.test_gpu_prefill_attn as one_group

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hd,H,KVH,q_len,offset,window,kv_dtype", [
    (256, 4, 2, 64, 0, 0, 1), (256, 4, 2, 65, 0, 0, 1), (256, 4, 2, 16, 49, 0, 0), (256, 4, 2, 97, 0, 0, 0),     # two heads a KV head, four groups
    (256, 16, 8, 300, 11, 100, 1), (256, 4, 4, 81, 3, 0, 1), (256, 8, 2, 130, 0, 40, 0), (256, 16, 1, 70, 30, 0, 1),   # windows, one, four and sixteen heads
    (256, 16, 8, 600, 0, 0, 1),                                                                                    # two groups of 32 rows
    (256, 4, 2, 80, 0, 0, 1), (256, 4, 2, 81, 0, 0, 0), (256, 4, 4, 1, 80, 0, 1), (256, 8, 2, 64, 0, 0, 0), (256, 8, 2, 65, 0, 0, 1),   # 80 and 81 keys; 64 and 65 of four heads a workgroup
    (512, 16, 1, 80, 0, 0, 1), (512, 4, 2, 81, 0, 0, 1), (512, 16, 1, 112, 0, 0, 0), (512, 2, 2, 113, 0, 0, 0),                         # 80 and 81 in FP8, 112 and 113 in bf16
    (512, 16, 1, 65, 0, 0, 1), (512, 16, 1, 64, 0, 0, 1), (512, 4, 2, 100, 7, 50, 0), (512, 2, 2, 90, 0, 0, 1), (512, 6, 2, 33, 64, 0, 0),
])
def test_key_groups(hd, H, KVH, q_len, offset, window, kv_dtype):
    one_group.test_prefill_attention_matches_float64(hd, H, KVH, q_len, offset, window, kv_dtype)
