"""How many columns a workgroup of the unquantised decode products owns (host arithmetic, no GPU): vmx_dense_decode_tiles."""
import pytest


@pytest.mark.parametrize("hidden", [512, 896, 1024, 1536, 2048, 2560, 3072, 4096, 8192])
@pytest.mark.parametrize("rows", [1, 2, 3, 4, 5, 16])
def test_few_workgroups_repeat_the_rows_work(hidden, rows):
    """Every workgroup norms or merges all rows.  Four columns a workgroup instead of sixteen are for products that leave half of the compute units
    idle, and only while rows times sixteen-column workgroups stay below the compute units (measured slower beyond, by up to half)."""
    from vllm_rust_amd._lib import lib
    tiles = lib._Z22vmx_dense_decode_tilesii(rows, hidden)
    narrow = rows <= 4 and hidden // 16 <= 128 and rows * (hidden // 16) <= 256
    assert tiles == hidden // (4 if narrow else 16)
