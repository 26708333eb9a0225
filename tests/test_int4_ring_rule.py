"""When the linears of 5 .. 16 rows end in the residual stream (host arithmetic, no GPU): vmx_int4_ring_resid_pays."""
import ctypes as C

import pytest


# columns, depth: one round of 256 compute units, more than half of one for the deepest sums, two rounds of sums half as deep as the columns are many
@pytest.mark.parametrize("N,K,pays", [
    (4096, 4096, True), (4096, 8192, True), (4096, 12288, True), (2048, 4096, True), (2048, 6144, True), (2048, 8192, True), (2048, 12288, False), (2064, 12288, True),
    (4112, 4096, False), (6144, 2048, True), (6144, 4096, False), (6144, 6144, False), (8192, 4096, True), (8192, 6144, False), (8192, 8192, False), (8208, 2048, False),
    (4096, 1024, False), (4096, 5120, False), (4096, 14336, False),
])
def test_where_a_layer_gains(N, K, pays):
    from vllm_rust_amd._lib import lib
    f = lib._Z24vmx_int4_ring_resid_paysiii
    f.restype = C.c_bool
    assert [f(M, N, K) for M in (4, 5, 16, 17)] == [False, pays, pays, False]
