"""Prefill-sized products that were not timed at start-up: which of them take the tiled GEMM, and what it gives there."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


# (the fewest and the most rows that a rule takes, and one row outside of it; row tiles full, with one row, and with all but one; fp16)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,n,k,silu,tiled", [
    (768, 2048, 13824, False, True), (767, 2048, 13824, False, False), (1024, 2048, 13824, False, True), (1025, 2048, 13824, False, True),
    (513, 2048, 13824, False, False),
    (1024, 2048, 13760, False, False), (2048, 2048, 13888, False, True), (469, 28672, 128, True, True), (468, 28672, 128, True, False),
    (512, 28672, 128, True, True), (513, 28672, 128, True, False)])
def test_layers_that_were_not_timed(dtype, rows, n, k, silu, tiled):
    from semi_pd_amd import ops
    from semi_pd_amd.layers import basic
    g = torch.Generator(device=DEV).manual_seed(rows + n)
    x = torch.randn(rows, k, generator=g, device=DEV).to(dtype)
    w = (k ** -0.5 * torch.randn(n, k, generator=g, device=DEV)).to(dtype)
    assert ops.tiled_gemm_fills_chip(n, k, rows, silu) == tiled
    was = basic.stream_linear_enabled()
    basic.set_stream_linear(True)
    try:
        assert basic._prefers_tiled_gemm(w, rows, silu) == tiled and ops.gemm_tall_is_supported(x, w, fuse_silu_mul=silu)
        got = ops.gemm_tall(x, w, fuse_silu_mul=silu) if silu else basic.dense_linear(x, w)
    finally:
        basic.set_stream_linear(was)
    want = x.float() @ w.float().t()
    half = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]             # of a value just above a power of two
    if silu:                                                                          # gate and up are rounded, then the product
        gate, up = want.to(dtype).float().chunk(2, -1)
        want, half = torch.nn.functional.silu(gate) * up, 4 * half
    # sums of up to 14 k terms of about k^-1/2 in 32 bits: sqrt(k) roundings of 2^-24 of a result of about 1
    torch.testing.assert_close(got.float(), want, rtol=half, atol=half * 0.05 + 2.0 ** -17)


def test_rule_is_for_the_whole_chip(monkeypatch):
    from semi_pd_amd import ops
    for cus, takes in ((0, True), (256, True), (128, False)):
        monkeypatch.setitem(ops._DENSE_GEMM, "cus", cus)
        assert ops.tiled_gemm_fills_chip(4096, 14336, 2048) == takes
