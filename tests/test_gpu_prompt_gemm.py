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


# (short last tiles: a free CU for each of them, two in turn to a free CU, a round of their own; of one row and of 64; and what goes to the library)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,n,k,tiled", [(800, 16384, 2048, True), (1088, 12288, 2048, True), (1089, 12288, 2048, False), (1345, 22016, 2048, False),
                                            (1281, 22016, 2048, True), (1025, 24576, 2048, False), (2049, 16384, 2048, True), (576, 32768, 4096, False)])
def test_gate_and_up_with_a_short_last_tile(dtype, rows, n, k, tiled, monkeypatch):
    """gate_up_silu takes the tiled GEMM by the rule and gives the pair's result."""
    from semi_pd_amd import ops
    from semi_pd_amd.layers import basic
    assert ops.tiled_gemm_short_tail(n, k, rows) == tiled and not ops.tiled_gemm_fills_chip(n, k, rows, True)
    g = torch.Generator(device=DEV).manual_seed(rows + n)
    x = torch.randn(rows, k, generator=g, device=DEV).to(dtype)
    layer = basic.MergedColumnParallelLinear(k, [n // 2, n // 2], params_dtype=dtype).to(DEV)
    layer.weight.data.copy_(k ** -0.5 * torch.randn(n, k, generator=g, device=DEV))
    called, gemm_tall = [], ops.gemm_tall
    monkeypatch.setattr(ops, "gemm_tall", lambda *a, **kw: called.append(1) or gemm_tall(*a, **kw))
    was = basic.stream_linear_enabled()
    basic.set_stream_linear(True)
    try:
        got = basic.gate_up_silu(x, layer, basic.SiluAndMul())
    finally:
        basic.set_stream_linear(was)
    assert bool(called) == tiled
    gate, up = (x.float() @ layer.weight.float().t()).to(dtype).float().chunk(2, -1)
    # sums in another order may round gate or up to the neighbour, 2 half of the value away (SiLU's slope is at most 1.1); the product is rounded once
    half, silu = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype], torch.nn.functional.silu(gate)
    bound = 2 * half * 1.1 * (gate * up).abs() + 2 * half * (silu * up).abs() + half * (silu * up).abs() + 2.0 ** -17
    assert ((got.float() - silu * up).abs() <= bound).all()


def test_rule_is_for_the_whole_chip(monkeypatch):
    from semi_pd_amd import ops
    for cus, takes in ((0, True), (256, True), (128, False)):
        monkeypatch.setitem(ops._DENSE_GEMM, "cus", cus)
        assert ops.tiled_gemm_fills_chip(4096, 14336, 2048) == takes


@pytest.mark.parametrize("form", ["weight off 16 bytes", "rows of x in one place", "out off 8 bytes", "out rows off 8 bytes", "no columns"])
def test_what_the_tiled_gemm_does_not_take_goes_to_the_library(form):
    """Sizes that the rule takes, operands that the kernel does not."""
    from semi_pd_amd import ops
    from semi_pd_amd.layers import basic
    rows, n, k = 1536, 0 if form == "no columns" else 1024, 13824
    assert n == 0 or ops.tiled_gemm_fills_chip(n, k, rows)
    g = torch.Generator(device=DEV).manual_seed(5)
    x = torch.randn(rows, k, generator=g, device=DEV).bfloat16()
    w = (k ** -0.5 * torch.randn(n * k + 1, generator=g, device=DEV)).bfloat16()
    w = (w[1:] if form == "weight off 16 bytes" else w[:-1]).view(n, k)
    out = None
    if form == "rows of x in one place":
        x = x[:1].expand(rows, k)
    elif form == "out off 8 bytes":
        out = torch.empty(rows * n + 1, device=DEV, dtype=torch.bfloat16)[1:].view(rows, n)
    elif form == "out rows off 8 bytes":
        out = torch.empty(rows, n + 1, device=DEV, dtype=torch.bfloat16)[:, :n]
    was = basic.stream_linear_enabled()
    basic.set_stream_linear(True)
    try:
        got = basic.dense_linear(x, w, out=out)
    finally:
        basic.set_stream_linear(was)
    assert out is None or got.data_ptr() == out.data_ptr()
    # sums of 14 k terms of about k^-1/2 in 32 bits, one rounding of the result
    torch.testing.assert_close(got.float(), x.float() @ w.float().t(), rtol=2.0 ** -8, atol=2.0 ** -8 * 0.05 + 2.0 ** -17)


@pytest.mark.parametrize("rows,timed,tiled", [(469, None, True), (468, None, False), (512, False, False), (468, True, True)])
def test_which_way_gate_and_up_go(rows, timed, tiled, monkeypatch):
    """Both sides of the rule's edge through the layer's own call; what was timed at start-up goes before the rule."""
    from semi_pd_amd import ops
    from semi_pd_amd.layers import basic
    k, ff = 128, 14336
    g = torch.Generator(device=DEV).manual_seed(rows)
    layer = basic.MergedColumnParallelLinear(k, [ff, ff], params_dtype=torch.bfloat16).to(DEV)
    layer.weight.data.copy_(k ** -0.5 * torch.randn(2 * ff, k, generator=g, device=DEV))
    x = torch.randn(rows, k, generator=g, device=DEV).bfloat16()
    calls, kernel = [], ops.gemm_tall
    monkeypatch.setattr(ops, "gemm_tall", lambda *a, **kw: calls.append(kw.get("fuse_silu_mul", False)) or kernel(*a, **kw))
    if timed is not None:
        monkeypatch.setattr(ops, "dense_gemm_is_tuned", lambda w: True)
        monkeypatch.setattr(ops, "tall_preferred", lambda w, n, fuse_silu_mul=False: timed and fuse_silu_mul)
        monkeypatch.setattr(ops, "dense_gemm", lambda x, w, bias=None, out=None: torch.nn.functional.linear(x, w, bias))
    was = basic.stream_linear_enabled()
    basic.set_stream_linear(True)
    try:
        got = basic.gate_up_silu(x, layer, basic.SiluAndMul())
    finally:
        basic.set_stream_linear(was)
    assert calls == ([True] if tiled else [])
    gate, up = (x.float() @ layer.weight.float().t()).bfloat16().float().chunk(2, -1)
    # gate and up are rounded, then the product
    torch.testing.assert_close(got.float(), torch.nn.functional.silu(gate) * up, rtol=2.0 ** -6, atol=2.0 ** -6 * 0.05)


def _long_k(rows, seed, n=1024, k=13824):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return torch.randn(rows, k, generator=g, device=DEV).bfloat16(), (k ** -0.5 * torch.randn(n, k, generator=g, device=DEV)).bfloat16()


def test_slices_of_several_threads_on_one_stream():
    """Each call has planes of its own: the results are those of one thread, bit for bit."""
    import threading
    from semi_pd_amd import ops
    inputs = [_long_k(1536, seed) for seed in (1, 2, 3)]
    want = [ops.gemm_tall(x, w, own_planes=True) for x, w in inputs]
    got = [[] for _ in inputs]

    def work(i):
        for _ in range(20):
            got[i].append(ops.gemm_tall(*inputs[i], own_planes=True))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(inputs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert all(len(g) == 20 and all(torch.equal(o, w) for o in g) for g, w in zip(got, want))


def test_slices_leave_the_planes_of_a_decode_batch(monkeypatch):
    """A prefill-sized product between a decode batch's planes and the norm that takes them."""
    from semi_pd_amd import ops
    from semi_pd_amd.layers import basic
    x, w = _long_k(16, 4)
    res, norm = torch.randn(16, 1024, device=DEV).bfloat16(), torch.rand(1024, device=DEV).bfloat16()
    results = []
    for between in (False, True):
        planes, r = ops.stream_linear_planes(x, w), res.clone()
        if between:
            big, weight = _long_k(1536, 5)
            monkeypatch.setitem(basic._STREAM_LINEAR, "enabled", True)
            assert basic._takes_tiled_gemm(big, weight)
            basic.dense_linear(big, weight)
        results.append((ops.fused_add_rmsnorm_planes(planes, r, norm, 1e-5), r))
    assert all(torch.equal(a, b) for a, b in zip(*results))


def test_without_room_for_slices(monkeypatch):
    """The device's memory at its end: one slice, another order of the sums."""
    from semi_pd_amd import ops
    x, w = _long_k(1536, 6)
    out, empty = torch.empty(1536, 1024, device=DEV, dtype=torch.bfloat16), torch.empty

    def full(*a, **kw):
        if kw.get("dtype") == torch.uint8:
            raise torch.OutOfMemoryError("no room")
        return empty(*a, **kw)

    monkeypatch.setattr(torch, "empty", full)
    got = ops.gemm_tall(x, w, out=out, own_planes=True)
    monkeypatch.undo()
    torch.testing.assert_close(got.float(), x.float() @ w.float().t(), rtol=2.0 ** -8, atol=2.0 ** -8 * 0.05 + 2.0 ** -17)
