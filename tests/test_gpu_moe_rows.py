"""Grouped GEMM of up to 320 routed rows a workgroup (csrc/moe_gemm_rows.h): a body for every 64 rows from 128 on."""
import pytest
import torch

from semi_pd_amd import ops
from test_gpu_moe_tail_tiles import _routed

pytestmark = pytest.mark.gpu
DEV = "cuda"
BM = 320


# (rows around every body's most, a whole tile and one more; two steps of K and an uneven count of pairs; columns that end inside a tile; few last
# row tiles among many, behind the others, on both sides of 64 of them; more than 256 row tiles; row tiles in turns within many column tiles)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("counts,K,n_out,div", [([1, 16, 17, 127, 128, 129, 0, 160, 192, 193, 255, 256, 257, 319, 320, 321, 640], 128, 48, 1),
                                                ([300, 500, 20, 290, 1000], 384, 1200, 5), ([96, 200], 640, 2320, 2),
                                                ([5] * 30 + [330] + [3] * 31 + [340, 0, 350, 9] + [2] * 8, 128, 304, 1), ([1] * 250 + [400, 2, 3, 0, 2000], 128, 32, 1),
                                                ([700, 30, 2900], 128, 2320, 1)])
def test_rows_of_every_body(counts, K, n_out, div, dtype):
    g = torch.Generator().manual_seed(K)
    total, E = sum(counts), len(counts)
    ids, experts = _routed(counts, BM, K)
    tokens = -(-total // div)
    a = torch.randn(tokens, K, generator=g).to(dtype)
    w = (torch.randn(E, 2 * n_out, K, generator=g) * K ** -0.5).to(dtype)
    weights = torch.rand(total, generator=g)
    expert_of = torch.empty(total, dtype=torch.long)
    for b, e in enumerate(experts.tolist()):
        mine = ids[b * BM: (b + 1) * BM]
        expert_of[mine[mine < total].long()] = e
    want, size = torch.empty(total, 2 * n_out, dtype=torch.float64), torch.empty(total, 2 * n_out, dtype=torch.float64)
    rows = a[torch.arange(total) // div]
    for e in range(E):
        mine = expert_of == e
        want[mine] = rows[mine].double() @ w[e].double().t()
        size[mine] = rows[mine].abs().double() @ w[e].abs().double().t()
    d = lambda t: t.to(DEV)                                                                              # noqa: E731
    npp = torch.tensor([ids.numel()], dtype=torch.int32, device=DEV)
    ids = torch.cat([ids, torch.full((BM,), total, dtype=torch.int32)])                                  # (a block nobody routed to)
    experts = torch.cat([experts, torch.zeros(1, dtype=torch.int32)])
    half = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    for scaled in (False, True):
        out = torch.full((total + 1, 2 * n_out), 77.0, dtype=dtype, device=DEV)
        ops.moe_gemm_tall(d(a), d(w), out[:total], d(weights), d(ids), d(experts), npp, total, div, scaled, False, block_m=BM)
        s = weights.double()[:, None] if scaled else 1.0
        # products are exact in fp32: K + 1 roundings of partial sums of at most `size`, one of the weight's product, one to the type
        bound = (half * (want * s).abs() + (K + 2) * 2.0 ** -24 * size * s) * 1.01 + 2.0 ** -24
        assert bool(((out[:total].cpu().double() - want * s).abs() <= bound).all())
        assert bool((out[total] == 77).all())
        if not scaled:
            plain = out[:total].clone()
    out = torch.full((total, n_out), 77.0, dtype=dtype, device=DEV)
    ops.moe_gemm_tall(d(a), d(w), out, None, d(ids), d(experts), npp, total, div, False, True, block_m=BM)
    assert torch.equal(out, ops.silu_and_mul(plain))


@pytest.mark.parametrize("n_out", [304, 2320])                                                          # few and many column tiles
def test_no_entry_is_one_of_the_experts(n_out):
    """A rank whose experts no token takes: nothing is written, and in front of the blocks there are nothing is read either (expert_ids is the
    start of its allocation)."""
    E, K, total = 4, 128, 700
    ids = torch.full((2 * BM,), total, dtype=torch.int32, device=DEV)
    experts, none = torch.full((2,), 1 << 30, dtype=torch.int32, device=DEV), torch.zeros(1, dtype=torch.int32, device=DEV)
    a, w = torch.ones(total, K, dtype=torch.bfloat16, device=DEV), torch.ones(E, 2 * n_out, K, dtype=torch.bfloat16, device=DEV)
    for fused in (False, True):
        out = torch.full((total, n_out if fused else 2 * n_out), 77.0, dtype=torch.bfloat16, device=DEV)
        ops.moe_gemm_tall(a, w, out, None, ids, experts, none, total, 1, False, fused, block_m=BM)
        assert bool((out == 77).all())


def test_layer_of_a_rank_that_no_token_routes_to():
    """The layer of such a rank is zero, in the blocks of up to 320 rows as in the others."""
    from semi_pd_amd.layers import moe
    E, K, F, T, top = 16, 512, 1024, 1200, 6
    assert moe._tall_block(256, T, top, E, K, F) == BM
    x = torch.randn(T, K, device=DEV).bfloat16()
    w1, w2 = torch.randn(E, 2 * F, K, device=DEV).bfloat16(), torch.randn(E, K, F, device=DEV).bfloat16()
    ids = torch.arange(T * top, device=DEV, dtype=torch.int32).view(T, top) % 16                          # of the first rank's experts
    out = moe.fused_experts(x, w1, w2, torch.rand(T, top, device=DEV), ids, expert_offset=48, partial_experts=True)
    assert bool((out == 0).all())
