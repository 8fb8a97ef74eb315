"""Grouped tiled GEMM (csrc/gemm8p.hip) where experts end inside a row tile: the quadrants of padding that are left out and the order
in which the tiles of an expert are dealt out."""
import pytest
import torch

from semi_pd_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _routed(counts, bm, seed):
    """Blocks of bm entries, one expert each; the entries of an expert in no order, filled up with an id past the last."""
    g = torch.Generator().manual_seed(seed)
    total = sum(counts)
    ids, experts, at, perm = [], [], 0, torch.randperm(total, generator=g)
    for e, n in enumerate(counts):
        blocks = -(-n // bm)
        mine = torch.full((blocks * bm,), total, dtype=torch.int32)
        mine[:n] = perm[at: at + n]
        at += n
        ids.append(mine)
        experts += [e] * blocks
    return torch.cat(ids), torch.tensor(experts, dtype=torch.int32)


# (rows on both sides of a quadrant, a half and a whole tile; pairs of tiles of one expert at even and odd places, an odd last tile;
# columns in one, part of a group of eight and more tiles)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("bm", [128, 256])
@pytest.mark.parametrize("counts,K,n_out", [([1, 31, 32, 33, 64, 65, 95, 97, 127, 128, 129, 0, 192, 193, 255, 256, 257], 192, 48),
                                            ([300, 500, 20, 290, 513], 128, 1200), ([700], 64, 2320)])
def test_tail_tiles(counts, bm, K, n_out, dtype):
    g = torch.Generator().manual_seed(K)
    total, E = sum(counts), len(counts)
    ids, experts = _routed(counts, bm, K + bm)
    a = torch.randn(total, K, generator=g).to(dtype)
    w = (torch.randn(E, 2 * n_out, K, generator=g) * K ** -0.5).to(dtype)
    weights = torch.rand(total, generator=g)
    expert_of = torch.empty(total, dtype=torch.long)
    for b, e in enumerate(experts.tolist()):
        mine = ids[b * bm: (b + 1) * bm]
        expert_of[mine[mine < total].long()] = e
    want, size = torch.empty(total, 2 * n_out, dtype=torch.float64), torch.empty(total, 2 * n_out, dtype=torch.float64)
    for e in range(E):
        rows = expert_of == e
        want[rows] = a[rows].double() @ w[e].double().t()
        size[rows] = a[rows].abs().double() @ w[e].abs().double().t()
    d = lambda t: t.to(DEV)                                                                              # noqa: E731
    npp = torch.tensor([ids.numel()], dtype=torch.int32, device=DEV)
    ids = torch.cat([ids, torch.full((bm,), total, dtype=torch.int32)])                                  # (a block nobody routed to)
    experts = torch.cat([experts, torch.zeros(1, dtype=torch.int32)])
    half = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    for scaled in (False, True):
        out = torch.full((total + 1, 2 * n_out), 77.0, dtype=dtype, device=DEV)
        ops.moe_gemm_tall(d(a), d(w), out[:total], d(weights), d(ids), d(experts), npp, total, 1, scaled, False, block_m=bm)
        s = weights.double()[:, None] if scaled else 1.0
        # products are exact in fp32: K + 1 roundings of partial sums of at most `size`, one of the weight's product, one to the type
        bound = (half * (want * s).abs() + (K + 2) * 2.0 ** -24 * size * s) * 1.01 + 2.0 ** -24
        assert bool(((out[:total].cpu().double() - want * s).abs() <= bound).all())
        assert bool((out[total] == 77).all())
        if not scaled:
            plain = out[:total].clone()
    out = torch.full((total, n_out), 77.0, dtype=dtype, device=DEV)
    ops.moe_gemm_tall(d(a), d(w), out, None, d(ids), d(experts), npp, total, 1, False, True, block_m=bm)
    assert torch.equal(out, ops.silu_and_mul(plain))
