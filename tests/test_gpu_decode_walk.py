"""Paged decode attention of grouped heads on the matrix cores (csrc/decode_mfma_walk.h) against a softmax in 64 bits, at the edges of its tiles
of 32 tokens and of its splits."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("rows", [torch.bfloat16, torch.float8_e4m3fn])
@pytest.mark.parametrize("H,G,D", [(8, 2, 128), (12, 4, 64), (16, 1, 128), (32, 1, 64), (10, 5, 96)])
@pytest.mark.parametrize("splits", [1, 3, 8])
@pytest.mark.parametrize("cap", [0.0, 2.0])
def test_decode_at_the_edges_of_tiles(rows, H, G, D, splits, cap):
    """Requests of one token, around whole tiles, shorter than their splits, and none; rows that belong to no request hold no numbers, and
    neither a tile's unused rows nor the row behind the last reach the result.  Weights are rounded to 16 bits once and so is the result:
    1.5 units of half a unit in the last place, as for prompts."""
    from semi_pd_amd import ops
    lens = [1, 2, 31, 32, 33, 0, 64, 65, 97, 200, 7]
    g = torch.Generator().manual_seed(H * D + splits)
    total = sum(lens)
    k, v = (torch.full((2 * total + 2, G, D), float("nan")) for _ in range(2))
    slots = torch.randperm(2 * total + 1, generator=g)[:total] + 1
    k[slots], v[slots] = torch.randn(total, G, D, generator=g), torch.randn(total, G, D, generator=g)
    k, v, q = k.to(rows), v.to(rows), torch.randn(len(lens), H, D, generator=g).bfloat16()
    starts = [0]
    for n in lens:
        starts.append(starts[-1] + n)
    out = torch.full((len(lens), H, D), 7.0, dtype=torch.bfloat16, device=DEV)
    parts = torch.empty(len(lens), H, splits, D + 1, device=DEV) if splits > 1 else None
    scale = D ** -0.5
    ops.decode_attention_fwd(q.to(DEV), k.to(DEV), v.to(DEV), out, torch.tensor(starts, dtype=torch.int32, device=DEV), slots.int().to(DEV), parts, splits,
                             scale, cap)
    got, want = out.cpu().double(), torch.zeros(len(lens), H, D, dtype=torch.float64)
    for b, n in enumerate(lens):
        at = slots[starts[b]: starts[b + 1]]
        for h in range(H):
            if n:
                s = k[at, h // (H // G)].double() @ q[b, h].double() * scale
                want[b, h] = torch.softmax(cap * torch.tanh(s / cap) if cap else s, 0) @ v[at, h // (H // G)].double()
    some = [b for b, n in enumerate(lens) if n]
    assert bool((got[lens.index(0)] == 0).all())
    ulp = 2.0 ** -8
    assert float((got[some] - want[some]).norm() / want[some].norm()) < 1.5 * ulp
    torch.testing.assert_close(got[some], want[some], rtol=6 * ulp, atol=12 * ulp)


@pytest.mark.parametrize("H,G,D,K", [(32, 8, 128, 4096), (32, 8, 64, 2048), (12, 6, 64, 768)])
@pytest.mark.parametrize("splits", [1, 2, 3, 5, 7, 8])
@pytest.mark.parametrize("rows", [torch.bfloat16, torch.float8_e4m3fn])
def test_one_launch_with_fewer_splits_than_waves_has_the_bits_of_three(H, G, D, K, splits, rows):
    """The one-launch form at the kv splits of the launches that it stands for: the same ranges of every request, so the same bits and the
    same pool rows, also of requests with fewer tokens than ranges and on the edges of ranges and tiles."""
    from semi_pd_amd import ops
    lens = [1, 2, splits, 8 * splits + 1, 32 * splits, 333, 32 * splits + 1]
    B, total = len(lens), sum(lens)
    g = torch.Generator().manual_seed(H + D + splits)
    ends = torch.cumsum(torch.tensor(lens), 0)
    starts = torch.cat([torch.zeros(1, dtype=torch.int64), ends]).int().to(DEV)
    slots = (torch.randperm(total + 9, generator=g)[:total] + 1).int()
    k, v = (torch.randn(total + 10, G, D, generator=g).bfloat16().to(rows).to(DEV) for _ in range(2))
    loc, slots = slots[ends - 1].long().to(DEV), slots.to(DEV)
    x, w = torch.randn(B, K, generator=g).bfloat16().to(DEV), (torch.randn((H + 2 * G) * D, K, generator=g) * 0.03).bfloat16().to(DEV)
    angles = torch.arange(1024.0)[:, None] * 10000.0 ** (-torch.arange(0, D, 2) / D)
    table, pos = torch.cat([angles.cos(), angles.sin()], 1).to(DEV), (torch.tensor(lens) - 1).to(DEV)
    k1, v1, k2, v2 = k.clone(), v.clone(), k.clone(), v.clone()
    q = ops.rope_and_store_kv_planes(pos, ops.stream_linear_planes(x, w), H, G, D, table, k1, v1, loc)
    want = torch.empty(B, H, D, dtype=torch.bfloat16, device=DEV)
    parts = torch.empty(B, H, splits, D + 1, device=DEV) if splits > 1 else None
    ops.decode_attention_fwd(q.view(B, H, D), k1, v1, want, starts, slots, parts, splits, D ** -0.5)
    got = ops.decode_rope_attention_planes(pos, ops.stream_linear_planes(x, w), H, G, D, table, k2, v2, loc, starts, slots, 8, D ** -0.5,
                                           num_kv_splits=splits)
    assert torch.equal(k1.view(torch.uint8), k2.view(torch.uint8)) and torch.equal(v1.view(torch.uint8), v2.view(torch.uint8))
    assert torch.equal(got.view(torch.int16), want.view(B, H * D).view(torch.int16))


@pytest.mark.parametrize("H,G,D,B", [(32, 8, 64, 150), (48, 8, 96, 131), (16, 4, 64, 280)])
def test_walk_that_pauses_has_the_bits_of_the_one_that_goes_on(H, G, D, B):
    """Between one and two workgroups a CU heads of up to 96 take the other walk: the same bits as in two calls of half the requests."""
    from semi_pd_amd import ops
    lens = [1 + (i * 37) % 131 for i in range(B)]
    g = torch.Generator().manual_seed(D + B)
    ends = torch.cumsum(torch.tensor(lens), 0)
    starts = torch.cat([torch.zeros(1, dtype=torch.int64), ends]).int()
    total = int(ends[-1])
    slots = (torch.randperm(total + 9, generator=g)[:total] + 1).int().to(DEV)
    k, v = (torch.randn(total + 10, G, D, generator=g).bfloat16().to(DEV) for _ in range(2))
    q = torch.randn(B, H, D, generator=g).bfloat16().to(DEV)

    def run(lo, hi):
        out = torch.empty(hi - lo, H, D, dtype=torch.bfloat16, device=DEV)
        ops.decode_attention_fwd(q[lo:hi], k, v, out, starts[lo: hi + 1].to(DEV), slots, None, 1, D ** -0.5)
        return out
    assert torch.equal(run(0, B).view(torch.int16), torch.cat([run(0, B // 2), run(B // 2, B)]).view(torch.int16))
