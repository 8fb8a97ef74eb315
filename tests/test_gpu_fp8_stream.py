"""Block-scaled fp8 expert GEMMs through LDS-DMA (csrc/fp8_stream.hip): blocks of 16, 32 and 64 rows."""
import pytest
import torch

from semi_pd_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


# (one, two and three slots of K with an odd and an even count of scale blocks, more slots than the ring; columns that end inside a workgroup's;
# experts with no row, one, a full block and more; entries that are no prefix of a block)
@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("bm", [16, 32, 64])
@pytest.mark.parametrize("K,N,block_n", [(128, 16, 128), (256, 80, 16), (384, 144, 128), (640, 64, 64), (2048, 272, 128), (8192, 48, 128)])
def test_every_entry_against_its_products(K, N, block_n, bm, out_dtype):
    g = torch.Generator().manual_seed(K + bm)
    div, counts = 3, [1, 0, bm, bm + 1, 7, 15]
    total, E = sum(counts), len(counts)
    tokens = -(-total // div)
    q = lambda *s: (torch.randn(*s, generator=g) * 100).clamp(-448, 448).to(torch.float8_e4m3fn)               # noqa: E731
    a, w = q(tokens, K), q(E, N, K)
    KB, NB = K // 128, -(-N // block_n)
    a_s, w_s = torch.rand(tokens, KB, generator=g) + 0.5, torch.rand(E, NB, KB, generator=g) + 0.5
    weights = torch.rand(total, generator=g)
    perm = torch.randperm(total, generator=g)
    expert_of = torch.empty(total, dtype=torch.long)

    def blocks(rows):
        ids, experts, at = [], [], 0
        for e, n in enumerate(counts):
            mine = torch.full((-(-n // rows) * rows,), total, dtype=torch.int32)
            mine[mine.numel() - n:] = perm[at: at + n]                                                     # (padding in front)
            expert_of[perm[at: at + n]] = e
            at += n
            ids.append(mine)
            experts += [e] * (-(-n // rows))
        npp = torch.tensor([sum(i.numel() for i in ids)], dtype=torch.int32, device=DEV)
        ids = torch.cat(ids + [torch.full((rows,), total, dtype=torch.int32)])                             # (a block nobody routed to)
        return ids.to(DEV), torch.tensor(experts + [0], dtype=torch.int32, device=DEV), npp

    small, large = blocks(bm), blocks(128)
    row = torch.arange(total) // div
    part = torch.einsum("tkc,tnkc->tnk", a.double().view(tokens, KB, 128)[row], w.double().view(E, N, KB, 128)[expert_of])
    size = torch.einsum("tkc,tnkc->tnk", a.double().abs().view(tokens, KB, 128)[row], w.double().abs().view(E, N, KB, 128)[expert_of])
    scale = a_s.double()[row][:, None] * w_s.double()[expert_of].repeat_interleave(block_n, 1)[:, :N]
    want, size = (part * scale).sum(-1), (size * scale).sum(-1)
    half = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -24}[out_dtype]
    down = 2.0 ** -12 if out_dtype == torch.float16 else 1.0                                                # (fp16 holds up to 65504)
    d = lambda t: t.to(DEV)                                                                              # noqa: E731
    for scaled in (False, True):
        s = weights.double()[:, None] if scaled else 1.0
        got = []
        for (ids, experts, npp), rows in ((small, bm), (large, 128)):
            out = torch.full((total + 1, N), 77.0, dtype=out_dtype, device=DEV)
            ops.moe_grouped_gemm_fp8(d(a), d(a_s * down), d(w), d(w_s), out[:total], d(weights), ids, experts, npp, total, div, scaled,
                                     [block_n, 128], rows)
            assert bool((out[total] == 77).all())
            got.append(out[:total])
        # the form of 128 rows: the same sums of scale blocks, folded in with one or two roundings each and one of the result; and the value,
        # to what the matrix unit keeps of the sum of a scale block (the largest product's place and 13 bits behind it, 2^-12 of the sum at most)
        one, other = got[0].cpu().double(), got[1].cpu().double()
        assert bool(((one - other).abs() <= half * 2 * one.abs() + (2 * KB + 2) * 2.0 ** -24 * size * s * down + 2.0 ** -24).all())
        bound = (half * (want * s).abs() + 2.0 ** -11 * size * s) * down + 2.0 ** -24
        assert bool(((one - want * s * down).abs() <= bound).all())


def test_small_blocks_keep_to_their_shapes():
    a, w = torch.zeros(4, 192, device=DEV, dtype=torch.float8_e4m3fn), torch.zeros(2, 32, 192, device=DEV, dtype=torch.float8_e4m3fn)
    ids, experts = torch.zeros(32, dtype=torch.int32, device=DEV), torch.zeros(2, dtype=torch.int32, device=DEV)
    s = torch.ones(4, 2, device=DEV)
    with pytest.raises(RuntimeError):
        ops.moe_grouped_gemm_fp8(a, s, w, torch.ones(2, 1, 2, device=DEV), torch.empty(4, 32, device=DEV), None, ids, experts,
                                 torch.full((1,), 16, dtype=torch.int32, device=DEV), 4, 1, False, [128, 128], 16)
