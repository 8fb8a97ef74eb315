"""Block-scaled fp8 expert GEMMs in blocks of 128 rows (csrc/fp8_rows.hip; fused_moe_triton/fused_moe.py:174-243)."""
import pytest
import torch

from semi_pd_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


# (one to five scale blocks of K around the three in turn, and many; columns of one group, of a workgroup and a rest; experts whose rows fill one half of
# a block, a row more, a block, a row more; an expert with none)
@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("K,N,block_n", [(128, 16, 128), (256, 256, 128), (384, 272, 16), (512, 48, 48), (640, 400, 128), (1408, 528, 128)])
def test_blocks_of_128_rows_against_their_products(K, N, block_n, out_dtype):
    g = torch.Generator().manual_seed(K + N)
    div, counts = 3, [1, 64, 65, 0, 128, 129]
    total, E, KB, NB = sum(counts), len(counts), K // 128, -(-N // block_n)
    tokens = -(-total // div)
    q = lambda *s: (torch.randn(*s, generator=g) * 100).clamp(-448, 448).to(torch.float8_e4m3fn)               # noqa: E731
    a, w = q(tokens, K), q(E, N, K)
    a_s, w_s = torch.rand(tokens, KB, generator=g) + 0.5, torch.rand(E, NB, KB, generator=g) + 0.5
    weights = torch.rand(total, generator=g)
    perm, expert_of, ids, experts, at = torch.randperm(total, generator=g), torch.empty(total, dtype=torch.long), [], [], 0
    for e, n in enumerate(counts):
        mine = torch.full((-(-n // 128) * 128,), total, dtype=torch.int32)
        mine[:n] = perm[at: at + n]
        expert_of[perm[at: at + n]] = e
        at += n
        ids.append(mine)
        experts += [e] * (-(-n // 128))
    npp = torch.tensor([sum(i.numel() for i in ids)], dtype=torch.int32, device=DEV)
    ids = torch.cat(ids + [torch.full((100,), total, dtype=torch.int32)])                                     # (room that nobody needs, no whole block)
    row = torch.arange(total) // div
    x, y = a.double().view(tokens, KB, 128)[row], w.double().view(E, N, KB, 128)[expert_of]
    scale = a_s.double()[row][:, None] * w_s.double()[expert_of].repeat_interleave(block_n, 1)[:, :N]
    want = (torch.einsum("tkc,tnkc->tnk", x, y) * scale).sum(-1)
    size = (torch.einsum("tkc,tnkc->tnk", x.abs(), y.abs()) * scale).sum(-1)
    half = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -24}[out_dtype]
    down = 2.0 ** -12 if out_dtype == torch.float16 else 1.0                                                # (fp16 holds up to 65504)
    d = lambda t: t.to(DEV)                                                                              # noqa: E731
    for scaled in (False, True):
        s = weights.double()[:, None] if scaled else 1.0
        out = torch.full((total + 1, N), 77.0, dtype=out_dtype, device=DEV)
        ops.moe_grouped_gemm_fp8(d(a), d(a_s * down), d(w), d(w_s), out[:total], d(weights), d(ids), d(torch.tensor(experts, dtype=torch.int32)), npp, total,
                                 div, scaled, [block_n, 128], 128)
        assert bool((out[total] == 77).all())
        # one rounding of the result, and what the matrix unit keeps of the sum of a scale block (the largest product's place and 13 bits behind
        # it: 2^-12 of the sum at most)
        bound = (half * (want * s).abs() + 2.0 ** -11 * size * s) * down + 2.0 ** -24
        assert bool(((out[:total].cpu().double() - want * s * down).abs() <= bound).all())


@pytest.mark.parametrize("last", [1, 40, 64, 65, 127])
def test_a_last_block_that_is_not_whole(last):
    """Entries and their count end within a block: its rows are multiplied, and nothing behind them is read."""
    g = torch.Generator().manual_seed(last)
    E, K, N, total = 2, 256, 272, 128 + last
    a, w = (torch.randn(*s, generator=g).to(torch.float8_e4m3fn).to(DEV) for s in ((total, K), (E, N, K)))
    a_s, w_s = (torch.rand(*s, generator=g).to(DEV) for s in ((total, K // 128), (E, -(-N // 128), K // 128)))
    experts = torch.tensor([1, 0], dtype=torch.int32, device=DEV)
    ids = torch.randperm(total, generator=g).int()
    outs = []
    for entries in (ids, torch.cat([ids, torch.full((256 - total,), total, dtype=torch.int32)])):
        memory = torch.zeros(256 + 128, dtype=torch.int32, device=DEV)                        # (behind the entries: row 0 of the result)
        memory[: entries.numel()] = entries.to(DEV)
        out = torch.full((total, N), 77.0, dtype=torch.bfloat16, device=DEV)
        ops.moe_grouped_gemm_fp8(a, a_s, w, w_s, out, None, memory[: entries.numel()], experts,
                                 torch.tensor([entries.numel()], dtype=torch.int32, device=DEV), total, 1, False, [128, 128], 128)
        outs.append(out)
    assert torch.equal(*outs)


def test_column_tiles_of_large_experts():
    """Experts of more than 24 MB take their column tiles in groups, 49 of them here and the last of one tile: the bits of the two halves of
    their columns, which are below that."""
    g = torch.Generator(device=DEV).manual_seed(3)
    E, K, N, at, counts = 2, 256, 98432, 49152, [129, 40]
    total = sum(counts)
    q = lambda *s: torch.randn(*s, generator=g, device=DEV).to(torch.float8_e4m3fn)                           # noqa: E731
    a, w = q(total, K), q(E, N, K)
    a_s, w_s = (torch.rand(*s, generator=g, device=DEV) for s in ((total, K // 128), (E, N // 128, K // 128)))
    ids = torch.full((384,), total, dtype=torch.int32, device=DEV)
    ids[:129], ids[256: 296] = torch.arange(129, device=DEV).int(), torch.arange(129, total, device=DEV).int()
    experts, npp = torch.tensor([1, 1, 0], dtype=torch.int32, device=DEV), torch.tensor([384], dtype=torch.int32, device=DEV)

    def run(lo, hi):
        out = torch.full((total, hi - lo), 77.0, dtype=torch.bfloat16, device=DEV)
        ops.moe_grouped_gemm_fp8(a, a_s, w[:, lo:hi].contiguous(), w_s[:, lo // 128: hi // 128].contiguous(), out, None, ids, experts, npp, total, 1, False,
                                 [128, 128], 128)
        return out
    assert torch.equal(run(0, N), torch.cat([run(0, at), run(at, N)], 1))
