"""RoPE of prompt batches, two items a lane (csrc/rope_pairs.hip): the bits of the same rows in smaller batches, which a lane an item takes."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _inputs(T, Hq, Hk, D, dtype, gap, vhead):
    g = torch.Generator().manual_seed(T + Hq * D)
    width = Hq * D + Hk * D + Hk * vhead + gap
    return (torch.randn(T, width, generator=g).to(dtype).to(DEV), torch.randint(0, 3000, (T,), generator=g).to(DEV),
            torch.randn(3000, D, generator=g).to(DEV), (torch.randperm(T + 5, generator=g)[:T]).to(DEV))


# (heads: one workgroup's lanes not full, an odd number, one kv head, as many as fit into a workgroup and more; values of another size than keys)
@pytest.mark.parametrize("Hq,Hk,D,vhead", [(32, 8, 128, 128), (5, 1, 64, 64), (7, 7, 128, 32), (16, 1, 256, 256), (64, 32, 128, 128), (3, 1, 16, 24)])
@pytest.mark.parametrize("dtype,rows", [(torch.bfloat16, torch.bfloat16), (torch.float16, torch.float8_e4m3fn), (torch.bfloat16, torch.float8_e5m2),
                                        (torch.float32, torch.float32)])
def test_bits_of_smaller_batches(Hq, Hk, D, vhead, dtype, rows):
    from semi_pd_amd import ops
    T = 1027
    qkv, pos, cache, loc = _inputs(T, Hq, Hk, D, dtype, 8, vhead)

    def run(step):
        x = qkv.clone()
        k_pool, v_pool = (torch.zeros(T + 5, Hk, d, device=DEV, dtype=dtype).to(rows) for d in (D, vhead))
        for t in range(0, T, step):
            q, k, v, _ = x[t: t + step].split([Hq * D, Hk * D, Hk * vhead, 8], 1)
            ops.rope_and_store_kv(pos[t: t + step], q, k, v, D, cache, True, k_pool, v_pool, loc[t: t + step])
        return x, k_pool, v_pool

    for a, b in zip(run(T), run(500)):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))


def test_without_pools():
    from semi_pd_amd import ops
    T, Hq, Hk, D = 1500, 12, 4, 64
    qkv, pos, cache, _ = _inputs(T, Hq, Hk, D, torch.bfloat16, 0, D)
    out = []
    for step in (T, 700):
        q, k = qkv[:, : Hq * D].clone(), qkv[:, Hq * D: (Hq + Hk) * D].clone()
        for t in range(0, T, step):
            ops.apply_rope_with_cos_sin_cache_inplace(pos[t: t + step], q[t: t + step], k[t: t + step], D, cache, True)
        out.append((q, k))
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1])
    assert not torch.equal(out[0][0], qkv[:, : Hq * D])
