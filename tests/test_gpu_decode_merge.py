"""The merge of a request's kv splits in one round trip (decode_merge.hip): numbers of splits around the forms' 8, 16 and 32, one and two
elements a thread, requests with fewer rows than splits or none, and anything in the places of splits without rows."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _truth(q, k, v, lens, slots, scale):
    out, at, group = [], 0, q.shape[1] // k.shape[1]
    for b, n in enumerate(lens):
        rows = slots[at: at + n].long()
        at += n
        if n == 0:
            out.append(torch.zeros(q.shape[1], v.shape[2], dtype=torch.float64))
            continue
        kk, vv = (t[rows].double().repeat_interleave(group, 1) for t in (k, v))
        p = torch.softmax(torch.einsum("hd,nhd->hn", q[b].double(), kk) * scale, -1)
        out.append(torch.einsum("hn,nhe->he", p, vv))
    return torch.stack(out)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("H,G,D,E", [(16, 1, 576, 512), (8, 2, 64, 64), (8, 2, 128, 128), (6, 2, 96, 96), (4, 4, 256, 256)])
def test_merge_of_the_splits(dtype, H, G, D, E):
    from semi_pd_amd import ops
    g = torch.Generator().manual_seed(D)
    lens = [1, 300, 5, 33, 0, 129]
    q = torch.randn(len(lens), H, D, generator=g).to(dtype)
    k = torch.randn(sum(lens) + 1, G, D, generator=g).to(dtype)
    v = k[..., :E] if D != E else torch.randn(sum(lens) + 1, G, E, generator=g).to(dtype)
    slots = (torch.randperm(sum(lens), generator=g) + 1).int()
    want = _truth(q, k, v, lens, slots, D ** -0.5)
    indptr = torch.tensor([0] + lens).cumsum(0).int().to(DEV)
    kd = k.to(DEV)
    vd = kd[..., :E] if D != E else v.to(DEV)
    for splits in (2, 3, 7, 8, 9, 15, 16, 17, 31, 32, 33):
        parts = torch.full((len(lens), H, splits, E + 1), float("nan"), device=DEV)
        out = torch.full((len(lens), H, E), 7.0, dtype=dtype, device=DEV)
        ops.decode_attention_fwd(q.to(DEV), kd, vd, out, indptr, slots.to(DEV), parts, splits, D ** -0.5)
        # weights and results are rounded to 16 bits: 2^-8 of the largest value (4.5 of them are normal) and of the result
        torch.testing.assert_close(out.cpu().double(), want, rtol=2.0 ** -7, atol=4.5 * 2.0 ** -8, msg=lambda m: f"{splits} splits: {m}")
