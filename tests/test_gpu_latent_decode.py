"""Decode attention over latent rows with up to 16 heads: lengths around a tile of 32 rows and around two of them in flight."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
LENS = [1, 31, 32, 33, 63, 64, 65, 96, 97, 130]


def _run(heads, splits, dtype):
    from semi_pd_amd import ops
    g = torch.Generator(device=DEV).manual_seed(heads * 10 + splits)
    total = sum(LENS)
    slots = torch.randperm(total, generator=g, device=DEV).int() + 1
    kv = torch.randn(total + 1, 1, 576, generator=g, device=DEV).to(dtype)
    q = torch.randn(len(LENS), heads, 576, generator=g, device=DEV).to(dtype)
    indptr = torch.tensor([0] + LENS, device=DEV).cumsum(0).int()
    out = torch.full((len(LENS), heads, 512), 7.0, device=DEV, dtype=dtype)
    parts = torch.empty(len(LENS), heads, splits, 513, device=DEV) if splits > 1 else None
    ops.decode_attention_fwd(q, kv, kv[..., :512], out, indptr, slots, parts, splits, 192 ** -0.5)
    want = torch.empty(len(LENS), heads, 512, dtype=torch.float64)
    for b, n in enumerate(LENS):
        rows = kv[slots[indptr[b]: indptr[b + 1]].long(), 0].double().cpu()
        p = torch.softmax(q[b].double().cpu() @ rows.t() * 192 ** -0.5, -1)
        want[b] = p @ rows[:, :512]
    return out.double().cpu(), want


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("splits", [1, 3, 8])
@pytest.mark.parametrize("heads", [1, 16])
def test_lengths_around_tiles(heads, splits, dtype):
    """The weights are rounded to the type once (half a unit, 2^-8 of one just above a power of two in bf16) against values of at most 5,
    and so is the result."""
    got, want = _run(heads, splits, dtype)
    half = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    torch.testing.assert_close(got, want, rtol=half, atol=5 * half)


@pytest.mark.parametrize("splits", [1, 3])
def test_infinity_in_the_last_row_of_a_request(splits):
    """It is in its column of its request alone: rows that stand in for those behind the end count for nothing."""
    column, last = 37, sum(LENS[:4]) - 1

    # (the scores of that row are infinite where the query's element is positive: keys without the column's part)
    from semi_pd_amd import ops
    g = torch.Generator(device=DEV).manual_seed(3)
    total = sum(LENS)
    slots = torch.arange(1, total + 1, device=DEV).int()
    kv = torch.randn(total + 1, 1, 576, generator=g, device=DEV).bfloat16()
    q = torch.randn(len(LENS), 16, 576, generator=g, device=DEV).bfloat16()
    q[:, :, column] = -0.5
    kv[slots[last].long(), 0, column] = float("inf")
    indptr = torch.tensor([0] + LENS, device=DEV).cumsum(0).int()
    out = torch.empty(len(LENS), 16, 512, device=DEV, dtype=torch.bfloat16)
    parts = torch.empty(len(LENS), 16, splits, 513, device=DEV) if splits > 1 else None
    ops.decode_attention_fwd(q, kv, kv[..., :512], out, indptr, slots, parts, splits, 192 ** -0.5)
    out = out.float().cpu()
    assert bool(torch.isfinite(out[torch.arange(len(LENS)) != 3]).all())
    keep = torch.arange(512) != column
    assert bool(torch.isfinite(out[3][:, keep]).all()) and not bool(torch.isfinite(out[3][:, column]).any())


@pytest.mark.parametrize("cap", [0.0, 3.0])
@pytest.mark.parametrize("rows", ["same", "e4m3", "e5m2"])
@pytest.mark.parametrize("heads", [5, 16])
def test_rows_of_every_type_and_capped_scores(heads, rows, cap):
    """Lengths that end in every place of a wave's eight rows, the last row of a tile among them; weights and result are rounded to bf16
    (see above), values are at most 6.  An fp8 row is exact in bf16."""
    from semi_pd_amd import ops
    lens = [8, 15, 23, 40, 57, 64, 95, 161]
    g = torch.Generator(device=DEV).manual_seed(heads)
    total = sum(lens)
    kind = {"same": torch.bfloat16, "e4m3": torch.float8_e4m3fn, "e5m2": torch.float8_e5m2}[rows]
    kv = torch.randn(total + 1, 1, 576, generator=g, device=DEV).to(kind)
    slots = torch.randperm(total, generator=g, device=DEV).int() + 1
    q = torch.randn(len(lens), heads, 576, generator=g, device=DEV).bfloat16()
    indptr = torch.tensor([0] + lens, device=DEV).cumsum(0).int()
    out = torch.empty(len(lens), heads, 512, device=DEV, dtype=torch.bfloat16)
    ops.decode_attention_fwd(q, kv, kv[..., :512], out, indptr, slots, None, 1, 192 ** -0.5, cap)
    parts = torch.empty(len(lens), heads, 3, 513, device=DEV)
    split = torch.empty_like(out)
    ops.decode_attention_fwd(q, kv, kv[..., :512], split, indptr, slots, parts, 3, 192 ** -0.5, cap)
    for b, n in enumerate(lens):
        r = kv[slots[indptr[b]: indptr[b + 1]].long(), 0].double().cpu()
        s = q[b].double().cpu() @ r.t() * 192 ** -0.5
        want = torch.softmax(cap * torch.tanh(s / cap) if cap else s, -1) @ r[:, :512]
        for got in (out, split):
            torch.testing.assert_close(got[b].double().cpu(), want, rtol=2.0 ** -8, atol=6 * 2.0 ** -8)
