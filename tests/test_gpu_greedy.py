"""Greedy tokens of rows around the pieces that a thread has under way at once (argmax_kernel)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# (a row's pieces: fewer than threads, four a thread, one more, a remainder that is no piece; rows off a 16-byte boundary)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("vocab", [1, 7, 1000, 8192, 16384, 16389, 24576, 32768, 32776, 65537])
def test_greedy_token(dtype, vocab):
    from semi_pd_amd import ops
    g = torch.Generator().manual_seed(vocab)
    x = torch.randn(6, vocab, generator=g).to(dtype)
    x[1] = 0.5                                                      # all equal: the first
    x[2] = float("-inf")
    x[3, vocab // 2:] = float("inf")                                # the first of the largest
    x[4] = float("nan")
    x[5, : vocab // 3] = float("nan")
    want = []
    for row in x.float():
        best, at = float("-inf"), -1
        vals = row.nan_to_num(nan=float("-inf"), posinf=float("inf"), neginf=float("-inf"))
        ok = ~row.isnan()
        if bool(ok.any()):
            best = float(vals[ok].max())
            at = int((ok & (row == best)).nonzero()[0])
        want.append(max(at, 0))
    assert ops.greedy_argmax(x.to(DEV)).cpu().tolist() == want
    wide = torch.zeros(6, vocab + 1, dtype=dtype)
    wide[:, 1:] = x
    assert ops.greedy_argmax(wide.to(DEV)[:, 1:]).cpu().tolist() == want


# (a row each CU and more: narrower workgroups; values with many equals, the first of which is wanted, and a few rows without any value)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,vocab", [(255, 24576), (256, 24576), (256, 24581), (300, 65528), (256, 65536)])
def test_greedy_tokens_of_many_rows(dtype, rows, vocab):
    from semi_pd_amd import ops
    g = torch.Generator().manual_seed(rows + vocab)
    x = torch.randint(-40, 41, (rows, vocab), generator=g).to(dtype)
    x[3] = float("-inf")
    x[5] = float("nan")
    x[7, : vocab - 1] = float("nan")
    want = x.float().nan_to_num(nan=float("-inf")).numpy().argmax(1).tolist()
    want[5] = 0
    assert ops.greedy_argmax(x.to(DEV)).cpu().tolist() == want
