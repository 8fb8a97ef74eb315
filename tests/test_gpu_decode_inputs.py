"""What a captured decode step reads of its batch, copied in one launch."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("batch,rows", [(1, 1), (3, 4), (5, 300), (256, 256), (257, 300)])
@pytest.mark.parametrize("state", [True, False])
def test_inputs_of_a_captured_step(batch, rows, state):
    from semi_pd_amd import ops
    g = torch.Generator().manual_seed(batch)
    own = [torch.full((rows + 2,), 7 + i, dtype=torch.int64, device=DEV) for i in range(5)]
    src = [torch.randint(1, 1 << 40, (batch,), generator=g).to(DEV) for _ in range(5 if state else 4)] + ([] if state else [None])
    assert ops.decode_inputs(own, src, rows, 9)
    for i, (got, want, pad) in enumerate(zip(own, src, (None, 0, 9, 0, 0))):
        got = got.cpu()
        if want is not None:
            assert torch.equal(got[:batch], want.cpu())
        else:                                                       # (no state rows of an earlier step)
            assert bool((got[:batch] == 0).all())
        assert bool((got[batch: rows] == (7 + i if pad is None else pad)).all()) and bool((got[rows:] == 7 + i).all())


def test_inputs_of_another_kind_are_left_to_copies():
    from semi_pd_amd import ops
    own = [torch.full((4,), 7, dtype=torch.int64, device=DEV) for _ in range(5)]
    good = [torch.ones(2, dtype=torch.int64, device=DEV) for _ in range(5)]
    for bad in (torch.ones(2, dtype=torch.int32, device=DEV), torch.ones(2, dtype=torch.int64), torch.ones(4, dtype=torch.int64, device=DEV)[::2]):
        for at in range(5):
            assert not ops.decode_inputs(own, good[:at] + [bad] + good[at + 1:], 4, 1)
    assert all(bool((t == 7).all()) for t in own)
