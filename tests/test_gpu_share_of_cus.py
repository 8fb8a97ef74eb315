"""Launches whose form counts on a CU for every workgroup, where the process has told a share of the CUs (semipd_gemm_tall_set_cus)."""
import contextlib

import pytest
import torch

from test_gpu_prompt_attention import _batch
from test_gpu_recurrence_chunks import _delta_inputs, _delta_run, _ssm_inputs, _ssm_run

pytestmark = pytest.mark.gpu
DEV = "cuda"


@contextlib.contextmanager
def _share(cus):
    from semi_pd_amd import _lib
    lib = _lib.load()
    _lib.check(lib.semipd_gemm_tall_set_cus(cus), "set_cus")
    try:
        yield
    finally:
        _lib.check(lib.semipd_gemm_tall_set_cus(256), "set_cus")


@pytest.mark.parametrize("kind", ["state_space", "delta_rule"])
def test_columns_of_a_workgroup_follow_the_share(kind):
    """256 workgroups of 32 columns are one round of the whole chip and two of half of it: there the request has the 64 columns a workgroup, and
    the bits, that it has next to another one."""
    H, G, N, E, lens = 64, 8, 128, 128, [97, 65]
    inputs, run, extra = (_ssm_inputs, _ssm_run, (H,)) if kind == "state_space" else (_delta_inputs, _delta_run, ())
    w, rows, state, before = inputs(H, G, N, E, 4, lens, torch.bfloat16, 5)
    both, both_state, _ = run(w, rows, state, before, [9, 9], H, G, N, E, *extra)
    one = (w, rows[:1], state[:1], before[:1], [9], H, G, N, E, *extra)
    with _share(128):
        half, half_state, _ = run(*one)
    assert torch.equal(half[0], both[0]) and torch.equal(half_state[0], both_state[0])
    whole, whole_state, _ = run(*one)
    assert not (torch.equal(whole[0], both[0]) and torch.equal(whole_state[0], both_state[0]))             # (the other form sums in another order)


@pytest.mark.parametrize("D,tokens,share", [(128, 300, 64), (64, 933, 128), (128, 1500, 160)])
def test_groups_of_waves_follow_the_share(D, tokens, share):
    """A prompt whose tiles have a CU each, or two of them one, on the whole chip and not on the share: there it has the bits of a batch in
    which a tile's steps are one group's."""
    from semi_pd_amd import ops
    H, G, lens = 32, 8, [tokens, 1100, 1300]
    t, _ = _batch(lens, [0, 0, 0], H, G, D, D, torch.bfloat16, D)
    d = {k: v.to(DEV) for k, v in t.items() if k != "totals"}

    def run(n):
        start = torch.tensor([0] + lens[:-1], dtype=torch.int32).cumsum(0).int()[:n]
        out = torch.empty(sum(lens[:n]), H * D, dtype=torch.bfloat16, device=DEV)
        ops.local_attention_fwd(d["q"][: sum(lens[:n])], out, d["k"], d["v"], d["table"], torch.arange(n, device=DEV),
                                torch.tensor(t["totals"][:n], device=DEV), start.to(DEV), torch.tensor(lens[:n], dtype=torch.int32, device=DEV),
                                max(lens[:n]), D ** -0.5, 0.0, 0, None, None)
        return out[:tokens]
    many = run(3)
    with _share(share):
        assert torch.equal(run(1), many)
    assert not torch.equal(run(1), many)


def test_many_short_tiles_have_one_group_each():
    """Two prompts of 600 tokens, 40 / 8 heads: 440 tiles, whose rows have the bits that they have in a batch whose tiles are one group's."""
    from semi_pd_amd import ops
    H, G, D, lens = 40, 8, 128, [600, 600, 600, 700]
    t, _ = _batch(lens, [0] * 4, H, G, D, D, torch.bfloat16, D)
    d = {k: v.to(DEV) for k, v in t.items() if k != "totals"}

    def run(n):
        start = torch.tensor([0] + lens[:-1], dtype=torch.int32).cumsum(0).int()[:n]
        out = torch.empty(sum(lens[:n]), H * D, dtype=torch.bfloat16, device=DEV)
        ops.local_attention_fwd(d["q"][: sum(lens[:n])], out, d["k"], d["v"], d["table"], torch.arange(n, device=DEV),
                                torch.tensor(t["totals"][:n], device=DEV), start.to(DEV), torch.tensor(lens[:n], dtype=torch.int32, device=DEV),
                                max(lens[:n]), D ** -0.5, 0.0, 0, None, None)
        return out[: 2 * 600]
    assert torch.equal(run(2), run(4))
