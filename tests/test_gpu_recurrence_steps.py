"""Decode steps of the recurrences where a workgroup's convolution channels meet the two a thread that are fetched in front of the state:
as many, fewer and more of them, and more taps than that form has (ssm_step_kernel, delta_step_kernel)."""
import pytest
import torch

import test_gpu_recurrence_chunks as steps

pytestmark = pytest.mark.gpu


# (channels of a workgroup of 256: 512, 504, 576, 40, 192, 576; taps in and beyond the early form)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,G,N,E,taps", [(6, 2, 240, 32, 3), (12, 1, 244, 16, 4), (4, 2, 256, 64, 4), (300, 4, 4, 32, 4), (10, 2, 64, 64, 5), (4, 2, 256, 64, 7)])
def test_state_space_step_channels(dtype, H, G, N, E, taps):
    steps.test_state_space_decode_step(dtype, H, G, N, E, taps, 1)


# (2 D + E H / G channels: 2336 for 512 threads, 1024 for 512, 384 for 1024, a head each of several workgroups; taps in and beyond the early form)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,G,D,E,taps", [(774, 86, 16, 256, 4), (6, 1, 128, 128, 4), (4, 1, 64, 64, 3), (24, 1, 128, 64, 4), (774, 86, 16, 256, 6), (8, 2, 128, 128, 5)])
def test_delta_rule_step_channels(dtype, H, G, D, E, taps):
    steps.test_delta_rule_decode_step(dtype, H, G, D, E, taps)


# (the form of two taps: a channel left over for a third thread, fewer than threads, a head each of several workgroups)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,G,D,E", [(774, 86, 16, 256), (4, 1, 64, 64), (24, 1, 128, 64), (4, 2, 128, 128)])
def test_delta_rule_step_of_two_taps(dtype, H, G, D, E):
    steps.test_delta_rule_decode_step(dtype, H, G, D, E, 2)


def _step_call(kind, T, g, dtype=torch.bfloat16):
    """ops.<kind> and the arguments of a decode batch of T requests, by name."""
    from semi_pd_amd import ops
    r = lambda *n, dt=torch.float32: torch.randn(*n, generator=g).to(dt).cuda()
    idx, lens = torch.arange(1, T + 1).cuda(), torch.arange(1, T + 1).cuda()
    if kind == "delta_rule":
        H, G, D, E = 4, 2, 64, 64
        gd, hv = G * D, H * E
        return ops.delta_rule, dict(
            proj=r(T, 2 * gd + 2 * hv + 2 * H, dt=dtype), offsets=[0, gd, 2 * gd, 2 * gd + hv, 2 * gd + 2 * hv, 2 * gd + 2 * hv + H],
            conv_q=r(gd, 4, dt=dtype), conv_k=r(gd, 4, dt=dtype), conv_v=r(hv, 4, dt=dtype), a_log=r(H), dt_bias=r(H), norm_weight=r(E, dt=dtype),
            eps=1e-5, state=r(T + 1, hv * D), conv_state=r(T + 1, 3 * (2 * gd + hv)), state_indices=idx, seq_lens=lens, q_start=None, q_len=None,
            num_heads=H, num_k_heads=G, k_dim=D, v_dim=E)
    H, G, N, E = 8, 2, 128, 64
    inner, C = H * E, H * E + 2 * G * N
    return ops.state_space, dict(
        proj=r(T, inner + C + H, dt=dtype), z_off=0, x_off=inner, dt_off=inner + C, conv_w=r(C, 4, dt=dtype), conv_b=r(C, dt=dtype), dt_bias=r(H),
        a_log=r(H), d_skip=r(H), norm_weight=r(inner, dt=dtype), norm_groups=1, eps=1e-5, state=r(T + 1, inner * N), conv_state=r(T + 1, 3 * C),
        state_indices=idx, seq_lens=lens, q_start=None, q_len=None, num_heads=H, groups=G, state_size=N, v_dim=E)


def _clone(args):
    return {k: v.clone() if isinstance(v, torch.Tensor) else v for k, v in args.items()}


@pytest.mark.parametrize("kind", ["delta_rule", "state_space"])
@pytest.mark.parametrize("T", [1, 3, 40])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_step_by_record_is_the_general_call(kind, T, dtype, monkeypatch):
    from semi_pd_amd import ops
    call, args = _step_call(kind, T, torch.Generator().manual_seed(T), dtype)
    columns = call(**_clone(args)).shape[1]
    for given in (False, True):
        a, b = ({**_clone(args), "out": torch.zeros(T, columns + 3, dtype=dtype, device="cuda")[:, :-3] if given else None} for _ in range(2))
        got = call(**a)
        monkeypatch.setattr(ops, "_delta_rule_step", lambda *_: None)
        monkeypatch.setattr(ops, "_state_space_step", lambda *_: None)
        want = call(**b)
        monkeypatch.undo()
        assert torch.equal(got, want) and torch.equal(a["state"], b["state"]) and torch.equal(a["conv_state"], b["conv_state"])


@pytest.mark.parametrize("kind", ["delta_rule", "state_space"])
def test_step_refuses_what_the_general_call_refuses(kind):
    call, args = _step_call(kind, 3, torch.Generator().manual_seed(1))
    conv = "conv_q" if kind == "delta_rule" else "conv_w"
    bad = {"proj": [args["proj"][0], args["proj"].t(), args["proj"].cpu(), args["proj"][:2], args["proj"][:, :-1], args["proj"].int()],
           conv: [args[conv][:-1], args[conv].float(), args[conv].t().contiguous().t(), args[conv].cpu()],
           "a_log": [args["a_log"][:-1], args["a_log"].double(), args["a_log"].cpu()],
           "norm_weight": [args["norm_weight"][1:], args["norm_weight"].float()],
           "state": [args["state"][:, 1:], args["state"].double(), args["state"].t(), args["state"].cpu()],
           "conv_state": [None, args["conv_state"][:, 1:], args["conv_state"].half()],
           "state_indices": [args["state_indices"].int()], "seq_lens": [args["seq_lens"].int(), args["seq_lens"][:2]],
           "q_start": [torch.zeros(3, dtype=torch.int32).cuda()], "out": [torch.empty(3, 5).cuda()]}
    if kind == "delta_rule":
        bad["offsets"] = [args["offsets"][:-1], [-1] + args["offsets"][1:], args["offsets"][:-1] + [args["proj"].shape[1]]]
    else:
        bad["dt_off"] = [-1, args["proj"].shape[1]]
    for name, values in bad.items():
        for value in values:
            with pytest.raises(RuntimeError):
                call(**{**args, name: value})
    # numbers of another kind go the general way
    eps = torch.tensor(1e-5)
    assert torch.equal(call(**_clone({**args, "eps": eps})), call(**_clone({**args, "eps": float(eps)})))


# (columns of a table, a length that all requests share: rows and lengths are the view's, not those of the memory behind its first element)
@pytest.mark.parametrize("kind", ["delta_rule", "state_space"])
@pytest.mark.parametrize("prompt", [False, True])
def test_rows_and_lengths_that_are_views(kind, prompt):
    T = 3
    call, args = _step_call(kind, T, torch.Generator().manual_seed(7))
    if prompt:
        args.update(q_start=torch.arange(T, dtype=torch.int32).cuda(), q_len=torch.ones(T, dtype=torch.int32).cuda())
    args["state_indices"] = torch.tensor([2, 3, 1]).cuda()
    table = torch.stack([torch.tensor([1, 1, 2]).cuda(), args["state_indices"], torch.tensor([3, 1, 1]).cuda()], 1)           # (all of it rows that there are)
    for lens, seen in ((torch.tensor([5, 1, 9]).cuda(), None), (torch.full((T,), 4).cuda(), torch.tensor([4]).cuda().expand(T))):
        dense, view = _clone({**args, "seq_lens": lens}), _clone(args)
        view["state_indices"] = table[:, 1]
        view["seq_lens"] = torch.stack([lens, lens.flip(0)], 1)[:, 0] if seen is None else seen
        assert not view["state_indices"].is_contiguous() and not view["seq_lens"].is_contiguous()
        assert torch.equal(call(**view), call(**dense))
        assert torch.equal(view["state"], dense["state"]) and torch.equal(view["conv_state"], dense["conv_state"])
