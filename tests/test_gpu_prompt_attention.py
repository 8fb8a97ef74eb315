"""Prompt attention with 32 query rows a wave (csrc/local_attention_prompt.h) against a dense softmax / sigmoid in 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
# heads over key/value heads: four heads a workgroup, two, one (three heads of a group), sixteen
GROUPS = {"4": (8, 2), "2": (4, 2), "3": (6, 2), "16": (16, 1)}


def _batch(lens, olds, H, G, D, E, dtype, seed, shared=False):
    g = torch.Generator().manual_seed(seed)
    totals = [n + m for n, m in zip(lens, olds)]
    slots = torch.randperm(sum(totals), generator=g) + 1
    table, at = torch.zeros(len(lens), max(totals), dtype=torch.int32), 0
    for b, n in enumerate(totals):
        table[b, :n] = slots[at: at + n]
        at += n
    t = dict(q=torch.randn(sum(lens), H * D, generator=g).to(dtype), k=torch.randn(sum(totals) + 1, G, D, generator=g).to(dtype),
             v=torch.randn(sum(totals) + 1, G, E, generator=g).to(dtype), table=table, totals=totals)
    return t, g


def _dense(t, lens, olds, H, G, D, E, see, weights, shared=False):
    out, at = [], 0
    for b, (n, m) in enumerate(zip(lens, olds)):
        rows = t["table"][b, : n + m].long()
        p, j = torch.arange(m, m + n)[:, None], torch.arange(n + m)[None]
        ok = see(p, j)
        heads = []
        for h in range(H):
            gk = h // (H // G)
            s = t["q"][at: at + n, h * D: (h + 1) * D].double() @ t["k"][rows, gk].double().t() * D ** -0.5
            v = t["v"][rows].double().reshape(n + m, -1) if shared else t["v"][rows, gk].double()
            heads.append(weights(s, ok, h) @ v)
        out.append(torch.stack(heads, 1))
        at += n
    return torch.cat(out).reshape(sum(lens), -1)


def _softmax(sink=None, cap=0.0):
    def f(s, ok, h):
        if cap:
            s = cap * torch.tanh(s / cap)
        s = s.masked_fill(~ok, -float("inf"))
        if sink is None:
            return torch.softmax(s, -1)
        return torch.softmax(torch.cat([s, sink[h].double().expand(s.shape[0], 1)], 1), -1)[:, :-1]
    return f


# rows: one tile of 32, its edges, several; keys: a step of 64 and its edges, behind cached tokens, a block / window edge inside a step
CASES = [([1, 33, 64], [0, 0, 5]), ([31, 129], [100, 0]), ([70], [63])]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("lens,olds", CASES)
@pytest.mark.parametrize("group,D", [("4", 128), ("2", 64), ("3", 128), ("16", 64)])
@pytest.mark.parametrize("form", ["block", "causal", "cap", "window", "keep", "sigmoid"])
def test_prompt_attention(dtype, lens, olds, group, D, form):
    """Weights are rounded to 16 bits once (half a unit in the last place each, independent) and so is the result: 1.5 units of the
    largest partial sums, which are a few times the result's own size."""
    from semi_pd_amd import ops
    H, G = GROUPS[group]
    t, g = _batch(lens, olds, H, G, D, D, dtype, H * D + len(lens))
    per_head, gate = torch.randn(H, generator=g), torch.randn(sum(lens), H * D, generator=g).to(dtype)
    n, start = torch.tensor(lens, dtype=torch.int32), torch.tensor([0] + lens[:-1], dtype=torch.int32).cumsum(0).int()
    d = {k: v.to(DEV) for k, v in t.items() if k != "totals"}
    out = torch.empty_like(d["q"])
    batch = (d["q"], out, d["k"], d["v"], d["table"], torch.arange(len(lens), device=DEV), torch.tensor(t["totals"], device=DEV), start.to(DEV),
             n.to(DEV), max(lens), D ** -0.5)
    head = per_head.to(DEV)
    if form == "block":
        ops.local_attention_fwd(*batch, 0.0, 48, head, gate.to(DEV))
        want = _dense(t, lens, olds, H, G, D, D, lambda p, j: (j <= p) & (j // 48 == p // 48), _softmax(per_head)) * torch.sigmoid(gate.double())
    elif form in ("causal", "cap"):
        cap = 2.0 if form == "cap" else 0.0
        ops.local_attention_fwd(*batch, cap, 0, None, None)
        want = _dense(t, lens, olds, H, G, D, D, lambda p, j: j <= p, _softmax(cap=cap))
    else:
        keep = 0 if form == "window" else 70 if form == "keep" else 3
        see = lambda p, j: (j <= p) & ((p - j < 40) | (j < keep))          # noqa: E731
        if form == "sigmoid":
            ops.window_attention_fwd(*batch, 40, keep, head, True, None, 1.2)
            want = _dense(t, lens, olds, H, G, D, D, see, lambda s, ok, h: 1.2 * torch.sigmoid(s + per_head[h].double()).masked_fill(~ok, 0.0))
        else:
            ops.window_attention_fwd(*batch, 40, keep, None, False, head, 1.0)
            want = _dense(t, lens, olds, H, G, D, D, see, _softmax(per_head))
    ulp = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    err = (out.cpu().double() - want).norm() / want.norm()
    assert float(err) < 1.5 * ulp, float(err)
    torch.testing.assert_close(out.cpu().double(), want, rtol=6 * ulp, atol=12 * ulp)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("value", [float("nan"), float("inf"), -float("inf")])
@pytest.mark.parametrize("form,D,E", [("causal", 128, 128), ("block", 64, 64), ("window", 64, 64), ("keep", 128, 128), ("sigmoid", 64, 64),
                                      ("shared", 128, 256), ("shared", 64, 128)])
def test_values_that_are_not_finite_stay_with_the_rows_that_see_them(dtype, value, form, D, E):
    """One element of the value rows of a few keys: rows that do not see them are as without them (to the rounding of their weights, as
    above), the others hold what the sum holds."""
    from semi_pd_amd import ops
    H, G, lens, olds = (4, 2, [150], [40]) if form != "shared" else (4, 2, [90, 70], [0, 33])
    t, g = _batch(lens, olds, H, G, D, E // 2 if form == "shared" else E, dtype, D + E)
    head = torch.randn(H, generator=g).to(DEV)
    n, start = torch.tensor(lens, dtype=torch.int32), torch.tensor([0] + lens[:-1], dtype=torch.int32).cumsum(0).int()
    bad = [3, 77, 101]                                                              # positions, of every request

    def run(v):
        d = {k: x.to(DEV) for k, x in t.items() if k != "totals"}
        d["v"] = v.to(DEV)
        out = torch.empty(sum(lens), H * E, dtype=dtype, device=DEV)
        batch = (d["q"], out, d["k"], d["v"], d["table"], torch.arange(len(lens), device=DEV), torch.tensor(t["totals"], device=DEV), start.to(DEV),
                 n.to(DEV), max(lens), D ** -0.5)
        if form == "shared":
            ops.shared_value_attention_fwd(*batch)
        elif form in ("causal", "block"):
            ops.local_attention_fwd(*batch, 0.0, 48 if form == "block" else 0, None, None)
        else:
            ops.window_attention_fwd(*batch, 40, 0 if form == "window" else 2 if form == "sigmoid" else 70, head, form == "sigmoid", None, 1.0)
        return out.cpu().float().view(-1, H, E)

    clean, v = run(t["v"]), t["v"].clone()
    for b in range(len(lens)):
        v[t["table"][b, bad].long(), 0, 5] = value
    got, at = run(v), 0
    heads = slice(0, H) if form == "shared" else slice(0, H // G)                    # (the first key/value head's, or the row that all share)
    hit = torch.zeros_like(got, dtype=torch.bool)
    for b, (new, old) in enumerate(zip(lens, olds)):
        p, j = torch.arange(old, old + new)[:, None], torch.tensor(bad)[None]
        see = {"causal": j <= p, "shared": j <= p, "block": (j <= p) & (j // 48 == p // 48)}.get(
            form, (j <= p) & ((p - j < 40) | (j < (0 if form == "window" else 2 if form == "sigmoid" else 70))))
        hit[at: at + new, heads, 5] = see.any(1)[:, None]
        at += new
    ulp = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    torch.testing.assert_close(got[~hit], clean[~hit], rtol=6 * ulp, atol=12 * ulp)
    assert bool(torch.isnan(got[hit]).all() if value != value else (got[hit] == value).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D", [64, 128])
def test_largest_weight_of_every_32_keys_is_not_rounded(dtype, D):
    """Two keys carry the weight, one in the first 32 and a larger one in the next 32, and their values cancel all but the rounding of
    the smaller one's weight to 16 bits.  Weight 1 at the time it is rounded, a factor in fp32 (four roundings of 2^-23, values of
    256) behind it; the result is rounded once."""
    from semi_pd_amd import ops
    H, G, n, small, large = 4, 1, 64, 5, 40
    scores = torch.linspace(0.1, 2.0, n - large).to(dtype)                        # of the larger key, row by row
    weight = torch.exp(-scores.double())
    q, k, v = torch.zeros(n, H, D), torch.zeros(n + 1, G, D), torch.zeros(n + 1, G, D)
    q[:, :, 1] = 1.0
    q[large:, :, 0] = scores.float()[:, None]
    k[1:, 0, 1] = -200.0
    k[1 + small, 0, 1], k[1 + large, 0, :2] = 0.0, torch.tensor([1.0, 0.0])
    v[1 + small, 0] = 256.0
    v[1 + large, 0, : n - large] = -256.0 * weight.to(dtype).float()
    q, k, v = (x.to(dtype).to(DEV) for x in (q.view(n, H * D), k, v))
    one = lambda x, t=torch.int32: torch.tensor([x], dtype=t, device=DEV)          # noqa: E731
    out = torch.empty_like(q)
    ops.local_attention_fwd(q, out, k, v, torch.arange(1, n + 1, dtype=torch.int32, device=DEV)[None], one(0, torch.int64), one(n, torch.int64),
                            one(0), one(n), n, 1.0, 0.0, 0, None, None)
    want = ((v[1 + small, 0].double().cpu() * weight[:, None] + v[1 + large, 0].double().cpu()) / (1 + weight[:, None]))[:, None]
    ulp = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    torch.testing.assert_close(out[large:].view(-1, H, D).double().cpu(), want.expand(-1, H, D), rtol=ulp, atol=256 * 2.0 ** -21)


# (requests: the scalar search and the one by lanes, whole and part waves of them; heads: one, two or four of a group in a workgroup)
@pytest.mark.parametrize("requests", [8, 9, 64, 65, 131])
@pytest.mark.parametrize("H,G,D,E", [(7, 1, 64, 64), (6, 2, 128, 128), (3, 3, 64, 64), (14, 2, 64, 128), (11, 1, 128, 256), (8, 4, 64, 64),
                                     (8, 8, 128, 128), (24, 12, 64, 64)])
def test_prompt_attention_of_many_requests(requests, H, G, D, E):
    """Short uneven prompts, some without a row in the launch, some behind cached tokens."""
    from semi_pd_amd import ops
    lens = [(20, 1, 0, 33, 9)[i % 5] for i in range(requests)]
    olds = [(0, 40, 3)[i % 3] if n else 5 for i, n in enumerate(lens)]
    shared = E != D
    t, g = _batch(lens, olds, H, G, D, E // G if shared else E, torch.bfloat16, requests + H)
    n, start = torch.tensor(lens, dtype=torch.int32), torch.tensor([0] + lens[:-1], dtype=torch.int32).cumsum(0).int()
    d = {k: v.to(DEV) for k, v in t.items() if k != "totals"}
    out = torch.full((sum(lens), H * E), 7.0, dtype=torch.bfloat16, device=DEV)
    batch = (d["q"], out, d["k"], d["v"], d["table"], torch.arange(requests, device=DEV), torch.tensor(t["totals"], device=DEV), start.to(DEV),
             n.to(DEV), max(lens), D ** -0.5)
    if shared:
        ops.shared_value_attention_fwd(*batch)
    else:
        ops.local_attention_fwd(*batch, 0.0, 0, None, None)
    want = _dense(t, lens, olds, H, G, D, E, lambda p, j: j <= p, _softmax(), shared=shared)
    assert float((out.cpu().double() - want).norm() / want.norm()) < 1.5 * 2.0 ** -8
    torch.testing.assert_close(out.cpu().double(), want, rtol=6 * 2.0 ** -8, atol=12 * 2.0 ** -8)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("lens,olds", CASES)
@pytest.mark.parametrize("H,G,D", [(16, 2, 128), (6, 2, 128), (8, 2, 64)])
def test_prompt_attention_over_shared_values(dtype, lens, olds, H, G, D):
    from semi_pd_amd import ops
    t, g = _batch(lens, olds, H, G, D, D, dtype, H * D)
    n, start = torch.tensor(lens, dtype=torch.int32), torch.tensor([0] + lens[:-1], dtype=torch.int32).cumsum(0).int()
    d = {k: v.to(DEV) for k, v in t.items() if k != "totals"}
    out = torch.empty(sum(lens), H * G * D, dtype=dtype, device=DEV)
    ops.shared_value_attention_fwd(d["q"], out, d["k"], d["v"], d["table"], torch.arange(len(lens), device=DEV),
                                   torch.tensor(t["totals"], device=DEV), start.to(DEV), n.to(DEV), max(lens), D ** -0.5)
    want = _dense(t, lens, olds, H, G, D, D, lambda p, j: j <= p, _softmax(), shared=True)
    ulp = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    assert float((out.cpu().double() - want).norm() / want.norm()) < 1.5 * ulp
    torch.testing.assert_close(out.cpu().double(), want, rtol=6 * ulp, atol=12 * ulp)


# heads over one and two tiles of 16 a key/value head, sums over one to four steps of 16, neither whole
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("H,G,E", [(32, 2, 128), (24, 2, 64), (40, 4, 16), (33, 1, 32), (64, 2, 16), (6, 3, 48), (40, 4, 64), (33, 1, 80), (64, 2, 64),
                                   (48, 8, 64), (16, 4, 64), (15, 3, 64)])
def test_talk_mix(dtype, H, G, E):
    """fp32 products and sums of at most 64 terms, the result rounded once.  With p significant bits half a unit in the last place of x is
    at most 2^-p |x| (just above a power of two): 2^-8 for bf16, 2^-11 for fp16; the sum: 64 roundings of 2^-24 of its terms."""
    from semi_pd_amd import ops
    g = torch.Generator().manual_seed(H + E)
    parts, talk = torch.randn(5, H * G * E, generator=g).to(dtype), torch.randn(H, H, generator=g)
    out = ops.talk_mix(parts.to(DEV), talk.to(DEV), G).cpu().double().view(5, H, E)
    x = parts.double().view(5, H, G, E)[:, :, torch.arange(H) // (H // G)]                    # [t, g, c(h), e]
    want = torch.einsum("hg,tghe->the", talk.double(), x)
    terms = torch.einsum("hg,tghe->the", talk.double().abs(), x.abs())
    half = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    assert bool(((out - want).abs() <= half * want.abs() + 64 * 2.0 ** -24 * terms + 1e-7).all())


# more tokens than the chip takes at once (a workgroup has several), by itself and among others, more 16-byte pieces a token than are fetched ahead
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("H,G,E,tokens", [(12, 2, 64, 4097), (24, 2, 128, 3001), (40, 4, 64, 2049), (64, 1, 256, 1300)])
def test_talk_mix_of_many_tokens(dtype, H, G, E, tokens):
    """Every token's row is what it is in a call of its own, and what is not finite in one stays in it."""
    from semi_pd_amd import ops
    g = torch.Generator(device=DEV).manual_seed(H)
    parts, talk = torch.randn(tokens, H * G * E, generator=g, device=DEV).to(dtype), torch.randn(H, H, generator=g, device=DEV)
    parts[tokens - 7, 3], parts[5, 70] = float("inf"), float("nan")
    out = ops.talk_mix(parts, talk, G)
    finite = torch.isfinite(out.float()).all(1)
    assert bool((finite == (torch.arange(tokens, device=DEV) != tokens - 7) & (torch.arange(tokens, device=DEV) != 5)).all())
    for t0 in (0, tokens // 2, tokens - 11):
        few = ops.talk_mix(parts[t0: t0 + 11].contiguous(), talk, G)
        same = out[t0: t0 + 11]
        assert bool(((few == same) | (torch.isnan(few) & torch.isnan(same))).all())


# few heads over many key/value heads, which do not fill a product's columns, on both sides of that line and of what the vector form stages
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("H,G,E", [(8, 8, 64), (8, 4, 128), (8, 2, 64), (8, 2, 128), (10, 10, 128), (10, 10, 192), (12, 12, 64), (14, 14, 64)])
def test_talk_mix_of_few_heads_over_many(dtype, H, G, E):
    from semi_pd_amd import ops
    g = torch.Generator().manual_seed(H + G)
    parts, talk = torch.randn(300, H, G, E, generator=g).to(dtype), torch.randn(H, H, generator=g)
    out = ops.talk_mix(parts.view(300, -1).to(DEV), talk.to(DEV), G).cpu().double()
    mine = parts.double()[:, :, torch.arange(H) // (H // G)]                                              # [token, weights of head, head, E]
    want = torch.einsum("hg,tghe->the", talk.double(), mine).reshape(300, -1)
    terms = torch.einsum("hg,tghe->the", talk.double().abs(), mine.abs()).reshape(300, -1)
    half = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    assert bool(((out - want).abs() <= half * want.abs() + 64 * 2.0 ** -24 * terms + 1e-7).all())


# (launches large enough that tiles go by their keys: blocks of 18 tiles, one row past a tile's edge in front; of 70, two of which are a level;
# requests without blocks, so many keys that three tiles are a level)
@pytest.mark.parametrize("block,lens,olds", [(576, [700, 0, 33, 400, 1], [545, 7, 5, 0, 576]), (2240, [500, 1, 600], [2000, 64, 3]), (2240, [1100], [1999]),
                                             (0, [900, 0, 1200, 130], [0, 9, 4001, 70]), (0, [300, 200, 260, 0, 330, 410, 290, 310], [0, 31, 32, 1, 64, 0, 5, 0])])
def test_prompt_attention_tiles_by_their_keys(block, lens, olds):
    """Every row is there once, whatever the order: against the dense form, into a result that holds something else."""
    _rows_once(64, 16, block, lens, olds)


# (runs of tiles: all XCDs share the heads, four or two do; one request, some without rows, more of them than eight; a launch that is hardly
# more than the chip takes at once, whose tiles go round the XCDs)
@pytest.mark.parametrize("H,G,block,lens,olds", [(6, 3, 256, [700], [300]), (4, 1, 192, [300, 0, 513, 261], [5, 9, 0, 100]), (12, 6, 100, [1030], [0]),
                                                 (28, 4, 256, [259, 270], [255, 0]), (9, 3, 0, [300, 0, 700, 260, 290, 310, 256, 400, 270, 33], [0, 4, 0, 1, 0, 8, 0, 0, 9, 0]),
                                                 (24, 3, 128, [550, 481, 512, 499, 530], [200, 0, 201, 9, 0])])
def test_prompt_attention_runs_of_tiles(H, G, block, lens, olds):
    _rows_once(H, G, block, lens, olds)


def _rows_once(H, G, block, lens, olds):
    from semi_pd_amd import ops
    D = 64
    t, g = _batch(lens, olds, H, G, D, D, torch.bfloat16, sum(lens))
    n, start = torch.tensor(lens, dtype=torch.int32), torch.tensor([0] + lens[:-1], dtype=torch.int32).cumsum(0).int()
    d = {k: v.to(DEV) for k, v in t.items() if k != "totals"}
    out = torch.full((sum(lens), H * D), 7.0, dtype=torch.bfloat16, device=DEV)
    ops.local_attention_fwd(d["q"], out, d["k"], d["v"], d["table"], torch.arange(len(lens), device=DEV), torch.tensor(t["totals"], device=DEV),
                            start.to(DEV), n.to(DEV), max(lens), D ** -0.5, 0.0, block, None, None)
    see = (lambda p, j: (j <= p) & (j // block == p // block)) if block else lambda p, j: j <= p          # noqa: E731
    got, at = out.cpu().double(), 0
    for b, (new, old) in enumerate(zip(lens, olds)):                                # (a few heads: the order is the same for all)
        rows, p, j = t["table"][b, : new + old].long(), torch.arange(old, old + new)[:, None], torch.arange(new + old)[None]
        for h in sorted({0, H // 3, H - 1}):
            s = t["q"][at: at + new, h * D: (h + 1) * D].double() @ t["k"][rows, h // (H // G)].double().t() * D ** -0.5
            want = torch.softmax(s.masked_fill(~see(p, j), -float("inf")), -1) @ t["v"][rows, h // (H // G)].double()
            torch.testing.assert_close(got[at: at + new, h * D: (h + 1) * D], want, rtol=6 * 2.0 ** -8, atol=12 * 2.0 ** -8)
        at += new


# (tiles of a launch: up to 256 of 64 rows and heads, of 128, more; a few steps for four groups of waves, and one or two fewer than the groups)
@pytest.mark.parametrize("lens,olds", [([150, 33, 64], [0, 30, 700]), ([500, 200], [0, 561]), ([900, 260], [60, 0]), ([1290], [3])])
@pytest.mark.parametrize("H,G,D,E,form", [(H, 8, D, D, form) for H, D in ((32, 128), (24, 64)) for form in ("causal", "cap", "window", "keep", "sigmoid")] +
                         [(16, 2, 128, 256, "causal"), (32, 8, 64, 128, "causal")])
def test_steps_in_turns(lens, olds, H, G, D, E, form):
    """Groups of waves that take a tile's steps in turn, and their sums together: tolerances as above."""
    from semi_pd_amd import ops
    dtype = torch.bfloat16
    t, g = _batch(lens, olds, H, G, D, E // G if E != D else E, dtype, H + D)
    per_head = torch.randn(H, generator=g)
    n, start = torch.tensor(lens, dtype=torch.int32), torch.tensor([0] + lens[:-1], dtype=torch.int32).cumsum(0).int()
    d = {k: v.to(DEV) for k, v in t.items() if k != "totals"}
    out = torch.empty(sum(lens), H * E, dtype=dtype, device=DEV)
    batch = (d["q"], out, d["k"], d["v"], d["table"], torch.arange(len(lens), device=DEV), torch.tensor(t["totals"], device=DEV), start.to(DEV),
             n.to(DEV), max(lens), D ** -0.5)
    head, causal = per_head.to(DEV), lambda p, j: j <= p
    if E != D:
        ops.shared_value_attention_fwd(*batch)
        want = _dense(t, lens, olds, H, G, D, E, causal, _softmax(), shared=True)
    elif form in ("causal", "cap"):
        cap = 2.0 if form == "cap" else 0.0
        ops.local_attention_fwd(*batch, cap, 0, head if form == "causal" else None, None)
        want = _dense(t, lens, olds, H, G, D, E, causal, _softmax(per_head if form == "causal" else None, cap=cap))
    else:
        keep = 0 if form == "window" else 70 if form == "keep" else 3
        see = lambda p, j: (j <= p) & ((p - j < 520) | (j < keep))          # noqa: E731
        if form == "sigmoid":
            ops.window_attention_fwd(*batch, 520, keep, head, True, None, 1.2)
            want = _dense(t, lens, olds, H, G, D, E, see, lambda s, ok, h: 1.2 * torch.sigmoid(s + per_head[h].double()).masked_fill(~ok, 0.0))
        else:
            ops.window_attention_fwd(*batch, 520, keep, None, False, head, 1.0)
            want = _dense(t, lens, olds, H, G, D, E, see, _softmax(per_head))
    ulp = 2.0 ** -8
    err = (out.cpu().double() - want).norm() / want.norm()
    assert float(err) < 1.5 * ulp, float(err)
    # (sigmoid weights are not divided by their sum: rounding of up to 520 of them where above there are 40, errors of the root of that)
    wide = (520 / 40) ** 0.5 if form == "sigmoid" else 1.0
    torch.testing.assert_close(out.cpu().double(), want, rtol=6 * ulp, atol=12 * ulp * wide)
