"""Grouped bf16 products: every tile form gives a row the bits of the plain any-shape product."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("out_f32,act", [(False, None), (True, None), (False, "relu2")])
@pytest.mark.parametrize("n,k", [(4, 64), (60, 128), (64, 192), (132, 448), (200, 1024)])
def test_blocks_of_every_size(n, k, out_f32, act):
    """Experts without a row, with one, around 16, 32, 64, 128 and 192 rows and more than 64 tiles' worth: tiles of few rows, pairs of tiles, a pair's
    odd last tile.  The reference reads rows that no 16-byte load may be used on, which takes the general form."""
    from nanovllm import ops
    sizes = [0, 1, 15, 16, 17, 32, 33, 64, 65, 127, 128, 129, 192, 0, 4200]
    g = torch.Generator().manual_seed(n + k)
    ids = torch.repeat_interleave(torch.arange(len(sizes)), torch.tensor(sizes))[torch.randperm(sum(sizes), generator=g)].int()[:, None].cuda()
    T = ids.shape[0]
    x = torch.randn(T, k, generator=g).bfloat16().cuda()
    w = (torch.randn(len(sizes), n, k, generator=g) * 0.1).bfloat16().cuda()
    plan = ops.moe_align(ids, len(sizes))
    at = plan["pos_of_pair"].long()
    odd = torch.empty(T, k + 1, dtype=x.dtype, device=x.device)
    odd[:, :k] = x
    want = ops.linear_grouped(odd[:, :k], w, plan, True, out_f32, act)[at]
    default = ops.GROUPED_MANY_ROWS
    try:
        for few in (1 << 30, 0):                             # the tiles for few rows an expert, and those for many
            ops.GROUPED_MANY_ROWS = few
            assert torch.equal(ops.linear_grouped(x, w, plan, True, out_f32, act)[at], want)
            rows = x[plan["src_token"].long()]
            assert torch.equal(ops.linear_grouped(rows, w, plan, False, out_f32, act)[at], want)
    finally:
        ops.GROUPED_MANY_ROWS = default


@pytest.mark.parametrize("experts,top,k", [(1, 1, 8), (3, 2, 1000), (16, 4, 1024), (64, 64, 1536), (65, 7, 520), (300, 80, 2048)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_routing(experts, top, k, dtype):
    """Choices and weights against the logits that the same launch hands out: the largest, ties to the lower number, -inf and NaN never before others."""
    from nanovllm import ops
    g = torch.Generator().manual_seed(experts * top)
    T = 9
    x, w = torch.randn(T, k, generator=g).to(dtype).cuda(), (torch.randn(experts, k, generator=g) * 0.1).to(dtype).cuda()
    if experts > 2:
        w[2] = w[0]                                          # a tie
    ids, weights, logits = ops.moe_route_linear(x, w, None, top, want_logits=True)
    want = x.double().cpu() @ w.double().cpu().t()
    assert ((logits.double().cpu() - want).abs() <= (k + 8) * 2.0 ** -24 * (x.double().abs().cpu() @ w.double().abs().cpu().t())).all()
    order = torch.sort(logits.cpu(), dim=1, descending=True, stable=True).indices[:, :top]
    assert torch.equal(ids.cpu().long(), order)
    soft = torch.softmax(logits.cpu().double().gather(1, order), 1)
    assert torch.allclose(weights.cpu().double(), soft, rtol=1e-5, atol=1e-12)
    ids, weights = ops.moe_route_linear(x, w, None, top, sigmoid_scores=True)
    assert torch.equal(ids.cpu().long(), order) and torch.allclose(weights.cpu().double(), torch.sigmoid(logits.cpu().double().gather(1, order)), rtol=1e-5, atol=1e-12)
    ids, weights, _, scores = ops.moe_route_scored(x, w, top, want_scores=True, renorm=True)
    order = torch.sort(scores.cpu(), dim=1, descending=True, stable=True).indices[:, :top]
    assert torch.equal(ids.cpu().long(), order)
    picked = scores.cpu().double().gather(1, order)
    assert torch.allclose(weights.cpu().double(), picked / picked.sum(1, keepdim=True), rtol=1e-5)
    x[0] = float("nan")                                      # whatever is chosen then are different experts of the list
    ids = ops.moe_route_scored(x, w, top)[0]
    assert ids[0].min() >= 0 and ids[0].max() < experts and ids[0].unique().numel() == top


@pytest.mark.parametrize("act,weighted", [("silu", False), ("gelu_tanh", False), ("relu2", False), ("glu_clamp", False), ("glu_clamp", True)])
@pytest.mark.parametrize("inter,k", [(2, 64), (30, 128), (32, 192), (66, 448), (384, 1024)])
def test_gated(inter, k, act, weighted):
    """The activation in the product's epilogue against the product and the activation as launches of their own, bit for bit: experts of every size,
    two and three choices a token, the tiles for few rows an expert and those for many; rows that no 16-byte load may be used on."""
    from nanovllm import ops
    g = torch.Generator().manual_seed(inter + k)
    T, E, top = 900, 9, 3
    chance = torch.tensor([0.0, 0.01, 0.02, 0.1, 0.2, 0.5, 1.0, 2.0, 6.0])
    ids = torch.multinomial(chance.expand(T, E) + 1e-6, top, generator=g).int().cuda()
    ids[5] = -1                                              # a row of padding: no expert
    x = torch.randn(T, k, generator=g).bfloat16().cuda()
    w = (torch.randn(E, 2 * inter, k, generator=g) * 0.2).bfloat16().cuda()
    weights = torch.rand(T, top, generator=g).cuda() if weighted else None
    plan = ops.moe_align(ids, E)
    first = ops.linear_grouped(x, w, plan, gather=True)
    want = ops.glu_clamp_pairs(first, plan, weights, 1.5, 1.702) if act == "glu_clamp" else ops.act_mul(first, act, True)
    odd = torch.empty(T, k + 1, dtype=x.dtype, device=x.device)
    odd[:, :k] = x
    at = plan["pos_of_pair"].long()
    at = at[at >= 0]
    assert at.numel() == (T - 1) * top and torch.equal(plan["src_token"].long()[at], torch.arange(T, device="cuda").repeat_interleave(top)[plan["pos_of_pair"] >= 0])
    default = ops.GROUPED_MANY_ROWS
    try:
        for few in (1 << 30, 0):
            ops.GROUPED_MANY_ROWS = few
            for rows in (x, odd[:, :k]):
                assert torch.equal(ops.linear_grouped_gated(rows, w, plan, act, weights, 1.5, 1.702)[at], want[at])
    finally:
        ops.GROUPED_MANY_ROWS = default


@pytest.mark.parametrize("experts,top,tokens", [(1, 1, 1), (16, 2, 64), (63, 3, 341), (64, 4, 1000), (65, 5, 1025), (200, 8, 700), (4096, 2, 300)])
def test_align(experts, top, tokens):
    """The order by expert: every pair has a place of its own in its expert's run, the tiles cover the runs; pairs that one pass of the threads holds and more."""
    from nanovllm import ops
    g = torch.Generator().manual_seed(experts + tokens)
    ids = torch.randint(-1, experts, (tokens, top), generator=g).int()
    plan = {k: v.cpu() if torch.is_tensor(v) else v for k, v in ops.moe_align(ids.cuda(), experts).items()}
    flat, pos = ids.flatten().long(), plan["pos_of_pair"].long()
    kept = flat >= 0
    assert (pos[~kept] == -1).all() and torch.equal(pos[kept].sort().values, torch.arange(int(kept.sum())))
    by_pos = torch.empty(int(kept.sum()), dtype=torch.long)
    by_pos[pos[kept]] = flat[kept]
    assert torch.equal(by_pos, flat[kept].sort().values)
    assert torch.equal(plan["src_token"].long()[pos[kept]], torch.arange(tokens * top)[kept] // top)
    tiles = [(int(e), int(r), int(n)) for e, r, n in zip(plan["tile_expert"], plan["tile_row0"], plan["tile_rows"]) if n > 0]
    count = torch.bincount(flat[kept], minlength=experts)
    starts = count.cumsum(0) - count
    assert tiles == [(e, int(starts[e]) + r, min(64, int(count[e]) - r)) for e in range(experts) for r in range(0, int(count[e]), 64)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("experts,k", [(5, 96), (16, 1000), (16, 1024), (30, 1536), (100, 1024), (100, 1000), (300, 2048), (300, 520)])
def test_routing_does_not_depend_on_the_number_of_tokens(experts, k, dtype):
    """More tokens than the rows' pieces are taken two at once for, against the same tokens in calls of few: choices, weights, scores and further products."""
    from nanovllm import ops
    g = torch.Generator().manual_seed(experts + k)
    T, top = 1030, min(experts, 4)
    x, w, aux = (torch.randn(n, k, generator=g).to(dtype).cuda() for n in (T, experts, 1))
    many = ops.moe_route_scored(x, w, top, aux=aux, want_scores=True, renorm=True)
    for lo, hi in ((0, 7), (500, 564), (1020, 1030)):
        few = ops.moe_route_scored(x[lo:hi], w, top, aux=aux, want_scores=True, renorm=True)
        assert all(torch.equal(m[lo:hi], f) for m, f in zip(many, few))
    many_linear, few_linear = ops.moe_route_linear(x, w, None, top, want_logits=True), ops.moe_route_linear(x[:9], w, None, top, want_logits=True)
    assert all(torch.equal(m[:9], f) for m, f in zip(many_linear, few_linear))
    size = x.double().abs() @ w.double().abs().t().contiguous()
    slack = (2 * (k + 8) * 2.0 ** -24 * size).amax(1, keepdim=True) + 2.0 ** -20          # (of the logits; softmax's relative error is at most twice theirs)
    scores = torch.softmax(x.double() @ w.double().t().contiguous(), 1)
    assert ((many[3].double() - scores).abs() <= scores * 2 * slack + 1e-30).all()


@pytest.mark.parametrize("experts,top,tokens", [(64, 8, 512), (64, 8, 513), (64, 8, 2048), (64, 8, 2049), (3, 2, 9000)])
def test_align_of_pairs_beyond_the_kept_ones(experts, top, tokens):
    """Around the numbers of pairs that the threads keep: those beyond are counted after the others' ranks are taken, and placed from their run's end."""
    test_align(experts, top, tokens)
