"""Steps in which every sequence starts: convolutions over time that leave the carried inputs in their own launch (nobody reads a slot then)."""
import pytest
import torch

pytestmark = pytest.mark.gpu

LENS = [[1], [2], [3, 1, 2, 5], [4, 64, 1, 15, 17, 2], [300, 3, 700],      # shorter than the taps, ends on and around the edges of tiles of 4, 16 and 64 tokens
        [1, 300, 2, 1, 700, 3, 1]]      # short portions among enough tokens for tiles of 2 and 4 of them (below 1024 tokens x heads there is one a workgroup)


def _step(lens, g):
    cu = torch.tensor([0] + lens).cumsum(0).int().cuda()
    slots = torch.randperm(len(lens) + 3, generator=g)[:len(lens)].int()
    slots[0] = -1 if len(lens) > 4 else slots[0]             # (a row without a slot)
    if len(lens) > 6:
        slots[2] = -1                                        # (and one of those that begin inside a tile)
    return cu, slots.cuda(), torch.tensor(lens).int().cuda()


@pytest.mark.parametrize("lens", LENS)
@pytest.mark.parametrize("taps", [2, 4, 5])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("dim", [1024, 2048, 36, 33])
def test_stream_conv(lens, taps, dtype, dim):
    from nanovllm import ops
    g = torch.Generator().manual_seed(sum(lens) + taps)
    cu, slots, ctx = _step(lens, g)
    x = torch.randn(sum(lens), dim, generator=g).cuda()
    w = torch.randn(dim, taps, generator=g).to(dtype).cuda()
    state = torch.randn(len(lens) + 3, taps - 1, dim, generator=g).cuda()
    other = state.clone()
    want = ops.stream_conv(x, w, state, slots, cu, ctx)
    got = ops.stream_conv(x, w, other, slots, cu, ctx, all_start=True)
    assert torch.equal(got, want) and torch.equal(other, state)


@pytest.mark.parametrize("lens", LENS)
@pytest.mark.parametrize("taps", [2, 4, 5])
@pytest.mark.parametrize("heads,qk,dk,dv", [(8, 8, 128, 128), (4, 2, 64, 64), (3, 1, 20, 12)])
def test_gated_delta(lens, taps, heads, qk, dk, dv):
    from nanovllm import ops
    g = torch.Generator().manual_seed(sum(lens) + taps)
    cu, slots, ctx = _step(lens, g)
    c, t = 2 * qk * dk + heads * dv, sum(lens)
    qkv = torch.randn(t, c, generator=g).bfloat16().cuda()
    b, a = torch.randn(t, heads, generator=g).bfloat16().cuda(), torch.randn(t, heads, generator=g).bfloat16().cuda()
    w = torch.randn(c, taps, generator=g).bfloat16().cuda()
    dt, al = torch.randn(heads, generator=g).bfloat16().cuda(), torch.randn(heads, generator=g).bfloat16().cuda()
    conv, mem = torch.randn(len(lens) + 3, taps - 1, c, generator=g).cuda(), torch.randn(len(lens) + 3, heads, dk, dv, generator=g).cuda()
    conv2, mem2 = conv.clone(), mem.clone()
    run = lambda cv, m, **kw: ops.gated_delta_rule(qkv, b, a, w, dt, al, cv, m, slots, cu, ctx, heads, qk, dk, dv, max_seqlen_q=max(lens), **kw)
    live = torch.cat([torch.full((n,), int(s) >= 0) for n, s in zip(lens, slots.cpu())]).cuda()          # (rows without a slot get no result)
    want, got = run(conv, mem), run(conv2, mem2, all_start=True)
    assert torch.equal(got[live], want[live]) and torch.equal(conv2, conv) and torch.equal(mem2, mem)


@pytest.mark.parametrize("lens", LENS)
@pytest.mark.parametrize("taps", [2, 4, 5])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("heads,kv,dim,vdim,own", [(16, 8, 64, 128, True), (3, 1, 20, 12, True), (4, 4, 128, 128, False)])
def test_attention_conv(lens, taps, dtype, heads, kv, dim, vdim, own):
    from nanovllm import ops
    g = torch.Generator().manual_seed(sum(lens) + taps)
    cu, slots, ctx = _step(lens, g)
    t, c = sum(lens), heads * dim + (kv * (dim + vdim) if own else 0)
    proj = torch.randn(t, c + 8, generator=g).to(dtype).cuda()
    w = torch.randn(c, taps, generator=g).to(dtype).cuda()
    state = torch.randn(len(lens) + 3, taps - 1, c, generator=g).cuda()
    pages = -(-t // 256)
    got = []
    for all_start in (False, True):
        s = state.clone()
        kc = torch.zeros(pages, 256, kv, dim, dtype=dtype, device="cuda") if own else None
        vc = torch.zeros(pages, kv, vdim, 256, dtype=dtype, device="cuda") if own else None
        q = ops.attn_conv_prep(proj, w, s, slots, cu, ctx, torch.arange(t).int().cuda() if own else None, kc, vc, heads, kv, dim, vdim, 1e-6, all_start=all_start)
        got.append([x for x in (q, s, kc, vc) if x is not None])
    assert all(torch.equal(x, y) for x, y in zip(*got))
