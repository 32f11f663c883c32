"""Short convolutions: several tokens a workgroup, and one-token steps that bring the carried inputs up to date themselves."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def portions(g, lens, carried):
    cu = torch.tensor([0] + lens).cumsum(0).int()
    slots = torch.randperm(len(lens) + 1, generator=g)[:len(lens)].int()
    slots[1] = -1
    return cu.cuda(), slots.cuda(), torch.tensor([n + c for n, c in zip(lens, carried)]).int().cuda()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("taps,dim", [(2, 4), (3, 1024), (4, 1028), (4, 2052), (5, 64), (4, 30)])
def test_stream(taps, dim, dtype):
    """Against the sum in float64: portions longer and shorter than the taps, across the workgroups' runs of tokens, fresh and carried, a padded row."""
    from nanovllm import ops
    g = torch.Generator().manual_seed(taps * dim)
    lens, carried = [1, 3, 2, 5, 4, 600, 1, 9], [0, 4, 7, 0, 3, 2, 9, 0]
    cu, slots, ctx = portions(g, lens, carried)
    x, w = torch.randn(sum(lens), dim, generator=g).cuda(), (torch.randn(dim, taps, generator=g) * 0.3).to(dtype).cuda()
    state = torch.randn(len(lens) + 1, taps - 1, dim, generator=g).cuda()
    before = state.clone()
    h = ops.stream_conv(x, w, state, slots, cu, ctx)
    for b, (n, c) in enumerate(zip(lens, carried)):
        own, lo = int(slots[b]), int(cu[b])
        old = before[own] if own >= 0 and c else torch.zeros_like(before[0])
        seq = torch.cat([old, x[lo:lo + n]]).double()
        want = x[lo:lo + n].double() + sum(seq[k:k + n] * w.double()[:, k] for k in range(taps))
        assert ((h[lo:lo + n].double() - want).abs() <= 2.0 ** -20 * want.abs().clamp(min=1) + (2.0 ** -8 * want.abs() if dtype is torch.bfloat16 else 0)).all()
        if own >= 0:
            assert torch.equal(state[own], seq[n:].float())
    B = len(lens)                                            # one token each: one launch, the bits of the two
    one, two, cu1 = before.clone(), before.clone(), torch.arange(B + 1, dtype=torch.int32).cuda()
    ctx1 = torch.tensor([1, 5, 2, 1, 9, 3, 4, 1]).int().cuda()
    assert torch.equal(ops.stream_conv(x[:B].contiguous(), w, one, slots, None, ctx1), ops.stream_conv(x[:B].contiguous(), w, two, slots, cu1, ctx1))
    assert torch.equal(one, two)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("taps,heads,inner,gn", [(4, 2, 64, 16), (2, 3, 48, 8), (3, 1, 20, 7), (5, 2, 32, 8), (4, 16, 4096, 1024)])
def test_ssd_step(taps, heads, inner, gn, dtype):
    from nanovllm import ops
    g = torch.Generator().manual_seed(taps * inner)
    B, c = 7, inner + 2 * gn
    def t(*shape):
        return torch.randn(*shape, generator=g).to(dtype).cuda()
    xbc, dt, w, bias, dtb, al = t(B, c), t(B, heads), t(c, taps), t(c), t(heads), t(heads)
    state = torch.randn(B + 1, taps - 1, c, generator=g).cuda()
    slots, ctx = torch.tensor([3, 0, -1, 7, 5, 1, 2]).int().cuda(), torch.tensor([1, 4, 3, 1, 2, 99, 3]).int().cuda()
    one, two = state.clone(), state.clone()
    a = ops.ssd_conv_prep(xbc, dt, w, bias, dtb, al, one, slots, None, ctx, heads, inner, gn)
    b = ops.ssd_conv_prep(xbc, dt, w, bias, dtb, al, two, slots, torch.arange(B + 1, dtype=torch.int32).cuda(), ctx, heads, inner, gn)
    assert all(torch.equal(p, q) for p, q in zip(a, b)) and torch.equal(one, two)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("taps,heads,groups,dk,dv", [(4, 16, 8, 64, 32), (2, 16, 16, 20, 24), (3, 8, 2, 128, 128), (5, 16, 8, 16, 16)])
def test_delta_operands(taps, heads, groups, dk, dv, dtype):
    """Many tokens (runs of them share a workgroup) against the same sequences one at a time: the same bits."""
    from nanovllm import ops
    g = torch.Generator().manual_seed(taps * dk)
    lens, carried = [5, 1, 300, 2, 210, 3, 8], [0, 4, 3, 0, 7, 1, 2]
    cu, slots, ctx = portions(g, lens, carried)
    T, c = sum(lens), 2 * groups * dk + heads * dv
    def t(*shape):
        return torch.randn(*shape, generator=g).to(dtype).cuda()
    qkv, b, a, w, dtb, al = t(T, c), t(T, heads), t(T, heads), t(c, taps), t(heads), t(heads)
    state = torch.randn(len(lens) + 1, taps - 1, c, generator=g).cuda()

    def operands(lo, hi, slots, cu, ctx):
        out = torch.empty(hi - lo, heads, 5 * dk + dv, device="cuda")
        rows = [v[lo:hi] for v in (qkv, b, a)]
        ops._hip.call("nvh_gated_delta_prep", rows[0].data_ptr(), c, rows[1].data_ptr(), heads, rows[2].data_ptr(), heads, w.data_ptr(), dtb.data_ptr(), al.data_ptr(),
                      state.data_ptr(), slots.data_ptr(), cu.data_ptr(), ctx.data_ptr(), out.data_ptr(), ctx.numel(), hi - lo, taps, heads, groups, dk, dv,
                      int(dtype is torch.float32), ops._stream())
        return out

    whole = operands(0, T, slots, cu, ctx)
    for i, n in enumerate(lens):
        lo = int(cu[i])
        alone = operands(lo, lo + n, slots[i:i + 1].contiguous(), torch.tensor([0, n]).int().cuda(), ctx[i:i + 1].contiguous())
        assert torch.equal(whole[lo:lo + n], alone)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("taps,dim", [(2, 1024), (3, 2052), (4, 1028)])
def test_stream_of_many_elements(taps, dim, dtype):
    """Runs of four tokens a workgroup (from 15 * 2^17 elements on) across the ends of sequences: the bits of a call per sequence, which takes a token each."""
    from nanovllm import ops
    g = torch.Generator().manual_seed(taps * dim)
    lens, carried = [1, 3, 2, 5, 4, 1900 * 1024 // dim, 1, 62, 9], [0, 4, 7, 0, 3, 2, 9, 0, 1]
    cu, slots, ctx = portions(g, lens, carried)
    assert sum(lens) * dim >= 15 << 17
    x, w = torch.randn(sum(lens), dim, generator=g).cuda(), (torch.randn(dim, taps, generator=g) * 0.3).to(dtype).cuda()
    state = torch.randn(len(lens) + 1, taps - 1, dim, generator=g).cuda()
    one, many = state.clone(), state.clone()
    h = ops.stream_conv(x, w, many, slots, cu, ctx)
    for b, n in enumerate(lens):
        lo = int(cu[b])
        alone = ops.stream_conv(x[lo:lo + n].contiguous(), w, one, slots[b:b + 1].contiguous(), torch.tensor([0, n]).int().cuda(), ctx[b:b + 1].contiguous())
        assert torch.equal(h[lo:lo + n], alone)
    assert torch.equal(one, many)
