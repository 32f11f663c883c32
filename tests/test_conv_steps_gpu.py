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
